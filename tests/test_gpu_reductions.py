"""Whole-grid reductions of the GPU library (CFL maxima, max |div B|, diagnostics) against numpy on grids
around the edges of their work split: one cell, rows shorter and longer than a workgroup, a last
workgroup that is nearly empty, more cells than one pass of the workgroups."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (3, 2, 5), (255, 1, 2), (257, 9, 1), (300, 2, 3), (16, 16, 2), (67, 61, 130), (128, 64, 129)]
G = 5.0 / 3.0


def _state(shape, seed=4):
    nx, ny, nz = shape
    r = np.random.default_rng(seed)
    u = r.uniform(-0.3, 0.3, (9, nz, ny, nx))
    u[0] = r.uniform(0.5, 2.0, (nz, ny, nx))
    u[4] = r.uniform(3.0, 4.0, (nz, ny, nx))
    return u


def _cfl(rho, m, E, B):
    v = m / rho
    p = (G - 1.0) * (E - 0.5 * rho * (v ** 2).sum(0) - 0.5 * (B ** 2).sum(0))
    a2, b2 = G * p / rho, (B ** 2).sum(0) / rho
    h = 0.5 * (a2 + b2)
    c = np.sqrt(h + np.sqrt(np.maximum(h * h - a2 * B * B / rho, 0.0)))
    return (np.abs(v) + c).sum(0).max(), c.max()


@pytest.mark.parametrize("shape", SHAPES)
def test_reductions_match_numpy(shape):
    import torch
    from glmmhdturb_amd import Params, Solver
    nx, ny, nz = shape
    u = _state(shape)
    s = Solver(Params(N=nx, nx=nx, ny=ny, nz=nz, gamma=G), "f64")
    d = torch.from_numpy(u).cuda()
    cfl, fast = _cfl(u[0], u[1:4], u[4], u[5:8])
    assert s.ctot_max(d) == pytest.approx(cfl, rel=1e-14)
    assert s.fast_max(d) == pytest.approx(fast, rel=1e-14)
    up = lambda f, ax: np.roll(f, -1, ax)  # noqa: E731
    bc = 0.5 * np.stack([u[5] + up(u[5], 2), u[6] + up(u[6], 1), u[7] + up(u[7], 0)])
    q = d[:8].contiguous()
    assert s.ct_ctot_max(q) == pytest.approx(_cfl(u[0], u[1:4], u[4], bc)[0], rel=1e-14)
    div = (up(u[5], 2) - u[5]) + (up(u[6], 1) - u[6]) + (up(u[7], 0) - u[7])
    assert s.ct_divb_max(q, 1.0) == pytest.approx(np.abs(div).max(), rel=1e-14, abs=1e-15)
    got = s.diagnostics(d)
    m2, b2 = (u[1:4] ** 2).sum(0), (u[5:8] ** 2).sum(0)
    want = {"mass": u[0], "ke2": m2 / u[0], "ekin": 0.5 * m2 / u[0], "emag": 0.5 * b2,
            "cross_helicity": (u[1:4] * u[5:8]).sum(0) / u[0], "etot": u[4], "psi2": u[8] ** 2}
    for k, x in want.items():   # compensated sums: each term within two ulps, no error from adding
        assert abs(got[k] - math.fsum(x.ravel())) <= 4 * np.finfo(float).eps * np.abs(x).sum(), k
    cen = sum(np.roll(u[5 + c], -1, 2 - c) - np.roll(u[5 + c], 1, 2 - c) for c in range(3))
    assert got["divbmax"] == pytest.approx(np.abs(cen).max() / (2.0 / nx), rel=1e-13, abs=1e-13)
    assert got["rhomin"] == u[0].min() and got["finite"]
    d[2, -1, -1, -1] = float("nan")
    assert not s.diagnostics(d)["finite"]
    assert math.isnan(s.ctot_max(d))
