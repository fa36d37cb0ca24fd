"""The two-wave fluxes (HLL and LLF: csrc/physics.hpp two_wave_x, csrc/hydro_march.hpp hy_riemann) against 80-bit
arithmetic on states down to Mach 0.01, where U_L - U_R has to be formed before it is multiplied by the wave speeds."""
import ctypes as C
import os

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "glmmhdturb_amd", "_build", "libfluxcheck.so")
G = 1.4
X = np.longdouble


def solve(name, kind, L, R):
    if not os.path.exists(LIB):
        pytest.skip("host flux build is missing (tests/native)")
    f = np.empty_like(L)
    ptr = [a.ctypes.data_as(C.c_void_p) for a in (L, R, f)]
    getattr(C.CDLL(LIB), name)(C.c_int(kind), *ptr, C.c_long(len(L)), C.c_double(G))
    return f


def pair(nv, mach, jump, dtype, n=4000):
    """Two states a face: the same one and up to `jump` of relative change in every value."""
    r = np.random.default_rng(5)
    b = np.zeros((n, nv))
    b[:, 0], b[:, 4] = r.uniform(0.5, 2, n), r.uniform(0.5, 2, n)
    a = np.sqrt(G * b[:, 4] / b[:, 0])
    b[:, 1:4] = mach * a[:, None] * r.uniform(-1, 1, (n, 3))
    if nv == 9:
        b[:, 5:8] = r.uniform(-1, 1, (n, 3))
    L, R = (b * (1 + jump * r.uniform(-1, 1, b.shape)) for _ in range(2))
    if nv == 9:
        R[:, 5] = L[:, 5]   # the face's normal field is one value
    return L.astype(dtype), R.astype(dtype)


def two_wave(L, R, llf, fast):
    """Weights and k of wL FL + wR FR + k (UL - UR) in 80 bits."""
    cl, cr = fast(L), fast(R)
    if llf:
        s = np.maximum(abs(L[1]) + cl, abs(R[1]) + cr)
        sl, sr = -s, s
    else:
        sl = np.minimum(np.minimum(L[1] - cl, R[1] - cr), 0)
        sr = np.maximum(np.maximum(L[1] + cl, R[1] + cr), 0)
    return sr / (sr - sl), -sl / (sr - sl), -sl * sr / (sr - sl)


@pytest.mark.parametrize("llf", [0, 1], ids=["hll", "llf"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("mach,jump", [(0.01, 0.02), (0.1, 0.02), (1.0, 0.02), (1.0, 0.5)])
def test_mhd_flux_error_follows_the_jump(mach, jump, dtype, llf):
    """Mass and transverse field, whose jump is exact: every term is a product of up to four rounded factors (the
    speeds to 4 ulp), so 8 ulp of the sum of their magnitudes.  Terms of +-k U would leave 0.5 ulp of k U each."""
    L, R = pair(9, mach, jump, dtype)
    f = solve("fc_mhd_f32" if dtype == np.float32 else "fc_mhd_f64", llf, L, R).T
    l, r = L.astype(X).T, R.astype(X).T

    def fast(q):
        b2 = q[5] ** 2 + q[6] ** 2 + q[7] ** 2
        h = 0.5 * (G * q[4] + b2) / q[0]
        return np.sqrt(h + np.sqrt(np.maximum(h * h - X(G) * q[4] * q[5] ** 2 / q[0] ** 2, 0)))

    wl, wr, k = two_wave(l, r, llf, fast)
    terms = {0: (l[0] * l[1], r[0] * r[1], k * (l[0] - r[0])),
             6: (l[6] * l[1] - l[5] * l[2], r[6] * r[1] - r[5] * r[2], k * (l[6] - r[6]))}
    size = {0: abs(l[0] * l[1]) + abs(r[0] * r[1]),
            6: abs(l[6] * l[1]) + abs(l[5] * l[2]) + abs(r[6] * r[1]) + abs(r[5] * r[2])}
    for c, (fl, fr, d) in terms.items():
        err = abs(f[c] - (wl * fl + wr * fr + d))
        assert np.all(err <= 8 * np.finfo(dtype).eps * (size[c] + abs(d))), (c, float((err / (size[c] + abs(d))).max()))


@pytest.mark.parametrize("llf", [0, 1], ids=["hll", "llf"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("mach,jump", [(0.01, 0.02), (0.1, 0.02), (1.0, 0.02), (1.0, 0.5)])
def test_hydro_flux_error_follows_the_jump(mach, jump, dtype, llf):
    """The mass flux, with the same bound."""
    L, R = pair(7, mach, jump, dtype)
    f = solve("fc_hydro_f32" if dtype == np.float32 else "fc_hydro_f64", llf, L, R).T
    l, r = L.astype(X).T, R.astype(X).T
    wl, wr, k = two_wave(l, r, llf, lambda q: np.sqrt(X(G) * q[4] / q[0]))
    fl, fr, d = l[0] * l[1], r[0] * r[1], k * (l[0] - r[0])
    err = abs(f[0] - (wl * fl + wr * fr + d))
    assert np.all(err <= 8 * np.finfo(dtype).eps * (abs(fl) + abs(fr) + abs(d)))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name", ["fc_hydro", "fc_hydro_sel"])
def test_supersonic_hydro_flux_is_the_upwind_sides(name, dtype):
    """Both waves to one side: that side's flux, with its own roundings only, whatever the other side holds."""
    name += "_f32" if dtype == np.float32 else "_f64"
    L, R = pair(7, 0.5, 0.1, dtype, 500)
    for q in (L, R):
        q[:, 1] = 3 + abs(q[:, 1])   # above every sound speed of the pair
        q[:, 5:] = 0.3
    m = L[:, 0] * L[:, 1]
    E = L[:, 4].astype(X) / (X(G) - 1) + L[:, 0] * (L[:, 1:4].astype(X) ** 2).sum(1) / 2
    up = solve(name, 0, L, R)
    assert np.array_equal(up[:, 0], m)
    for c in (2, 3, 5, 6):
        assert np.array_equal(up[:, c], m * L[:, c])
    # the product and the sum with p, whether fused or not; E's terms, p and the product with u
    eps = np.finfo(dtype).eps
    assert np.all(abs(up[:, 1] - (L[:, 0].astype(X) * L[:, 1] * L[:, 1] + L[:, 4])) <= 2 * eps * abs(up[:, 1]))
    assert np.all(abs(up[:, 4] - (E + L[:, 4]) * L[:, 1]) <= 6 * eps * abs(up[:, 4]))
    flip = np.array([1, -1, 1, 1, 1, 1, 1], dtype)   # the mirrored face
    down = solve(name, 0, R * flip, L * flip)
    assert np.array_equal(down * flip, -up)
    for v, x in [(0, np.nan), (1, np.nan), (2, np.nan), (3, np.inf), (4, np.nan), (5, np.nan), (6, np.inf), (1, np.inf), (0, np.inf)]:
        bad = R.copy()
        bad[:, v] = x
        assert np.array_equal(solve(name, 0, L, bad), up), (v, x)
        assert np.array_equal(solve(name, 0, bad * flip, L * flip), down), (v, x)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_hydro_update_rounds_a_value_once(dtype):
    """Density, momenta and scalars: one rounding at the value's size and one at the change's."""
    q, div = pair(7, 1.0, 0.5, dtype)
    q[:, 5:] = 0.3
    u = np.empty_like(q)
    ptr = [a.ctypes.data_as(C.c_void_p) for a in (q, div, u)]
    if not os.path.exists(LIB):
        pytest.skip("host flux build is missing (tests/native)")
    k = dtype(0.05)
    getattr(C.CDLL(LIB), "fc_update_f32" if dtype == np.float32 else "fc_update_f64")(*ptr, C.c_long(len(q)), C.c_double(k))
    for c in (0, 1, 2, 3, 5, 6):
        d = X(k) * div[:, c]
        x = (q[:, 0].astype(X) * q[:, c] if c else q[:, 0].astype(X)) - d
        assert np.all(abs(u[:, c] - x) <= 0.5 * np.finfo(dtype).eps * (1.001 * abs(x) + abs(d))), c
