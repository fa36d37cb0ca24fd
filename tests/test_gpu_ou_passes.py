"""The OU advance over the forms its transforms take (csrc/ou.hip: the y and z passes as one kernel where a plane's
band fits LDS, separate passes for wide bands): narrow and full bands, odd and even grids, the largest plane
of the one-kernel form and the first past it, against the oracle's dense transform."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import OUForcing  # noqa: E402
from glmmhdturb_amd import Params, Solver  # noqa: E402


# (g, kmax): nb = min(2 floor(kmax) + 1, g), a plane takes nb * g * 16 bytes of at most 64 KiB
@pytest.mark.parametrize("g,kmax", [(2, 1.0), (5, 2.0), (16, 3.0), (33, 5.0), (64, 3.0), (64, 32.0), (66, 31.0)])
def test_ou_advance_matches_dense_transform(orc, g, kmax):
    p = Params(N=8, turb_gs=g, turb_kmin=1.0, turb_kmax=kmax, turb_T=0.5, turb_Ndt=10, turb_seed=7)
    s = Solver(p, "f64")
    f = s.setup_forcing(p, 3.0)
    fo = OUForcing(orc, g, 1.0, kmax, 0.5, 10, p.comp_frac, 3.0, 7)
    for _ in range(2):
        f.advance()
        fo.advance()
    got = s.afield().cpu().numpy().reshape(-1)
    # nb terms an axis, each within a few ulps of the largest partial sum
    assert np.max(np.abs(got - fo.afield)) <= 1e-13 * g * max(np.max(np.abs(fo.afield)), 1e-300)


# separate passes for the box alone (96 or 192 planes of many terms), one kernel for the boxes together
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n,g,kmax", [(4, 32, 5.0), (4, 33, 16.0), (3, 64, 3.0), (2, 64, 31.0)])
def test_a_box_alone_and_among_others_has_the_same_bits(n, g, kmax, prec):
    from glmmhdturb_amd.ensemble import BoxSpec, Ensemble, single_box_run
    boxes = [BoxSpec(N=8, seed=7 + b, amp=3e3, turb_gs=g, turb_kmax=kmax, turb_Ndt=20) for b in range(n)]
    ens = Ensemble(boxes, precision=prec)
    ens.step(5)
    ens.sync()
    log = ens.log(n - 1, 5)
    assert log[0]["ou_due"] and log[4]["ramp"] > 0
    _, u, _ = single_box_run(boxes[-1], ens.scheme, 5, prec, log=log)
    assert torch.equal(ens.current(n - 1), u) and float(u[1].abs().max()) > 0
    ens.close()
