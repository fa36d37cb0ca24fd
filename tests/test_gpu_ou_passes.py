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
