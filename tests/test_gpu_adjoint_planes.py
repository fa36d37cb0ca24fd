"""The reverse step on z planes at the reach of the back half's 32-bit offsets: the largest plane its
z-march takes and the first that goes to the separate passes (csrc/adj.hip), against those passes."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from glmmhdturb_amd import Params, Solver, step_args  # noqa: E402


@pytest.mark.parametrize("ny", [1620, 1621])
def test_reverse_step_at_the_offset_limit(ny):
    """1600 x 1620 cells x 207 scratch planes x 8 bytes is the last multiple below 4 GiB."""
    nx, nz = 1600, 2
    assert (nx * 207 * 8 * ny <= 2**32 - 1) == (ny == 1620)
    p = Params(N=nx, nx=nx, ny=ny, nz=nz, gamma=5.0 / 3.0, courant=0.4)
    s = Solver(p, "f64")
    g = torch.Generator(device="cuda").manual_seed(ny)
    u = torch.rand((9, nz, ny, nx), generator=g, device="cuda", dtype=torch.float64) * 0.1
    u[0] += 1.0
    u[4] += 2.0
    u[5] += 0.5
    w = torch.randn(u.shape, generator=g, device="cuda", dtype=torch.float64)
    a = step_args(p, 1e-4, 0.0, want_cfl=False, riemann="hlld", recon="ppm")
    out = []
    for passes in (False, True):
        lam0 = s.new_state()
        s.step_adjoint(u, w, lam0, a, passes=passes)
        out.append(lam0)
    assert torch.isfinite(out[1]).all()
    # the same sums in another order, as between the two paths on small grids
    assert (out[0] - out[1]).abs().max() <= 1e-13 * out[1].abs().max()
    s.close()
