"""The GLM and CT marches on z planes at the reach of their 32-bit offsets (csrc/march_impl.hpp Column,
csrc/ct_march.hpp CmColumn): the largest FP32 plane below 4 GiB and the first at 4 GiB, each a periodic
repetition of a small grid, so that every cell must come out with the bits of the small grid's step."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from glmmhdturb_amd import Params, Solver, step_args  # noqa: E402


@pytest.mark.parametrize("ct", [False, True], ids=["glm", "ct"])
@pytest.mark.parametrize("ny,py", [(32767, 217), (32768, 256)])
def test_step_at_the_offset_limit(ny, py, ct):
    nx, px = 32768, 32
    assert (4 * nx * ny <= 2**32 - 1) == (ny == 32767)
    if torch.cuda.mem_get_info()[0] < 100e9:
        pytest.skip("two FP32 states of a billion cells take 77 GB")
    g = torch.Generator(device="cuda").manual_seed(ny)
    nv = 8 if ct else 9
    u = torch.rand((nv, 1, py, px), generator=g, device="cuda", dtype=torch.float32) * 0.1
    u[0] += 1.0
    u[4] += 2.0
    u[5] += 0.5

    def step(q):
        p = Params(N=px, nx=q.shape[3], ny=q.shape[2], nz=1, gamma=5.0 / 3.0, courant=0.4)
        s = Solver(p, "f32")
        out = torch.empty_like(q)
        a = step_args(Params(N=px, nx=px, ny=py, nz=1, gamma=5.0 / 3.0, courant=0.4), 1e-3, 0.0, want_cfl=True)
        if ct:
            s.ct_step(q, out, a)
            c = 0.0
        else:
            s.step(q, out, a)
            c = s.cfl_max()
        s.close()
        return out, c

    small, c0 = step(u)
    big, c1 = step(u.repeat(1, 1, ny // py, nx // px))
    for v in range(nv):
        assert bool((big[v, 0].view(ny // py, py, nx // px, px) == small[v, 0].view(1, py, 1, px)).all()), v
    assert c1 == c0
