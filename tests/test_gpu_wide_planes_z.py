"""The GLM and CT marches on z planes at the reach of their 32-bit offsets, with two different planes: the plane's own
address and the offset within it are added, and neither path may leave its plane.  Both precisions and the
species builds; each grid is a periodic repetition of a small one, whose bits every cell must have."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from glmmhdturb_amd import Params, Solver, step_args  # noqa: E402

NX, PX, NZ = 32768, 32, 2
# precision -> (ny, rows of the small grid): the largest plane below 4 GiB and the first of 4 GiB
SIZES = {"f32": ((32767, 217), (32768, 256)), "f64": ((16383, 129), (16384, 256))}


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("kind,prec,nsp", [("glm", "f32", 0), ("glm", "f64", 0), ("glm", "f32", 2), ("ct", "f32", 0),
                                           ("ct", "f64", 0), ("ct", "f64", 2)])
def test_two_planes_at_the_offset_limit(kind, prec, nsp, wide):
    ny, py = SIZES[prec][wide]
    size = 4 if prec == "f32" else 8
    assert (size * NX * ny > 2**32 - 1) == wide
    nv = (8 if kind == "ct" else 9) + nsp
    if torch.cuda.mem_get_info()[0] < 2.2 * nv * NZ * NX * ny * size:
        pytest.skip("two states of 8 GiB a variable do not fit")
    g = torch.Generator(device="cuda").manual_seed(ny + nv)
    u = torch.rand((nv, NZ, py, PX), generator=g, device="cuda", dtype=torch.float32 if prec == "f32" else torch.float64) * 0.1
    u[0] += 1.0
    u[4] += 2.0
    u[5] += 0.5
    a = step_args(Params(N=PX, nx=PX, ny=py, nz=NZ, gamma=5.0 / 3.0, courant=0.4), 1e-3, 0.0, want_cfl=True)

    def step(q):
        s = Solver(Params(N=PX, nx=q.shape[3], ny=q.shape[2], nz=NZ, gamma=5.0 / 3.0, courant=0.4), prec)
        out = torch.full_like(q, float("nan"))
        if kind == "ct":
            s.ct_step_species(q, out, a) if nsp else s.ct_step(q, out, a)
        else:
            s.step_species(q, out, a) if nsp else s.step(q, out, a)
        s.close()
        return out

    small = step(u)
    assert torch.isfinite(small).all() and not torch.equal(small[:, 0], small[:, 1])
    big = step(u.repeat(1, 1, ny // py, NX // PX))
    for v in range(nv):
        for k in range(NZ):
            assert bool((big[v, k].view(ny // py, py, NX // PX, PX) == small[v, k].view(1, py, 1, PX)).all()), (v, k)
    del big
    torch.cuda.empty_cache()
