"""Every z-chunk length gives the same bits (the automatic one follows the kernel's occupancy): the GLM, CT and hydro
marches over their solvers, reconstructions and predictors, both precisions, against one chunk of all planes."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from glmmhdturb_amd import Params, Solver, hydro_args, step_args  # noqa: E402

NX, NY, NZ = 37, 29, 13   # ragged tiles, a last chunk shorter than the others
CHUNKS = (0, 1, 2, 5)


def state(nv, prec, mag=True):
    """A transonic random state with jumps between cells, mag: with a magnetic field."""
    g = torch.Generator(device="cuda").manual_seed(7)
    dt = torch.float64 if prec == "f64" else torch.float32
    r = lambda: torch.rand((NZ, NY, NX), generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    u = torch.zeros((nv, NZ, NY, NX), device="cuda", dtype=torch.float64)
    u[0] = 0.3 + 2.0 * r()
    for c in (1, 2, 3):
        u[c] = u[0] * (1.6 * r() - 0.8)
    u[4] = 0.4 + r() + 0.5 * (u[1] ** 2 + u[2] ** 2 + u[3] ** 2) / u[0]
    if mag:
        for c in (5, 6, 7):
            u[c] = r() - 0.5
        u[4] += 0.5 * ((u[5:8].abs() + 0.5) ** 2).sum(0)
    for s in range(9 if nv > 9 else (8 if mag else 5), nv):
        u[s] = (0.1 * (r() - 0.5)) if nv == 9 else u[0] * r()
    return u.to(dt)


def same_bits(step, u):
    out = {}
    for z in (NZ,) + CHUNKS:
        o = torch.full_like(u, float("nan"))
        step(u, o, z)
        out[z] = o
    assert torch.isfinite(out[NZ]).all()
    for z in CHUNKS:
        assert torch.equal(out[z], out[NZ]), (z, [int((out[z][v] != out[NZ][v]).sum()) for v in range(len(u))])


P = Params(N=NX, nx=NX, ny=NY, nz=NZ, gamma=5.0 / 3.0, courant=0.4)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("pred", ["full", "oned"])
@pytest.mark.parametrize("riemann", ["llf", "llf_bound", "hll", "hlld"])
@pytest.mark.parametrize("recon", ["plm", "ppm", "ppm_spike"])
def test_glm(prec, pred, riemann, recon):
    s = Solver(P, prec)
    same_bits(lambda u, o, z: s.step(u, o, step_args(P, 2e-3, 0.0, riemann=riemann, recon=recon, predictor=pred, zchunk=z)),
              state(9, prec))
    s.close()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("riemann", ["llf", "hll", "hlld"])
@pytest.mark.parametrize("recon", ["plm", "ppm_spike"])
@pytest.mark.parametrize("nsp", [0, 2])
def test_ct(prec, riemann, recon, nsp):
    s = Solver(P, prec)
    a = lambda z: step_args(P, 2e-3, 0.0, riemann=riemann, recon=recon, predictor="oned", zchunk=z)  # noqa: E731
    same_bits(lambda u, o, z: s.ct_step_species(u, o, a(z)) if nsp else s.ct_step(u, o, a(z)), state(8 + nsp, prec))
    s.close()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("variant", ["plm", "fallback", "ppm", "donor"])
@pytest.mark.parametrize("nsp", [0, 2])
def test_hydro(prec, variant, nsp):
    s = Solver(P, prec)
    kw = {"fallback": dict(fallback=(0.6, 0.6)), "ppm": dict(ppm=True)}.get(variant, {})
    same_bits(lambda u, o, z: s.hydro_step(u, o, hydro_args(0.05, zchunk=z, **kw), nsp=nsp, cma=nsp > 0,
                                           donor=variant == "donor"), state(5 + nsp, prec, mag=False))
    s.close()
