"""The FP32 hydro march around the edges of its work split (see test_gpu_hydro_tiles.py for the sizes): its builds have
another register budget and take supersonic faces by a branch."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import HydroScheme  # noqa: E402
from glmmhdturb_amd import Params, Solver, hydro_args  # noqa: E402
from test_gpu_hydro import G, run_oracle, voids  # noqa: E402
from test_gpu_hydro_tiles import GRIDS  # noqa: E402
from test_gpu_hydro_variants import run, with_species  # noqa: E402
from test_hydro_oracle import smooth_hydro  # noqa: E402


@pytest.mark.parametrize("variant", ["plm", "fallback", "ppm", "donor"])
@pytest.mark.parametrize("nsp", [0, 2])
def test_tile_edges_fp32_vs_oracle(orc, variant, nsp):
    """Two steps against the FP64 oracle on the same rounded state, with the FP64 test's bar in FP32's ulp (1e-13 is
    450 of FP64's)."""
    for nx, ny, nz in GRIDS:
        u = (voids if variant == "fallback" else smooth_hydro)(nx, ny, nz, 3 + nx)
        if nsp:
            u = with_species(u, 5)
        u = u.astype(np.float32).astype(np.float64)
        fb = (1e-3, 1e-3) if variant == "fallback" else None
        sc = HydroScheme(gamma=G, dtdx=0.04, nsp=nsp, cma=nsp > 0, ppm=variant == "ppm", donor=variant == "donor",
                         fallback=fb is not None)
        s = Solver(Params(N=nx, nx=nx, ny=ny, nz=nz, gamma=G), "f32")
        got = run(s, u, hydro_args(0.04, G, ppm=variant == "ppm", fallback=fb), 2, nsp=nsp, cma=nsp > 0,
                  donor=variant == "donor")
        ref = run_oracle(orc, u, sc, 2)
        err = np.abs(got - ref).reshape(5 + nsp, -1).sum(1) / (np.abs(ref[0]).sum() + np.abs(ref[4]).sum())
        assert np.all(err <= 450 * np.finfo(np.float32).eps), (variant, nsp, (nx, ny, nz), err)
        s.close()
