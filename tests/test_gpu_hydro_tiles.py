"""The hydro march around the edges of its work split (csrc/hydro_march.hpp: 30 x 16 column tiles, rows of 32
lanes, two rows a lane; donor seams every 32 x 8 cells): grids one cell short of, at and past a tile, odd
row counts, single cells, against the CPU oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import HydroScheme  # noqa: E402
from glmmhdturb_amd import hydro_args  # noqa: E402
from test_gpu_hydro import G, run_oracle, solver, voids  # noqa: E402
from test_gpu_hydro_variants import run, with_species  # noqa: E402
from test_hydro_oracle import smooth_hydro  # noqa: E402

GRIDS = [(1, 1, 1), (2, 3, 1), (29, 15, 2), (30, 16, 3), (31, 17, 2), (32, 8, 1), (60, 33, 5), (64, 47, 2), (95, 4, 7)]


@pytest.mark.parametrize("variant", ["plm", "fallback", "ppm", "donor"])
@pytest.mark.parametrize("nsp", [0, 2])
def test_tile_edges_fp64_vs_oracle(orc, variant, nsp):
    """Two steps; the summed error of a variable is at most 1e-13 of the summed density and energy (a few
    tens of roundings of the terms of an update, each within an ulp)."""
    for nx, ny, nz in GRIDS:
        u = (voids if variant == "fallback" else smooth_hydro)(nx, ny, nz, 3 + nx)
        if nsp:
            u = with_species(u, 5)
        fb = (1e-3, 1e-3) if variant == "fallback" else None
        sc = HydroScheme(gamma=G, dtdx=0.04, nsp=nsp, cma=nsp > 0, ppm=variant == "ppm", donor=variant == "donor",
                         fallback=fb is not None)
        s = solver(nx, ny, nz)
        got = run(s, u, hydro_args(0.04, G, ppm=variant == "ppm", fallback=fb), 2, nsp=nsp, cma=nsp > 0,
                  donor=variant == "donor")
        ref = run_oracle(orc, u, sc, 2)
        err = np.abs(got - ref).reshape(5 + nsp, -1).sum(1) / (np.abs(ref[0]).sum() + np.abs(ref[4]).sum())
        assert np.all(err <= 1e-13), (variant, nsp, (nx, ny, nz), err)
        s.close()
