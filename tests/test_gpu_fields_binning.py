"""The no-allocation cell fields' own binning against the allocating entry
point, bit for bit, at the sizes where its scan and sort change: cell counts
around one block's scan (4,096 entries) and a scan tile, one particle, cells
in order and out of it, runs past the sorting network, a segment whose runs
do not fit the staging, most cells empty."""
import numpy as np
import pytest

from src_incompressible_openmp_amd.params import poiseuille_params, to_struct
from tests.test_zz_no_alloc import FIELDS, hip_runtime, run_noalloc

pytestmark = pytest.mark.gpu

CASES = {
    "one_particle": (7, 5, 1, 1.0, False),
    "below_one_block": (65, 63, 20000, 1.0, False),   # 4,095 cells + 1 = 4,096 entries
    "past_one_block": (64, 64, 20000, 1.0, False),
    "odd_tiles": (123, 101, 60000, 1.0, True),
    "long_runs": (16, 16, 12000, 1.0, False),         # 47 per cell, 12,000 in one segment
    "few_cells_hold_all": (40, 30, 3000, 0.15, False),
    "in_order": (50, 50, 25000, 1.0, True),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_matches_allocating_entry_point(name):
    from src_incompressible_openmp_amd import gpu

    nx, ny, n, part, ordered = CASES[name]
    hip = hip_runtime(gpu)
    p = to_struct(poiseuille_params(Nx=nx, Ny=ny, gamma=max(1.0, n / (nx * ny))))
    p.n = n
    rng = np.random.default_rng(5)
    x = rng.random((n, 2)) * np.array([p.Lx, p.Ly]) * part
    if ordered:
        cell = (x[:, 1] * (ny / p.Ly)).astype(int) + ny * (x[:, 0] * (nx / p.Lx)).astype(int)
        x = np.ascontiguousarray(x[np.argsort(cell, kind="stable")])
    v = rng.normal(size=(n, 2))
    want = gpu.compute_cell_fields(p, x.reshape(-1), v.reshape(-1), 3.0)
    got = run_noalloc(gpu, hip, p, x.reshape(-1).copy(), v.reshape(-1).copy(), 3.0)
    for k in ("N",) + FIELDS:
        assert np.asarray(got[k]).tobytes() == np.asarray(want[k]).tobytes(), k
