"""The band heights of the column-walking y sweeps: every height gives bitwise
the wave-strip sweeps' state, on meshes with a last band of one row, a whole
one, and fewer rows than a band."""
import numpy as np
import pytest

import mahyco_amd

from gpu_helpers import field_names, log
from test_gpu_fixed_options import problem
from test_gpu_variants import env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("rows", [4, 8, 16, 32, 64])
@pytest.mark.parametrize("m,nx,ny,pp", [(1, 65, 33, 0), (2, 64, 16, 0), (3, 30, 3, 0), (2, 66, 65, 1)])
def test_band_heights(m, nx, ny, pp, rows, precision):
    cfg = problem(m, nx, ny, "minmod", precision, pp)
    log(f"[walk] m={m} {nx}x{ny} pp={pp} rows={rows} precision={precision}")
    with env("MAHYCO_SWEEP_Y", "wave"):
        strip = mahyco_amd.Context(cfg)
    with env("MAHYCO_SWEEP_Y", "walk"), env("MAHYCO_WALK_ROWS", str(rows)), env("MAHYCO_LAG_Y", "separate"):
        walk = mahyco_amd.Context(cfg)
    try:
        for n in (1, 1, 10):
            strip.run(n)
            walk.run(n)
            diff = [f"{f}[{k}]" for f, k in field_names(cfg) if not np.array_equal(strip.get(f, k), walk.get(f, k))]
            assert not diff, diff
    finally:
        strip.close()
        walk.close()
