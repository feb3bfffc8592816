"""The Lagrange update inside the column-walking first y sweep: bitwise the strips'
state, with a last band of one row, a whole one, and fewer rows than a band; with
options that have no such kernel the strips run."""
import numpy as np
import pytest

import mahyco_amd

from gpu_helpers import field_names, log
from test_gpu_fixed_options import problem
from test_gpu_variants import env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("lim", ["minmod", "superBee", "vanLeer"])
@pytest.mark.parametrize("m,nx,ny,rows", [(1, 65, 33, 32), (1, 5, 3, 8), (2, 64, 16, 16), (3, 130, 9, 8), (3, 63, 65, 64)])
def test_fused_walk(m, nx, ny, rows, lim, precision):
    cfg = problem(m, nx, ny, lim, precision, 0)
    log(f"[lag walk] m={m} {nx}x{ny} rows={rows} {lim} precision={precision}")
    with env("MAHYCO_LAG_Y", "fused"):
        strip = mahyco_amd.Context(cfg)
    with env("MAHYCO_LAG_Y", "walk"), env("MAHYCO_WALK_ROWS", str(rows)):
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
