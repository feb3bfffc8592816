"""mhy_kernel_bytes of one-material contexts: the material fields that are stored only
where they differ from the means are not counted, one flag is."""
import pytest

import mahyco_amd

from gpu_helpers import log
from test_gpu_fixed_options import problem
from test_gpu_variants import env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("centred", [0, 1])
@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_compact_bytes(precision, centred):
    cfg = problem(1, 37, 21, "minmod", precision)
    cfg.pseudo_centree = centred
    log(f"[kernel bytes] precision={precision} centred={centred}")
    got = {}
    for compact in ("0", "1"):
        with env("MAHYCO_COMPACT", compact):
            ctx = mahyco_amd.Context(cfg)
        got[compact] = {k: v["bytes"] for k, v in ctx.kernel_stats().items()}
        ctx.close()
    cells, r, d = 37 * 21, (4 if precision else 8), 8
    less = {k: got["0"][k] - got["1"][k] for k in got["0"]}
    # the final remap: f_k, M_k (FP64), mu, rho, e, p, c of the material
    final = cells * (2 * d + 5 * r - 1)
    # the Lagrange update: f_k, M_k and mu, rho, e, p of the material, for M, e and p of the cell
    lagrange = cells * (2 * d + 4 * r - d - 2 * r - 1)
    for k in ("sweep_x", "sweep_y", "remap_final"):
        assert less[k] == final, k
    for k in ("lagrange_cell", "lagrange_sweep_x", "lagrange_sweep_y"):
        assert less[k] == lagrange, k
    assert all(less[k] == 0 for k in ("dt_reduce", "lagrange_node", "dual_x", "dual_y", "dual_both"))
