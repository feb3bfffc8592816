"""MAHYCO_LAG_Y: mhy_tuned_kernels reports the variant that runs, also where the
options have no kernel for the forced one (walking bands with fixed options only;
PenteBorne and third order keep the Lagrange update a kernel of its own in y-first steps)."""
import pytest

import mahyco_amd

from gpu_helpers import log
from test_gpu_fixed_options import problem
from test_gpu_variants import env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("forced,lim,pp,order,runs", [
    ("walk", "minmod", 0, 2, "walk"), ("walk", "superBee", 0, 2, "walk"), ("walk", "vanLeer", 0, 2, "fused"),
    ("fused", "minmod", 0, 2, "fused"), ("separate", "minmod", 0, 2, "separate"), ("fused", "superBee", 1, 2, "separate"),
    ("walk", "superBee", 1, 2, "separate"), ("walk", "minmod", 0, 3, "separate")])
def test_report_is_what_runs(forced, lim, pp, order, runs):
    cfg = problem(2, 70, 40, lim, 0, pp)
    cfg.projection_order = order
    log(f"[lag forced] {forced} {lim} pp={pp} order={order}")
    with env("MAHYCO_LAG_Y", forced):
        ctx = mahyco_amd.Context(cfg)
    try:
        assert ctx.tuned_kernels() == f"lagrange_y={runs}"
        ctx.run(1)
        ctx.enable_timing()
        ctx.run(1)  # the second step is the first along y
        n = {k: v["launches"] for k, v in ctx.kernel_stats().items()}
        assert n["lagrange_sweep_y"] == (1 if runs != "separate" else 0), n
        assert n["lagrange_cell"] == (1 if runs == "separate" else 0), n
    finally:
        ctx.close()
