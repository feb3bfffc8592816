"""Phase-level steps after a finished time loop (mhy_simulate ends without the n / n+1
swap of its last step): the time step of each is reduced from its own state, also
where the last whole step had left a CFL minimum (bands of 16 node rows)."""
import numpy as np
import pytest

import mahyco_amd
from mahyco_amd import configs

from gpu_helpers import field_names, log
from test_gpu_phases import step_by_phases
from test_gpu_variants import env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_phases_after_simulate(precision):
    cfg = configs.point_explosion(96)
    cfg.ny, cfg.precision, cfg.max_time_iterations = 50, precision, 7
    log(f"[phases after simulate] precision={precision}")
    with env("MAHYCO_DUAL_ROWS", "16"):
        kept = mahyco_amd.Context(cfg)
    with env("MAHYCO_DUAL_ROWS", "2"):
        reduced = mahyco_amd.Context(cfg)
    try:
        for ctx in (kept, reduced):
            ctx.simulate()
        for _ in range(4):
            for ctx in (kept, reduced):
                step_by_phases(ctx)
            diff = [f"{f}[{k}]" for f, k in field_names(cfg) if not np.array_equal(kept.get(f, k), reduced.get(f, k))]
            assert not diff, diff
            assert kept.time_state().deltat_n == reduced.time_state().deltat_n
    finally:
        kept.close()
        reduced.close()
