"""A problem of an ensemble stepped by itself between the ensemble's steps.  Seven
problems of 300 x 300 cells leave enough waves for bands of 16 node rows, whose
nodal remap also reduces the next step's CFL minimum; the problem alone runs bands of 2
rows and reduces it in a kernel of its own.  Neither's captured steps may depend on
which of the two came before: bitwise the state of the same problem run alone."""
import numpy as np
import pytest

import mahyco_amd
from mahyco_amd import configs

from gpu_helpers import field_names, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_member_steps_after_the_ensemble(precision):
    cfg = configs.riemann(300, 0.45, 1.0, 1.0, 0.125, 0.1, 1.4, 1.67)
    cfg.precision = precision
    log(f"[batch member] precision={precision}")
    batch = mahyco_amd.Batch([cfg] * 7)
    single = mahyco_amd.Context(cfg)
    member = batch.problem(0)
    try:
        for n in (2, 6, 12):  # even: the problem keeps the ensemble's parity; the last in replays
            batch.run(n)
            member.run(n)
            single.run(2 * n)
            diff = [f"{f}[{k}]" for f, k in field_names(cfg) if not np.array_equal(member.get(f, k), single.get(f, k))]
            assert not diff, diff
            assert member.time_state().deltat_n == single.time_state().deltat_n
    finally:
        single.close()
        batch.close()
