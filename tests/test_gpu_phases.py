"""Whole steps fold the time step into the node update; the phase-level calls
(mhy_compute_dt, mhy_lagrange, mhy_remap_sweep, ...) form it in a kernel of
its own.  Both must give the oracle's state: the operations are the same in
the same order, so FP64 fields are equal bit for bit.  Meshes at the edges of
the node layout: no interior row or column, one block of a row and one node
more, boundary nodes filling whole blocks."""
import pytest

import mahyco_amd
from mahyco_amd import configs
from oracle import refcpu

from gpu_helpers import compare_state, log

pytestmark = pytest.mark.gpu


def step_by_phases(ctx):
    L = mahyco_amd.library()
    for call, args in ((L.mhy_compute_dt, ()), (L.mhy_lagrange, ()), (L.mhy_prepare_remap, ()),
                       (L.mhy_remap_sweep, (1,)), (L.mhy_remap_sweep, (2,)), (L.mhy_remap_final, ()),
                       (L.mhy_end_iteration, ())):
        assert call(ctx.h, *args) == 0


@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 2), (2, 3), (200, 5), (256, 3), (257, 4), (258, 2), (5, 130)])
def test_steps_and_phases_equal_oracle(nx, ny):
    cfg = configs.point_explosion(64)
    cfg.nx, cfg.ny = nx, ny
    log(f"[phases] {nx}x{ny}")
    whole, parts, orc = mahyco_amd.Context(cfg), mahyco_amd.Context(cfg), refcpu.Oracle(cfg)
    try:
        for n in (1, 1, 5):
            whole.run(n)
            orc.step(n)
            for _ in range(n):
                step_by_phases(parts)
            for ctx in (whole, parts):
                _, name, bitwise = compare_state(ctx, orc, cfg)
                assert bitwise, name
            assert whole.time_state().deltat_n == parts.time_state().deltat_n == orc.time_state().deltat_n
    finally:
        whole.close()
        parts.close()
        orc.close()
