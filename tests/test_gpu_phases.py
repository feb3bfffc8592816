"""Whole steps fold the time step into the node update; the phase-level calls
(mhy_compute_dt, mhy_lagrange, mhy_remap_sweep, ...) form it in a kernel of
its own; a step also leaves the next one's CFL minimum, which a field written
from the host invalidates.  All must give the oracle's state: the operations are the same in
the same order, so FP64 fields are equal bit for bit.  Meshes at the edges of
the node layout: no interior row or column, one block of a row and one node
more, boundary nodes filling whole blocks."""
import numpy as np
import pytest

import mahyco_amd
from mahyco_amd import configs
from oracle import refcpu

from gpu_helpers import compare_state, log
from test_gpu_variants import env

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


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("name,factor", [("velocity_x", 40.0), ("sound_speed", 0.5), ("pressure", 3.0)])
@pytest.mark.parametrize("rows", [2, 16])  # bands of 16 rows leave the next step's CFL minimum
def test_time_step_after_a_field_is_written(rows, name, factor, precision):
    """The time step and the pressure cap of the next step come from the new
    field: the same as in a context that reduces them in every step."""
    cfg = configs.point_explosion(96)
    cfg.ny, cfg.precision = 50, precision
    log(f"[phases] set {name} precision={precision}")
    with env("MAHYCO_DUAL_ROWS", str(rows)):
        kept, reduced = mahyco_amd.Context(cfg), mahyco_amd.Context(cfg)
    run = mahyco_amd.library().mhy_run
    try:
        for n in (1, 300, 3):  # past the ramp: the CFL condition binds
            kept.run(n)
            for _ in range(n):
                step_by_phases(reduced)
            for ctx in (kept, reduced):
                ctx.set(name, ctx.get(name) * factor)
            status = run(kept.h, 1)  # eager, the reduction kernel
            step_by_phases(reduced)
            if status == 0:
                status = run(kept.h, 4)  # replays
                for _ in range(4):
                    step_by_phases(reduced)
            # (a state the scheme cannot follow ends in NaN, in both)
            assert kept.time_state().status == reduced.time_state().status == status
            for f in ("density", "energy", "velocity_x", "velocity_y", "pseudo"):
                assert np.array_equal(kept.get(f), reduced.get(f), equal_nan=True), f
            assert kept.time_state().deltat_n == reduced.time_state().deltat_n
            if status != 0:
                break
            for ctx in (kept, reduced):  # kept: the accumulators of the replay, a finalize kernel
                step_by_phases(ctx)
            assert np.array_equal(kept.get("energy"), reduced.get("energy"))
    finally:
        kept.close()
        reduced.close()
