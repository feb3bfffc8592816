"""The nodal remap of both sweeps in one kernel against one kernel per sweep
(MAHYCO_DUAL_Y=wave): the same operations on the same operands, so every
field is equal bit for bit.  Node columns around the 59 and 60 updated by a
wave, node rows around the band heights, the smallest meshes; one to three
materials, both limiters, both storage forms, both sweep orders (every
second step), eager steps, graph replays and ensembles."""
import numpy as np
import pytest

import mahyco_amd

from gpu_helpers import field_names, log
from test_gpu_fixed_options import problem
from test_gpu_variants import env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 9), (57, 5), (58, 4), (59, 3), (60, 7), (61, 8), (117, 15), (118, 33), (119, 2)])
@pytest.mark.parametrize("m,limiter,pp", [(1, "minmod", 0), (2, "superBee", 0), (2, "superBee", 1), (3, "minmod", 0)])
@pytest.mark.parametrize("rows", [2, 16])  # without and with the next step's CFL reduction
def test_both_sweeps_in_one_kernel(rows, m, limiter, pp, nx, ny, precision):
    cfg = problem(m, max(nx, 8), ny, limiter, precision, pp)
    cfg.nx = nx
    log(f"[dual] rows={rows} m={m} {nx}x{ny} {limiter} pp={pp} precision={precision}")
    with env("MAHYCO_DUAL_ROWS", str(rows)):
        both = mahyco_amd.Context(cfg)
    with env("MAHYCO_DUAL_Y", "wave"):
        one = mahyco_amd.Context(cfg)
    try:
        for eager, n in ((True, 1), (True, 2), (False, 30)):
            for ctx in (both, one):
                ctx.step(n) if eager else ctx.run(n)
            assert both.time_state().deltat_n == one.time_state().deltat_n
            diff = [f"{f}[{k}]" for f, k in field_names(cfg)
                    if not np.array_equal(both.get(f, k), one.get(f, k), equal_nan=True)]
            assert not diff, diff
    finally:
        both.close()
        one.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("rows", [4, 16])
def test_ensemble_equals_single_problems(rows, precision):
    cfgs = [problem(2, 40 + 21 * i, 70 - 13 * i, "minmod", precision) for i in range(4)]
    log(f"[dual] ensemble rows={rows} precision={precision}")
    with env("MAHYCO_DUAL_ROWS", str(rows)):
        batch = mahyco_amd.Batch(cfgs)
    with env("MAHYCO_DUAL_Y", "wave"):
        singles = [mahyco_amd.Context(c) for c in cfgs]
    try:
        for n in (1, 14, 4, 4):
            batch.run(n)
            for i, s in enumerate(singles):
                s.run(n)
                p = batch.problem(i)
                for f in ("velocity_x", "velocity_y", "density", "energy"):
                    assert np.array_equal(p.get(f), s.get(f)), (i, f)
            # a field written from the host: the problem's dt is reduced again
            for ctx in (batch.problem(1), singles[1]):
                ctx.set("sound_speed", ctx.get("sound_speed") * 2.0)
    finally:
        batch.close()
        for s in singles:
            s.close()
