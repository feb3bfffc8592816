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
def test_both_sweeps_in_one_kernel(m, limiter, pp, nx, ny, precision):
    cfg = problem(m, max(nx, 8), ny, limiter, precision, pp)
    cfg.nx = nx
    log(f"[dual] m={m} {nx}x{ny} {limiter} pp={pp} precision={precision}")
    both = mahyco_amd.Context(cfg)
    with env("MAHYCO_DUAL_Y", "wave"):
        one = mahyco_amd.Context(cfg)
    try:
        for eager, n in ((True, 1), (True, 2), (False, 30)):
            for ctx in (both, one):
                ctx.step(n) if eager else ctx.run(n)
            diff = [f"{f}[{k}]" for f, k in field_names(cfg)
                    if not np.array_equal(both.get(f, k), one.get(f, k), equal_nan=True)]
            assert not diff, diff
    finally:
        both.close()
        one.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_ensemble_equals_single_problems(precision):
    cfgs = [problem(2, 40 + 21 * i, 70 - 13 * i, "minmod", precision) for i in range(4)]
    log(f"[dual] ensemble precision={precision}")
    batch = mahyco_amd.Batch(cfgs)
    with env("MAHYCO_DUAL_Y", "wave"):
        singles = [mahyco_amd.Context(c) for c in cfgs]
    try:
        for n in (1, 14):
            batch.run(n)
            for i, s in enumerate(singles):
                s.run(n)
                p = batch.problem(i)
                for f in ("velocity_x", "velocity_y", "density", "energy"):
                    assert np.array_equal(p.get(f), s.get(f)), (i, f)
    finally:
        batch.close()
        for s in singles:
            s.close()
