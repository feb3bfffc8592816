"""The sweeps compiled for fixed options (a classic limiter, second order,
...) against the same sweeps reading their options at run time
(MAHYCO_FIXED_OPTIONS=0): the same operations in the same order, so every
field is equal bit for bit.  Meshes with ragged strips and bands; each kind
of sweep (fused Lagrange, first, second, walking), both limiters, one to three
materials, both storage forms, PenteBorne, Eucclhyd with and without mixte."""
import numpy as np
import pytest

import mahyco_amd
from mahyco_amd import abi, configs

from oracle import refcpu

from gpu_helpers import MAT, compare_state, field_names, log
from test_gpu_variants import env

pytestmark = pytest.mark.gpu


def problem(m, nx, ny, limiter, precision=0, pp=0):
    if m == 1:
        c = configs.point_explosion(nx)
    elif m == 2:
        c = configs.riemann_perturbed(nx)
        c.pp = 0
    else:
        c = configs.triple_layout(nx, ny)
    c.nx, c.ny, c.limiter, c.precision, c.pp = nx, ny, abi.LIM[limiter], precision, pp
    return c


def eucclhyd(nx, ny, mixte):
    c = configs.default_config()
    c.schema, c.test_case, c.nbmat = abi.SCHEMA_EUCCLHYD, abi.CASE["BiSodCaseX"], 2
    c.nx, c.ny, c.dx, c.dy = nx, ny, 1.0 / 128, 1.0 / 128
    c.deltat_init, c.deltat_min = 1.0e-3, 1.0e-12
    c.limiter, c.pp, c.pp_mixte, c.limiter_pure = abi.LIM["superBee"], 1, mixte, abi.LIM["arithmeticG"]
    return c


def assert_equal_runs(make, names, chunks=(1, 2, 9)):
    ref = make()
    with env("MAHYCO_FIXED_OPTIONS", "0"):
        alt = make()
    try:
        for n in chunks:
            ref.run(n)
            alt.run(n)
            diff = [f"{f}[{k}]" for f, k in names if not np.array_equal(ref.get(f, k), alt.get(f, k), equal_nan=True)]
            assert not diff, diff
    finally:
        ref.close()
        alt.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("limiter", ["minmod", "superBee"])
@pytest.mark.parametrize("m,nx,ny", [(1, 121, 37), (2, 65, 26), (3, 60, 13)])
@pytest.mark.parametrize("kernels", [{}, {"MAHYCO_SWEEP_Y": "walk", "MAHYCO_LAG_Y": "separate"},
                                     {"MAHYCO_FUSE_LAGRANGE": "0"}], ids=["fused", "walk", "separate"])
def test_limited_slopes(m, nx, ny, limiter, precision, kernels):
    cfg = problem(m, nx, ny, limiter, precision)
    log(f"[fixed] m={m} {nx}x{ny} {limiter} precision={precision} {kernels}")

    def make():
        with env("MAHYCO_SWEEP_Y", kernels.get("MAHYCO_SWEEP_Y", "wave")), \
             env("MAHYCO_LAG_Y", kernels.get("MAHYCO_LAG_Y", "fused")), \
             env("MAHYCO_FUSE_LAGRANGE", kernels.get("MAHYCO_FUSE_LAGRANGE", "1")):
            return mahyco_amd.Context(cfg)
    assert_equal_runs(make, field_names(cfg))


@pytest.mark.parametrize("limiter", ["minmod", "superBee"])
@pytest.mark.parametrize("m,nx,ny", [(1, 61, 25), (2, 120, 37), (3, 119, 12)])
def test_penteborne(m, nx, ny, limiter):
    cfg = problem(m, nx, ny, limiter, pp=1)
    log(f"[fixed] PenteBorne m={m} {nx}x{ny} {limiter}")
    assert_equal_runs(lambda: mahyco_amd.Context(cfg), field_names(cfg), chunks=(1, 2, 60))


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("m,nx,ny", [(1, 2, 2), (1, 250, 26), (2, 251, 27), (3, 253, 3), (1, 8, 55), (2, 9, 29)])
def test_third_order(m, nx, ny, precision):
    """Tiles of 250 columns and of 8 columns x 26 rows; FP64 also against the oracle."""
    cfg = problem(m, max(nx, 8), ny, "superBee", precision)
    cfg.nx, cfg.projection_order = nx, 3
    log(f"[fixed] order 3 m={m} {nx}x{ny} precision={precision}")
    assert_equal_runs(lambda: mahyco_amd.Context(cfg), field_names(cfg))
    if precision == 0:
        ctx, orc = mahyco_amd.Context(cfg), refcpu.Oracle(cfg)
        try:
            for n in (1, 2, 9):
                ctx.run(n)
                orc.step(n)
                _, name, bitwise = compare_state(ctx, orc, cfg)
                assert bitwise, name
        finally:
            ctx.close()
            orc.close()


@pytest.mark.parametrize("mixte", [0, 1])
def test_eucclhyd(mixte):
    cfg = eucclhyd(125, 27, mixte)
    log(f"[fixed] Eucclhyd mixte={mixte}")
    names = [("density", 0), ("energy", 0), ("cell_velocity_x", 0), ("cell_velocity_y", 0), ("mixte", 0), ("pure", 0)]
    names += [(n, k) for n in ("fracvol", "density_env", "energy_env") for k in range(2)]
    assert_equal_runs(lambda: mahyco_amd.Context(cfg), names, chunks=(1, 2, 60))


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("limiters", [("minmod", "minmod"), ("superBee", "superBee"), ("minmod", "superBee")])
def test_ensemble(limiters, precision):
    """One limiter for all problems (fixed), or two (run-time sweeps)."""
    cfgs = [problem(2, 65 + 40 * i, 40 - 11 * i, lim, precision) for i, lim in enumerate(limiters)]
    log(f"[fixed] ensemble {limiters} precision={precision}")
    both = mahyco_amd.Batch(cfgs)
    with env("MAHYCO_FIXED_OPTIONS", "0"):
        alt = mahyco_amd.Batch(cfgs)
    try:
        for n in (1, 14):  # tuning steps, then graph replays
            both.run(n)
            alt.run(n)
            for i in range(len(cfgs)):
                a, b = both.problem(i), alt.problem(i)
                for f, k in [("density", 0), ("energy", 0), ("velocity_x", 0), ("velocity_y", 0)] + [(n2, 1) for n2 in MAT]:
                    assert np.array_equal(a.get(f, k), b.get(f, k), equal_nan=True), (i, f, k)
    finally:
        both.close()
        alt.close()
