"""Field access of the mixed form, whose values the device widens to FP64 and
narrows, and of the mixed / pure flags, kept in one byte: every value is exactly the FP32 rounding of what
was written, the flags equal the oracle's.  Lengths around a block of 256."""
import numpy as np
import pytest

import mahyco_amd
from oracle import refcpu

from gpu_helpers import log
from test_gpu_fixed_options import problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(2, 2), (8, 32), (257, 3), (16, 16)])
def test_mixed_fields_round_trip(nx, ny):
    cfg = problem(2, 16, 16, "minmod", precision=1)
    cfg.nx, cfg.ny = nx, ny
    log(f"[fields] {nx}x{ny}")
    ctx = mahyco_amd.Context(cfg)
    rng = np.random.default_rng(7)
    try:
        for name, k in (("density", 0), ("velocity_x", 0), ("energy_env", 1)):
            n = ctx.field_id(name, k)[1]
            v = rng.uniform(-1.0, 1.0, n) * 10.0 ** rng.uniform(-30, 30, n)
            v[:2] = [0.0, -0.0]
            ctx.set(name, v, k)
            got = ctx.get(name, k)
            assert np.array_equal(got, v.astype(np.float32).astype(np.float64)), name
            assert np.array_equal(np.signbit(got), np.signbit(v)), name
        for name in ("fracvol", "mass_env"):  # FP64 in both forms
            v = rng.uniform(0.0, 1.0, nx * ny)
            ctx.set(name, v)
            assert np.array_equal(ctx.get(name), v), name
    finally:
        ctx.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_flags(precision):
    cfg = problem(2, 51, 47, "superBee", precision)
    ctx, orc = mahyco_amd.Context(cfg), refcpu.Oracle(cfg)
    try:
        for n in (0, 1, 5):
            ctx.step(n)
            orc.step(n)
            for name in ("mixte", "pure"):
                assert np.array_equal(ctx.get(name), orc.get(name)), (n, name)
    finally:
        ctx.close()
        orc.close()
