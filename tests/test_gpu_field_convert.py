"""Where the mixed form's fields are converted: on the device for pinned buffers from
2^17 values on, and for pageable ones from 2^21 (written) and 2^22 values (read) on; on
the host below.  Every value is exactly the FP32 rounding of what was written, subnormals,
infinities and signed zeros too, on both sides of each line and with either buffer."""
import ctypes
from contextlib import contextmanager

import numpy as np
import pytest

import mahyco_amd

from gpu_helpers import log
from test_gpu_fixed_options import problem

pytestmark = pytest.mark.gpu


@contextmanager
def buffers(n, pinned):
    """Two arrays of n values, from the HIP runtime the library runs on where pinned."""
    if not pinned:
        yield np.zeros(n), np.zeros(n)
        return
    L, p = mahyco_amd.library(), ctypes.c_void_p()
    assert L.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(16 * n), ctypes.c_uint(0)) == 0
    try:
        both = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_double)), shape=(2 * n,))
        yield both[:n], both[n:]
    finally:
        assert L.hipHostFree(p) == 0


@pytest.mark.parametrize("pinned", [True, False], ids=["pinned", "pageable"])
@pytest.mark.parametrize("nx,ny", [(511, 256), (512, 256), (2049, 1023), (2048, 1024), (2049, 2047), (2048, 2048)])
def test_round_trip(nx, ny, pinned):
    cfg = problem(1, nx, ny, "minmod", precision=1)
    log(f"[field convert] {nx}x{ny} pinned={pinned}")
    L, ptr = mahyco_amd.library(), ctypes.POINTER(ctypes.c_double)
    ctx = mahyco_amd.Context(cfg)
    rng = np.random.default_rng(11)
    try:
        for name in ("density", "velocity_y"):
            fid, n = ctx.field_id(name)
            with buffers(n + 1, pinned) as (v, got):
                v, got = v[1:], got[1:]  # one value off the start of the allocation
                v[:] = rng.uniform(-1.0, 1.0, n) * 10.0 ** rng.uniform(-44, 37, n)
                v[:6] = [0.0, -0.0, 1.0e-41, -1.4e-45, np.inf, -np.inf]
                got[:] = 0.0
                assert L.mhy_set_field(ctx.h, fid, v.ctypes.data_as(ptr), n) == 0
                assert L.mhy_get_field(ctx.h, fid, got.ctypes.data_as(ptr), n) == 0
                assert np.array_equal(got, v.astype(np.float32).astype(np.float64)), name
                assert np.array_equal(np.signbit(got), np.signbit(v)), name
    finally:
        ctx.close()
