"""Device memory.  A context fits wherever it would with one nodal remap per sweep, a
stored U_2 and the mixed / pure flags in two integers per cell: its buffers for the nodal
remap of both sweeps take more, and a device without room for them gets the same
context without U_2.  2047^2 cells: node arrays of 32 MiB, cell and face arrays just below."""
import ctypes

import numpy as np
import pytest

import mahyco_amd

from gpu_helpers import log
from test_gpu_fixed_options import problem

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def free_bytes():
    """Free device memory, from the HIP runtime the library runs on."""
    L, free, total = mahyco_amd.library(), ctypes.c_size_t(), ctypes.c_size_t()
    assert L.hipDeviceSynchronize() == 0
    assert L.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def needed(m, precision):
    """MiB of that layout."""
    nc = 3 * m + 1
    fp64 = 1 + 2 * m + 1 + 3 * nc + 3 + m + 3 + 1  # vol, f_k, M_k, M, U, V_L and centroid, G, UD1, XL2
    bulk = 2 * (6 + 5 * m) + 4 + m + 1            # states, velocities, mu_k, node mass
    return 32 * fp64 + (16 if precision else 32) * bulk + 2 * 16 + 4  # + flags, stored-material flags


@pytest.mark.parametrize("m,precision", [(2, 1), (3, 0)])
def test_context_fits_a_nearly_full_device(m, precision):
    cfg = problem(m, 2047, 2047, "minmod", precision)
    names = [("density", 0), ("energy", 0), ("velocity_x", 0), ("pseudo", 0), ("fracvol", m - 1)]

    def fields():
        ctx = mahyco_amd.Context(cfg)
        try:
            ctx.run(40)  # the tuning steps, then replays
            return [ctx.get(n, k) for n, k in names], (free - free_bytes()) / MIB
        finally:
            ctx.close()

    free = free_bytes()
    want, roomy = fields()
    room = needed(m, precision) + 24  # (the runtime's own)
    filler = []
    try:
        for _ in range(3):  # (the runtime hands memory of its own back on the way)
            more = free_bytes() - room * MIB
            if more >= 4 * MIB:
                block = ctypes.c_void_p()
                assert mahyco_amd.library().hipMalloc(ctypes.byref(block), ctypes.c_size_t(more)) == 0
                filler.append(block)
        free = free_bytes()
        assert abs(free / MIB - room) <= 24
        got, tight = fields()
        log(f"[footprint] m={m} precision={precision}: {roomy:.0f} MiB, with {room} MiB free {tight:.0f} MiB")
        assert tight < roomy
        for (n, k), a, b in zip(names, got, want):
            assert np.array_equal(a, b), (n, k)
    finally:
        for block in filler:
            assert mahyco_amd.library().hipFree(block) == 0


def test_field_access_allocates_nothing():
    """Reading and writing fields leaves the device's free memory as it is, also in the
    mixed form, whose values are widened and narrowed on the device."""
    cfg = problem(1, 1500, 1500, "minmod", 1)
    ctx = mahyco_amd.Context(cfg)
    try:
        ctx.run(1)
        free = free_bytes()
        rho = ctx.get("density")
        ctx.set("density", rho)
        ctx.get("velocity_x")
        assert free_bytes() == free
    finally:
        ctx.close()
