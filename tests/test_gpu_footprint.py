"""Device memory.  A context fits wherever it would with one nodal remap per sweep, a
stored U_2 and the mixed / pure flags in two integers per cell: its buffers for the nodal
remap of both sweeps take more, and a device without room for them gets the same
context without U_2.  2047^2 cells: node arrays of 32 MiB, cell and face arrays just below."""
import numpy as np
import pytest
import torch

import mahyco_amd

from gpu_helpers import log
from test_gpu_fixed_options import problem

pytestmark = pytest.mark.gpu

MIB = 1 << 20


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
            return [ctx.get(n, k) for n, k in names], (free - torch.cuda.mem_get_info()[0]) / MIB
        finally:
            ctx.close()

    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    want, roomy = fields()
    room = needed(m, precision) + 24  # (the runtime's own)
    filler = []
    try:
        for _ in range(3):  # (the runtime hands memory of its own back on the way)
            more = torch.cuda.mem_get_info()[0] - room * MIB
            if more >= 4 * MIB:
                filler.append(torch.empty(more, dtype=torch.uint8, device="cuda"))
        free = torch.cuda.mem_get_info()[0]
        assert abs(free / MIB - room) <= 24
        got, tight = fields()
        log(f"[footprint] m={m} precision={precision}: {roomy:.0f} MiB, with {room} MiB free {tight:.0f} MiB")
        assert tight < roomy
        for (n, k), a, b in zip(names, got, want):
            assert np.array_equal(a, b), (n, k)
    finally:
        filler.clear()
        torch.cuda.empty_cache()


def test_field_access_allocates_nothing():
    """Reading and writing fields leaves the device's free memory as it is, also in the
    mixed form, whose values are widened and narrowed on the device."""
    cfg = problem(1, 1500, 1500, "minmod", 1)
    ctx = mahyco_amd.Context(cfg)
    try:
        ctx.run(1)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        rho = ctx.get("density")
        ctx.set("density", rho)
        ctx.get("velocity_x")
        assert torch.cuda.mem_get_info()[0] == free
    finally:
        ctx.close()
