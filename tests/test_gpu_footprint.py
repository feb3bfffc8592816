"""Device memory of a context: no more than with one nodal remap per sweep, a stored
U_2 and the mixed / pure flags in two integers per cell, so that every mesh which fits
the card that way still does.  2047^2 cells: node arrays of 32 MiB, cell and face arrays
just below."""
import pytest
import torch

import mahyco_amd

from gpu_helpers import log
from test_gpu_fixed_options import problem

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def arrays(m, pp):
    """FP64 and bulk arrays of that layout."""
    nc = 3 * m + 1
    fp64 = 1 + 2 * m + 1 + 3 * nc + 3 + (1 if pp else 0) + m + 3 + 1  # vol, f_k, M_k, M, U, V_L .., q_L, G, UD1, XL2
    bulk = 2 * (6 + 5 * m) + 4 + m + 1                               # states, velocities, mu_k, node mass
    return fp64, bulk


@pytest.mark.parametrize("m,limiter,precision,pp", [(1, "minmod", 0, 0), (1, "minmod", 1, 0), (1, "vanLeer", 0, 0),
                                                    (2, "superBee", 0, 1), (2, "minmod", 1, 0), (3, "minmod", 0, 0)])
def test_context_is_no_larger(m, limiter, precision, pp):
    mahyco_amd.Context(problem(m, 64, 64, limiter, precision, pp)).close()  # (the library's own set-up)
    cfg = problem(m, 2047, 2047, limiter, precision, pp)
    fp64, bulk = arrays(m, pp)
    allowed = 32 * fp64 + (16 if precision else 32) * bulk + 2 * 16 + 4 + 4  # + flags, stored-material flags, scalars
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    ctx = mahyco_amd.Context(cfg)
    try:
        ctx.run(2)
        taken = (free - torch.cuda.mem_get_info()[0]) / MIB
        log(f"[footprint] m={m} {limiter} precision={precision} pp={pp}: {taken:.0f} MiB, allowed {allowed}")
        assert 0.8 * allowed < taken <= allowed
    finally:
        ctx.close()


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
