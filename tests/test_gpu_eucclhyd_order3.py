"""Third-order Eucclhyd sweeps of a conservative projection (remap vectors of 6, 9 and
12 components, up to 76 KiB of LDS per tile): field by field against the CPU oracle,
bitwise, on meshes of whole, ragged and single tiles."""
import numpy as np
import pytest

import mahyco_amd
from mahyco_amd import abi
from oracle import refcpu

from gpu_helpers import log
from test_gpu_eucclhyd import _fields, _from

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("base,kw", [
    ("SOD_X_Mono_mat_proj_ordre_3", dict(nx=250, ny=26, dx=1.0 / 256)), ("SOD_Y_Mono_mat_proj_ordre_3", dict(nx=9, ny=53, dy=1.0 / 64)),
    ("SOD_X_bi_mat_proj_ordre_3", dict(nx=251, ny=27, dx=1.0 / 256)), ("SOD_Y_bi_mat_proj_ordre_3", dict(nx=8, ny=52, dy=1.0 / 64)),
    ("POINT_TRIPLE_proj_ordre_3", dict(nx=140, ny=60, dx=0.0005, dy=0.0005)), ("POINT_TRIPLE_proj_ordre_3", dict())])
def test_conservative_third_order(base, kw):
    cfg = _from(base, **kw)
    cfg.projection_conservative = 1
    log(f"[euc order 3] conservative m={cfg.nbmat} {cfg.nx}x{cfg.ny}")
    assert cfg.projection_order == 3
    gpu, orc = mahyco_amd.Context(cfg), refcpu.Oracle(cfg)
    try:
        for n in (1, 2, 40):
            gpu.run(n)
            assert orc.step(n) == abi.MHY_OK
            diff = [f"{f}[{k}]" for f, k in _fields(cfg) if not np.array_equal(gpu.get(f, k), orc.get(f, k), equal_nan=True)]
            assert not diff, diff
    finally:
        gpu.close()
        orc.close()
