"""The pickers of the kernels with fixed options: a kernel for every kind that is
compiled, null for every other limiter and kind (the caller then takes the run-time
form or fails), never another sweep's kernel.  Host functions: nothing is launched."""
import ctypes

import pytest

import mahyco_amd
from mahyco_amd.abi import LIM

# symbol, direction argument (None: the picker has none), first kind compiled
P = {"sweepFixedX fp64": ("_ZN3mhy11sweepFixedXIdEEPFvNS_3KPTIT_EEEiii", None, 0),
     "sweepFixedX mixed": ("_ZN3mhy11sweepFixedXIfEEPFvNS_3KPTIT_EEEiii", None, 0),
     "sweepFixedY fp64": ("_ZN3mhy11sweepFixedYIdEEPFvNS_3KPTIT_EEEiii", None, 0),
     "sweepFixedY mixed": ("_ZN3mhy11sweepFixedYIfEEPFvNS_3KPTIT_EEEiii", None, 0),
     "sweepFixedWalk fp64": ("_ZN3mhy14sweepFixedWalkIdEEPFvNS_3KPTIT_EEEiii", None, 0),
     "sweepFixedWalk mixed": ("_ZN3mhy14sweepFixedWalkIfEEPFvNS_3KPTIT_EEEiii", None, 0),
     "sweepFixedXBatch fp64": ("_ZN3mhy16sweepFixedXBatchIdEEPFvNS_12BatchLaunchTIT_EEEiii", None, 0),
     "sweepFixedXBatch mixed": ("_ZN3mhy16sweepFixedXBatchIfEEPFvNS_12BatchLaunchTIT_EEEiii", None, 0),
     "sweepFixedYBatch fp64": ("_ZN3mhy16sweepFixedYBatchIdEEPFvNS_12BatchLaunchTIT_EEEiii", None, 1),
     "sweepFixedYBatch mixed": ("_ZN3mhy16sweepFixedYBatchIfEEPFvNS_12BatchLaunchTIT_EEEiii", None, 1),
     "sweepFixedPP x": ("_ZN3mhy12sweepFixedPPEbiii", True, 0),
     "sweepFixedPP y": ("_ZN3mhy12sweepFixedPPEbiii", False, 1)}


def picker(symbol, direction):
    fn = getattr(mahyco_amd.library(), symbol)
    fn.restype = ctypes.c_void_p
    if direction is None:
        fn.argtypes = [ctypes.c_int] * 3
        return fn
    fn.argtypes = [ctypes.c_bool] + [ctypes.c_int] * 3
    return lambda lim, m, kind: fn(direction, lim, m, kind)


@pytest.mark.parametrize("name", sorted(P))
def test_picker(name):
    symbol, direction, first = P[name]
    pick = picker(symbol, direction)
    seen = set()
    for lim in LIM:
        for m in (1, 2, 3):
            for kind in range(-1, 4):
                k = pick(LIM[lim], m, kind)
                assert bool(k) == (lim in ("minmod", "superBee") and first <= kind <= 2), (lim, m, kind)
                if k:
                    assert k not in seen, (lim, m, kind)  # each its own kernel
                    seen.add(k)


@pytest.mark.parametrize("symbol", ["_ZN3mhy12sweepFixedO3IdEEPFvNS_3KPTIT_EEEbii", "_ZN3mhy12sweepFixedO3IfEEPFvNS_3KPTIT_EEEbii"])
def test_third_order_picker(symbol):
    fn = getattr(mahyco_amd.library(), symbol)
    fn.restype, fn.argtypes = ctypes.c_void_p, [ctypes.c_bool, ctypes.c_int, ctypes.c_int]
    picked = [fn(xd, m, kind) for xd in (True, False) for m in (1, 2, 3) for kind in (1, 2)]
    assert all(picked) and len(set(picked)) == 12
    assert not any(fn(xd, m, kind) for xd in (True, False) for m in (1, 2, 3) for kind in (-1, 0, 3))
