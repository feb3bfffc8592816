"""Which sites the launch-shape tuner has, by options, and its results.  With fixed
options the nodal remap is one kernel for both sweeps, and the y-first Lagrange update
runs on strips or bands; with run-time options (another limiter, or
MAHYCO_FIXED_OPTIONS=0) the five nodal remaps along y and the separate Lagrange kernel
are timed.  Tuned runs are bitwise the untuned ones through the tuning steps and replays."""
import numpy as np
import pytest

import mahyco_amd
from mahyco_amd import abi, configs

from gpu_helpers import field_names, log
from test_gpu_variants import env

pytestmark = pytest.mark.gpu

ONE_SWEEP = {"tile", "wave", "walk", "tile32", "tile64"}


def _case(name):
    if name == "penteborne":
        return configs.riemann_perturbed(n=1024)
    cfg = configs.riemann(1024, 0.45, 1.0, 1.0, 0.125, 0.1, 1.4, 1.67)
    cfg.limiter = abi.LIM[name]
    return cfg


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("name,fixed", [("minmod", "1"), ("minmod", "0"), ("vanLeer", "1"), ("penteborne", "1"), ("penteborne", "0")])
def test_sites(name, fixed, precision):
    cfg = _case(name)
    cfg.precision = precision
    compiled = fixed == "1" and name != "vanLeer"
    log(f"[tuner sites] {name} fixed={fixed} precision={precision}")
    with env("MAHYCO_FIXED_OPTIONS", fixed):
        tuned = mahyco_amd.Context(cfg)
        with env("MAHYCO_AUTOTUNE", "0"):
            plain = mahyco_amd.Context(cfg)
    try:
        # two rounds over the candidates, two steps each
        steps = 4 * ((0 if compiled else 5) + 2 + (2 if cfg.pp != 1 else 0))
        tuned.run(steps - 1)
        plain.run(steps - 1)
        assert tuned.tuned_kernels() == ""
        for n in (1, 6):  # the last tuning step, then replays
            tuned.run(n)
            plain.run(n)
            diff = [f"{f}[{k}]" for f, k in field_names(cfg)
                    if not np.array_equal(tuned.get(f, k), plain.get(f, k), equal_nan=True)]
            assert not diff, diff
        choice = dict(s.split("=") for s in tuned.tuned_kernels().split())
        log(f"[tuner sites] {choice}")
        assert choice.pop("dual_y") in ({"both"} if compiled else ONE_SWEEP)
        assert choice.pop("sweep_y") in {"wave", "walk"}
        if cfg.pp != 1:
            assert choice.pop("lagrange_y") in ({"fused", "walk"} if compiled else {"fused", "separate"})
        assert not choice
    finally:
        tuned.close()
        plain.close()
