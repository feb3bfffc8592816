"""The tuning steps of an ensemble time each kernel's own launches: with fixed
options the Lagrange kernel runs on y-first steps only and the dt reduction in the
first step, so a step that does not launch a kernel adds nothing to its times, and the
workgroup count kept is the one with the shortest mean of what was timed."""
import re
from collections import defaultdict

import pytest

import mahyco_amd
from mahyco_amd import configs

from gpu_helpers import log
from test_gpu_variants import env

pytestmark = pytest.mark.gpu

DT, NODE, CELL = 0, 1, 2  # kernel numbers of the tuner's report
CANDIDATES = [0, 1024, 2048, 4096, 8192]


@pytest.mark.parametrize("fixed", ["1", "0"], ids=["fixed", "run-time"])
def test_a_kernel_is_timed_where_it_runs(fixed, capfd):
    cfgs = configs.ensemble(n=5, side_min=64, side_max=400)
    log(f"[batch tuner] fixed options {fixed}")
    with env("MAHYCO_FIXED_OPTIONS", fixed), env("MAHYCO_DUAL_ROWS", "16"), env("MAHYCO_BATCH_VERBOSE", "1"):
        batch = mahyco_amd.Batch(cfgs)
        try:
            batch.run(10)  # two steps per candidate
        finally:
            batch.close()
    text = capfd.readouterr().err
    times = defaultdict(lambda: defaultdict(list))
    for k, c, ms in re.findall(r"kernel (\d+) blocks (\d+): ([\d.]+) ms", text):
        times[int(k)][int(c)].append(float(ms))
    kept = {int(k): int(c) for k, c in re.findall(r"kernel (\d+) -> (\d+)", text)}
    assert set(kept) == set(range(8)), text
    # (fixed options: every second step has a Lagrange kernel, the first a dt reduction)
    per = 1 if fixed == "1" else 2
    assert {c: len(t) for c, t in times[CELL].items()} == {c: per for c in CANDIDATES}, text
    assert sum(len(t) for t in times[DT].values()) == (1 if fixed == "1" else 10), text
    assert NODE not in times  # one form whatever the candidate
    for k, by in times.items():
        mean = {c: sum(t) / len(t) for c, t in by.items()}
        # (the report rounds to 1e-4 ms)
        assert mean[kept[k]] <= min(mean.values()) + 1.0e-4, (k, mean, kept[k])
