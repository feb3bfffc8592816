"""The picking rule of the ensembles' workgroup tuner, built for the host: the
candidate with the shortest mean over its own launches, also for a kernel that
only every second step launches."""
import os
import subprocess

import pytest

from mahyco_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("bt") / "block_tuner")
    cmd = [build.hipcc(), "-x", "hip", "--cuda-host-only", "-O2", "-std=c++17",
           "-I", os.path.join(os.path.dirname(HERE), "mahyco_amd", "csrc"),
           os.path.join(HERE, "host", "block_tuner.cc"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


@pytest.mark.parametrize("every", [(4, 3, 5, 6), (1, 2, 3, 4), (4, 3, 2, 1)])
@pytest.mark.parametrize("second", [(3, 2, 4, 5), (1, 2, 3, 4), (9, 8, 7, 5)])
def test_the_fastest_candidate_is_kept(driver, every, second):
    r = subprocess.run([driver, *map(str, every + second)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    picks, samples = ([int(v) for v in line.split()] for line in r.stdout.splitlines())
    # (a kernel timed with the default only keeps the default)
    assert picks == [every.index(min(every)), second.index(min(second)), 0]
    assert samples == [1, 1, 1, 1]
