"""The few-pair sums of the register time kernels (few_pairs and its layouts
in fastddm_amd/csrc/fddm_time_wave.hpp) on the CPU: compiled for the host,
with arrays that check every index, so that no lane reads outside the slice of
last samples its layout allocates."""

import os
import subprocess

import pytest

from fastddm_amd import _build

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "fastddm_amd", "csrc")


@pytest.mark.skipif(not os.path.isfile(_build.hipcc()), reason="hipcc not available")
def test_reads_stay_in_the_slice(tmp_path):
    exe = str(tmp_path / "ranges")
    subprocess.run([_build.hipcc(), "--offload-host-only", "-x", "hip", "-std=c++17", "-O1", "-I", CSRC,
                    os.path.join(HERE, "few_pairs_ranges.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True, timeout=180)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
    lines = res.stdout.split("\n")[:-1]
    assert len(lines) == 6
    for line in lines:
        assert line.endswith("out_of_range=0 wrong=0"), res.stdout
