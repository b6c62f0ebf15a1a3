"""Building the SELL copy of a small system (CPU, no GPU): short ranges, which a batch of few
rows is cut into, cost about what whole ones do.  (With a thread for every range they took
eight times as long, two copies a system in a mixed batch.)"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "npb-gpu_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_short_ranges_of_a_small_system(tmp_path):
    exe = tmp_path / "sell_build_time"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", CSRC,
                    os.path.join(ROOT, "tests", "c", "sell_build_time.cpp"),
                    os.path.join(CSRC, "tiled_layout.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    short, whole = map(float, out.split())
    assert short < 3 * whole, out
