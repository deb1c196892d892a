"""The deposit's fixed-point arithmetic (aprl_amd/csrc/fixedsum.hpp), compiled
for the host and compared with 128-bit integers (tests/cpp/fixedsum_check.cpp):
a tap is its product rounded once, and the quintic's weights applied to raw
sums lose nothing."""
import os
import subprocess

import harness as H


def test_fixed_point_sums(tmp_path):
    exe = str(tmp_path / "fixedsum_check")
    cmd = ["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas",
           "-I", os.path.join(H.ROOT, "aprl_amd", "csrc"),
           os.path.join(H.ROOT, "tests", "cpp", "fixedsum_check.cpp"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    run = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and "fixed-point check passed" in run.stdout, run.stdout + run.stderr[-2000:]
