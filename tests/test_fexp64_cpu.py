"""exp, tanh and the logistic function of synaptik_amd/csrc/fexp64.h, built for the host with g++
and compared with the library's binary64 functions rounded once to binary32. The device kernels
compile the same header (their quotient alone is formed differently, see quotient_12)."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


def test_binary64_evaluations_round_like_the_library(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "fexp64_harness"
    subprocess.run([gxx, "-O2", "-ffp-contract=off", "-o", str(exe),
                    str(HERE / "fexp64_harness.cpp"), "-lm"], check=True)
    out = subprocess.run([str(exe), "389"], check=True, capture_output=True, text=True)
    lines = [list(map(int, line.split())) for line in out.stdout.splitlines()]
    for n, differing, max_ulp in lines[:3]:
        assert n > 10_000_000
        # a few units of 2^-52 against ties of binary32: about one argument in 10^7
        assert max_ulp <= 1 and differing <= n // 1_000_000
    assert lines[3] == [1]  # NaNs and the signs of zeros
