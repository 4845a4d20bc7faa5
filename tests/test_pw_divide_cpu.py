"""The chain interpreter's division of ordinals by the row width (synaptik_amd/csrc/pw_divide.h),
built for the host and compared with '/'."""
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


def test_ordinals_divide_exactly(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "pw_divide_harness"
    subprocess.run([gxx, "-O2", "-std=c++17", "-o", str(exe), str(HERE / "pw_divide_harness.cpp")],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True).stdout.strip()
    assert out == "ok", out
