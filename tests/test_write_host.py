"""The DPR4 writer's threads (tests/write_check.cpp): the same bytes for any
number of them, and a failing allocation reaches the caller."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_writer_threads_and_failing_allocations(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "write_check"
    subprocess.run([gxx, "-O1", "-g", "-std=c++17", "-pthread", str(ROOT / "tests" / "write_check.cpp"), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stderr[-500:])
    assert int(r.stdout) > 10
