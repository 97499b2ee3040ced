"""The pool of idle capture streams (tests/pool_check.cpp), under TSan."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_idle_pool(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "pool_check"
    subprocess.run([gxx, "-O1", "-g", "-std=c++17", "-fsanitize=thread", "-pthread",
                    str(ROOT / "tests" / "pool_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])
