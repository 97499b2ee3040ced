"""The pre-pass's verdict on meshlets that end early, by what it meets first:
strip lengths that do not add up (5) or a field past the range (2)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_meshlets_cut_after_every_bit(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path / "scan_check"
    subprocess.run([gxx, "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=undefined", str(ROOT / "tests" / "scan_check.cpp"), "-o", str(exe)],
                   check=True)

    def verdicts(length):
        r = subprocess.run([str(exe), str(length)], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        return [int(x) for x in r.stdout.split()]
    ok = verdicts(1)
    assert ok[-1] == 0 and set(ok[:-1]) == {2}     # every cut loses a bit of some field
    # a length that does not add up is reported as such wherever the range ends, also inside the header
    for length in (0, 2, 300):
        assert set(verdicts(length)) == {5}
