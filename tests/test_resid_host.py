"""The residual lanes and code chains of the two-pass decode, compiled for
the host under ASan and UBSan with exactly sized buffers, against its axis
lanes: golden and hand-built streams, sizes around the 32-entry chunks, 16-bit
codes, and outliers whose codewords pass 32 bits."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from tests.conftest import encode_with_oracle, ribbon, small_meshes

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def resid_check(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("resid") / "resid_check"
    subprocess.run([gxx, "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=undefined", str(ROOT / "tests" / "resid_check.cpp"), "-o", str(exe)],
                   check=True)
    return exe


def spiky(n):
    """A ribbon of 2 x n vertices with far outliers: long unary prefixes."""
    V, T = ribbon(n)
    V[::37, 2] += 40.0
    return V, T


def streams(kind):
    from tests.test_oracle import hand_stream_fifo, hand_stream_small
    if kind == "golden":
        return [z["data"].tobytes() for p in sorted((ROOT / "tests" / "golden").glob("*_*.npz"))
                if not p.stem.startswith("pdlt_") for z in [np.load(p)] if "data" in z] \
            + [hand_stream_small()[0], hand_stream_fifo()[0]]
    if kind == "small":
        return [encode_with_oracle(V, T, pred=pred)[1] for _, V, T in small_meshes()
                for pred in ("canonical", ([[33, 32, -33], [31, 34, -33], [32, 32, -32]], [5, 5, 5]))]
    if kind == "spiky":
        return [encode_with_oracle(*spiky(300), precision_error=e)[1] for e in (1e-2, 2e-3)]
    # one meshlet of 2 n vertices: chunks of 32 entries end at, before and after 2 n
    return [encode_with_oracle(*ribbon(n))[1] for n in (2, 3, 4, 5, 15, 16, 17, 31, 32, 33, 48, 64, 96, 127, 128)]


@pytest.mark.parametrize("kind", ["golden", "small", "spiky", "chunk_edges"])
def test_residual_lanes_match_axis_lanes(resid_check, tmp_path, kind):
    compared = 0
    for data in streams(kind):
        src = tmp_path / "s.dpr4"
        src.write_bytes(data)
        r = subprocess.run([str(resid_check), str(src)], capture_output=True, text=True)
        assert r.returncode == 0, (r.returncode, r.stderr[-2000:])
        compared += int(r.stdout.split()[1])
    assert compared > 0
