"""The PDLT v5 decode with code waves, compiled for the host under ASan and
UBSan with exactly sized buffers, against the oracle: sizes around the
32-entry chunks and the 8-entry groups of the chain, the three axis coders,
strips past 257 triangles, both chains."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from oracle import pdlt_oracle as PO
from tests.conftest import ribbon, small_meshes
from tests.test_pdlt_host import GOLD, long_strip_stream

ROOT = Path(__file__).resolve().parents[1]
SIZES = {0, 1, 7, 8, 9, 31, 32, 33, 255, 256}   # n_int to be met


@pytest.fixture(scope="module")
def code_check(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("code") / "pdlt_code_check"
    subprocess.run([gxx, "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=undefined", "-ffp-contract=off", "-pthread",
                    str(ROOT / "tests" / "pdlt_code_check.cpp"), "-o", str(exe)], check=True)
    return exe


def band(n, spike=0.0):
    """n vertices in a zigzag strip of n - 2 triangles: one meshlet whose
    vertices are all interior."""
    rng = np.random.default_rng(n)
    i = np.arange(n)
    V = np.stack([0.05 * i, 0.1 * (i & 1), 0.05 * rng.standard_normal(n)], 1)
    V[::37, 2] += spike
    T = np.array([(k, k + 1, k + 2) if k % 2 == 0 else (k + 1, k, k + 2) for k in range(n - 2)])
    return V, T


def prepared(V, T, **kw):
    from meshpress_amd.encoder.prep import prepare
    p = prepare(V, T, **kw)
    d = dict(p)
    d["plans"] = p["native"].export_plans()
    return d


def streams(kind):
    from meshpress_amd import workloads as w
    from meshpress_amd.encoder.paradelta_v5 import encode_v5
    if kind == "golden":
        return [np.load(p)["data"].tobytes() for p in GOLD]
    if kind == "meshes":
        out = [encode_v5(V, T) for _, V, T in small_meshes()]
        out += [encode_v5(*w.displaced_torus(40, 16, 1.0, 0.3, 0.05, 4, 5), max_verts=mv, max_tris=mt)
                for mv, mt in ((8, 6), (64, 96), (256, 400))]
        return out + [encode_v5(*w.displaced_torus(400, 3, 1.0, 0.1, 0.02, 4, 5), max_tris=400),
                      long_strip_stream(400)]
    if kind == "sizes":
        return [encode_v5(*band(n)) for n in (3, 4, 7, 8, 9, 15, 16, 17, 31, 32, 33, 64, 255, 256)]
    # coders: 0 fixed width, 1 Rice, 2 Exp-Golomb; outliers pass 32-bit codewords
    V, T = band(200, spike=3.0)
    return [PO.encode_v5(prepared(V, T, precision_error=e), force_tags=lambda m, tag=tag: [tag] * 3)
            for tag in (0, 1, 2) for e in (1e-2, 2e-4)] + [
            PO.encode_v5(prepared(*ribbon(300)), force_tags=lambda m: [m % 3, (m + 1) % 3, (m + 2) % 3])]


def test_code_waves_match_the_oracle(code_check, tmp_path):
    met = set()
    for kind in ("golden", "meshes", "sizes", "coders"):
        for i, data in enumerate(streams(kind)):
            src, fv, ft = (tmp_path / n for n in ("s.pdlt", "v.f32", "t.u32"))
            src.write_bytes(data)
            Vo, To = PO.decode_v5(data)
            V32, _ = PO.decode_v5(data, chain="f32")
            for gs, lds, chain32, tg, staged in ((16, 20480, 0, 4, 1), (1, 4096, 1, 1, 0), (3, 12288, 1, 64, 1),
                                                 (2, 65536, 0, 2, 0)):
                r = subprocess.run([str(code_check), str(src), str(fv), str(ft)] +
                                   [str(x) for x in (gs, lds, chain32, tg, staged)],
                                   capture_output=True, text=True)
                assert r.returncode == 0, (kind, i, r.returncode, r.stderr[-2000:])
                V = np.fromfile(fv, np.float32).reshape(-1, 3)
                T = np.fromfile(ft, np.uint32).reshape(-1, 3)
                assert np.array_equal(T.astype(np.int64), To), (kind, i)
                assert np.array_equal(V.view(np.uint32), (V32 if chain32 else Vo).view(np.uint32)), (kind, i, gs)
                met |= {int(x) for x in r.stdout.split()}
    assert SIZES <= met, SIZES - met
