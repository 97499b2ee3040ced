"""CPU tests of the PDLT v5 decoder's set-up and kernel logic, compiled for
the host (tests/pdlt_lane_check.cpp, under ASan + UBSan), against the oracle
(oracle/pdlt_oracle.py)."""
from pathlib import Path

import numpy as np
import pytest

from oracle import pdlt_oracle as PO
from tests.conftest import small_meshes

ROOT = Path(__file__).resolve().parents[1]
GOLD = sorted((ROOT / "tests" / "golden").glob("pdlt_*.npz"))
LAYOUTS = [(16, 32768), (1, 4096), (5, 16384), (16, 65536)]


@pytest.fixture(scope="module")
def pdlt_check(tmp_path_factory):
    import shutil
    import subprocess
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("pdlt") / "pdlt_lane_check"
    subprocess.run([gxx, "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=undefined", "-ffp-contract=off", "-pthread",
                    str(ROOT / "tests" / "pdlt_lane_check.cpp"), "-o", str(exe)], check=True)
    return exe


def run(exe, data, tmp_path, gs=16, lds=32768, world=True, chain32=False, two_pass=0, k0=16):
    """two_pass: 0 one pass, 1 token lanes then the chain pass, 2 token
    chains (about k0 a meshlet) then the chain pass."""
    import subprocess
    src = tmp_path / "s.pdlt"
    src.write_bytes(data)
    fv, ft = tmp_path / "v.f32", tmp_path / "t.u32"
    r = subprocess.run([str(exe), str(src), str(fv), str(ft), str(gs), str(lds),
                        "0" if world else "1", "1" if chain32 else "0", str(int(two_pass)), str(k0)],
                       capture_output=True, text=True)
    if r.returncode != 0:
        return r.returncode, r.stderr, None
    return 0, np.fromfile(fv, np.float32).reshape(-1, 3), np.fromfile(ft, np.uint32).reshape(-1, 3)


def same(V, T, Vo, To):
    return (V.shape == Vo.shape and np.array_equal(V.view(np.uint32), Vo.view(np.uint32))
            and np.array_equal(T.astype(np.int64), To))


@pytest.mark.parametrize("path", GOLD, ids=lambda p: p.stem)
def test_lane_logic_matches_oracle_on_goldens(pdlt_check, tmp_path, path):
    data = np.load(path)["data"].tobytes()
    Vo, To = PO.decode_v5(data)
    for gs, lds in LAYOUTS:
        for two_pass in (0, 1, 2):
            rc, V, T = run(pdlt_check, data, tmp_path, gs, lds, two_pass=two_pass)
            assert rc == 0, V
            assert same(V, T, Vo, To), (gs, lds, two_pass)
    for k0 in (2, 5, 8):
        rc, V, T = run(pdlt_check, data, tmp_path, two_pass=2, k0=k0)
        assert rc == 0 and same(V, T, Vo, To), k0
    rc, V, T = run(pdlt_check, data, tmp_path, world=False)
    Vn, _ = PO.decode_v5(data, world=False)
    assert rc == 0 and same(V, T, Vn, To)
    for world in (True, False):
        V32, _ = PO.decode_v5(data, world=world, chain="f32")
        # the float32 chain pass's blocks hold no refs slot (two-pass)
        for two_pass in (0, 1, 2):
            rc, V, T = run(pdlt_check, data, tmp_path, 7, 20480, world=world, chain32=True,
                           two_pass=two_pass)
            assert rc == 0 and same(V, T, V32, To), (world, two_pass)


def test_lane_logic_matches_oracle_on_fresh_streams(pdlt_check, tmp_path):
    from meshpress_amd import workloads as w
    from meshpress_amd.encoder.paradelta_v5 import encode_v5
    cases = [(m[1], m[2], {}) for m in small_meshes()]
    cases.append(w.heightfield(90, 0.1, 6, 7) + ({},))
    cases.append(w.displaced_icosphere(4, 0.08, 6, 1) +
                 (dict(precision_error=1.0 / 65534.5, precision_mode="bbox_frac"),))
    cases.append(w.displaced_torus(40, 16, 1.0, 0.3, 0.05, 4, 5) + (dict(max_verts=64, max_tris=96),))
    for V, T, kw in cases:
        data = encode_v5(V, T, **kw)
        rc, Vl, Tl = run(pdlt_check, data, tmp_path)
        assert rc == 0
        assert same(Vl, Tl, *PO.decode_v5(data))
        V32 = PO.decode_v5(data, chain="f32")
        for two_pass in (0, 2):
            rc, Vl, Tl = run(pdlt_check, data, tmp_path, chain32=True, two_pass=two_pass)
            assert rc == 0
            assert same(Vl, Tl, *V32), two_pass
        rc, Vl, Tl = run(pdlt_check, data, tmp_path, 7, 12288, two_pass=1)
        assert rc == 0
        assert same(Vl, Tl, *PO.decode_v5(data))
        for k0 in (4, 16):
            rc, Vl, Tl = run(pdlt_check, data, tmp_path, 7, 12288, two_pass=2, k0=k0)
            assert rc == 0
            assert same(Vl, Tl, *PO.decode_v5(data))


def strip_lengths(data):
    """(bit position, length) of every strip length field of a PDLT v5
    stream: each meshlet from its offset, the header, boundary refs and
    strip tokens walked as encoder/paradelta_v5.py:345-420 lays them out."""
    h = PO.read_header(data)
    out = []
    for off in h["offsets"]:
        r = PO.BitReader(data, off)
        n_bnd, n_int, _n_tris, n_strips = (r.get(16) for _ in range(4))
        if n_bnd > 0:
            r.get(32)
            if n_bnd > 1:
                k = r.get(8)
                for _ in range(n_bnd - 1):
                    r.rice(k)
        ib = PO.idx_bits_for(n_bnd + n_int)
        for _s in range(n_strips):
            at = r.pos
            L = r.get(16)
            out.append((at, L))
            for t in range(3 + max(L - 1, 0)):
                if t >= 3:
                    r.get(1)
                r.get(5 if r.get(1) == 0 else ib)
    return out


def long_strip_stream(n_tris):
    """The one-triangle golden stream with its strip stretched to n_tris
    triangles: the three root tokens, then n_tris - 1 body tokens (edge bit
    0, FIFO hit on the oldest entry), the residual section kept (no token
    names a new vertex).  Layout as encoder/paradelta_v5.py:144-283 writes it:
    the meshlet header at the first offset, n_tris in its third field, the
    strip length after the header, 3-bit root tokens for 3 locals."""
    data = np.load(ROOT / "tests" / "golden" / "pdlt_one_tri.npz")["data"].tobytes()
    h = PO.read_header(data)
    assert (h["n_meshlets"], h["n_boundary"], h["n_t"]) == (1, 0, 1)
    bits = "".join(f"{b:08b}" for b in data)
    m0 = h["meshlets_bit"]
    assert bits[m0:m0 + 80] == f"{0:016b}{3:016b}{1:016b}{1:016b}{1:016b}"
    head = bits[:m0]
    head = head[:57 * 8] + f"{n_tris:032b}" + head[61 * 8:]        # header n_t
    body = (f"{0:016b}{3:016b}{n_tris:016b}{1:016b}{n_tris:016b}" + bits[m0 + 80:m0 + 89]
            + "0" * 7 * (n_tris - 1) + bits[m0 + 89:])
    out = head + body
    out += "0" * (-len(out) % 8)
    return bytes(int(out[i:i + 8], 2) for i in range(0, len(out), 8))


def test_long_strip_meshlets(pdlt_check, tmp_path):
    """One meshlet of 8,000 and one of 20,000 triangles in a single strip:
    the first runs the chain token pass as one chain (more than 511
    tokens), the second needs more LDS for its token records than a chain
    wave has (its layout is refused; the decoder then runs token lanes)."""
    for n in (8000, 20000):
        data = long_strip_stream(n)
        Vo, To = PO.decode_v5(data)
        assert To.shape == (n, 3)
        for two_pass in (0, 1):
            rc, V, T = run(pdlt_check, data, tmp_path, two_pass=two_pass)
            assert rc == 0 and same(V, T, Vo, To), (n, two_pass)
        rc, V, T = run(pdlt_check, data, tmp_path, two_pass=2)
        if n == 8000:
            assert rc == 0 and same(V, T, Vo, To)
        else:
            assert rc == 2 and "too large for the chain token pass" in V


def test_zero_length_strips_decode_as_length_one(pdlt_check, tmp_path):
    """A strip length of 0 stands for one triangle (its three roots), as
    length 1 does (decode_paradelta_v5 runs L - 1 body steps): rewriting
    every length-1 field to 0 leaves the decode unchanged on every path."""
    from meshpress_amd import workloads as w
    from meshpress_amd.encoder.paradelta_v5 import encode_v5
    V, T = w.displaced_torus(40, 16, 1.0, 0.3, 0.05, 4, 5)
    data = encode_v5(V, T, max_verts=64, max_tris=96)
    Vo, To = PO.decode_v5(data)
    ones = [at for at, L in strip_lengths(data) if L == 1]
    assert ones, "no length-1 strip to rewrite"
    d = bytearray(data)
    for at in ones:
        assert (d[(at + 15) >> 3] >> (7 - ((at + 15) & 7))) & 1
        d[(at + 15) >> 3] &= ~(1 << (7 - ((at + 15) & 7))) & 0xFF
    d = bytes(d)
    assert same(*PO.decode_v5(d), Vo, To)
    for two_pass, k0 in ((0, 16), (1, 16), (2, 2), (2, 16)):
        rc, Vl, Tl = run(pdlt_check, d, tmp_path, two_pass=two_pass, k0=k0)
        assert rc == 0, Vl
        assert same(Vl, Tl, Vo, To), (two_pass, k0)


def test_prepass_rejects_or_matches_under_bit_flips(pdlt_check, tmp_path):
    """Whenever the host-built pre-pass accepts a corrupted stream, the lane
    decoder's output equals the oracle's (the oracle must not reject it)."""
    base = bytearray(np.load(ROOT / "tests" / "golden" / "pdlt_hf_24_tags.npz")["data"].tobytes())
    rng = np.random.default_rng(7)
    accepted = 0
    for trial in range(80):
        d = bytearray(base)
        pos = int(rng.integers(8 * 81, 8 * len(d)))
        d[pos >> 3] ^= 1 << (7 - (pos & 7))
        rc, V, T = run(pdlt_check, bytes(d), tmp_path)
        if rc != 0:
            assert rc == 2, V
            continue
        accepted += 1
        try:
            Vo, To = PO.decode_v5(bytes(d))
        except (ValueError, IndexError) as e:
            raise AssertionError(f"trial {trial}: pre-pass accepted a stream the oracle rejects: {e}")
        assert same(V, T, Vo, To), trial
    assert accepted > 0


def test_truncated_and_bad_headers_rejected(pdlt_check, tmp_path):
    data = np.load(ROOT / "tests" / "golden" / "pdlt_uv_12x24.npz")["data"].tobytes()
    for cut in (3, 40, 81, 100, len(data) // 2, len(data) - 1):
        rc, msg, _ = run(pdlt_check, data[:cut], tmp_path)
        assert rc == 2, cut
    bad = bytearray(data)
    bad[4] = 4
    rc, msg, _ = run(pdlt_check, bytes(bad), tmp_path)
    assert rc == 2 and "expected v5, got v4" in msg
    bad = bytearray(data)
    bad[0] = 0
    rc, msg, _ = run(pdlt_check, bytes(bad), tmp_path)
    assert rc == 2 and "bad magic" in msg


@pytest.mark.parametrize("n", [255, 256, 257, 258, 259, 260, 300, 400, 509])
def test_long_strips_cut_into_chains(pdlt_check, tmp_path, n):
    """One strip of n triangles, n + 2 tokens: up to 511 tokens are cut into
    chains, and the chain cuts' scan counts past the 258 tokens of the longest
    DPR4 strip."""
    data = long_strip_stream(n)
    Vo, To = PO.decode_v5(data)
    assert To.shape == (n, 3)
    for two_pass, k0 in ((0, 16), (1, 16), (2, 1), (2, 2), (2, 5), (2, 16)):
        rc, V, T = run(pdlt_check, data, tmp_path, two_pass=two_pass, k0=k0)
        assert rc == 0 and same(V, T, Vo, To), (two_pass, k0)


@pytest.mark.parametrize("mesh", ["torus", "tubes"])
def test_long_strips_of_meshes(pdlt_check, tmp_path, mesh):
    """Meshlets of up to 400 triangles, whose strips pass 257 triangles."""
    from meshpress_amd import workloads as w
    from meshpress_amd.encoder.paradelta_v5 import encode_v5
    if mesh == "torus":
        V, T = w.displaced_torus(60, 20, 1.0, 0.3, 0.05, 4, 5)
    else:
        V, T = w.displaced_torus(400, 3, 1.0, 0.1, 0.02, 4, 5)
    data = encode_v5(V, T, max_verts=256, max_tris=400)
    assert max(L for _, L in strip_lengths(data)) > 257
    Vo, To = PO.decode_v5(data)
    V32, _ = PO.decode_v5(data, chain="f32")
    for two_pass, k0 in ((0, 16), (1, 16), (2, 2), (2, 8), (2, 16)):
        rc, Vl, Tl = run(pdlt_check, data, tmp_path, two_pass=two_pass, k0=k0)
        assert rc == 0 and same(Vl, Tl, Vo, To), (two_pass, k0)
    rc, Vl, Tl = run(pdlt_check, data, tmp_path, chain32=True, two_pass=2)
    assert rc == 0 and same(Vl, Tl, V32, To)
