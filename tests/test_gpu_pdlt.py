"""GPU parity of the PDLT v5 decoder (ParaDeltaV5GpuDecoder on PDLT v5
streams) against the oracle (oracle/pdlt_oracle.py), itself pinned to the
reference's decode_paradelta_v5 by the golden vectors: float32 positions
bit for bit (tolerance 0 ulp), indices exactly."""
from pathlib import Path

import numpy as np
import pytest

from oracle import pdlt_oracle as PO
from tests.conftest import gpu_available, small_meshes

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]

GOLD = sorted((Path(__file__).resolve().parent / "golden").glob("pdlt_*.npz"))
# mode 4: token pass + chain pass (default); mode 3: one kernel.  Token lanes
# (tok_chains 0): stage_words is the token pass's LDS budget in words.
LANES = dict(tok_chains=0, tok_group=64)
LAYOUTS = [dict(mode=4, group_size=16, lds_bytes=32768, stage_words=8192, **LANES),
           dict(mode=3, group_size=16, lds_bytes=32768, **LANES),
           dict(mode=4, group_size=1, lds_bytes=4096, stage_words=1024, **LANES),
           dict(mode=3, group_size=5, lds_bytes=16384, **LANES),
           dict(mode=4, group_size=16, lds_bytes=65536, stage_words=16384, **LANES)]
# mode 4 with token chains: about tok_chains chains a meshlet, tok_group
# meshlets (and up to 64 chains) a token wave
CHAIN_LAYOUTS = [dict(mode=4, group_size=16, lds_bytes=24576, tok_chains=16, tok_group=4),
                 dict(mode=4, group_size=8, lds_bytes=16384, tok_chains=4, tok_group=16),
                 dict(mode=4, group_size=16, lds_bytes=24576, tok_chains=1, tok_group=64),
                 dict(mode=4, group_size=5, lds_bytes=16384, tok_chains=7, tok_group=3)]


def decoder(data, chain="f64", **tune):
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    dec = ParaDeltaV5GpuDecoder(data, chain=chain)
    if tune:
        dec.set_tune(**tune)
    return dec


def assert_same(V, T, Vo, To):
    assert V.dtype == np.float32 and T.dtype == np.uint32
    assert V.shape == Vo.shape and T.shape == To.shape
    assert np.array_equal(T.astype(np.int64), To)
    assert np.array_equal(V.view(np.uint32), Vo.view(np.uint32))


@pytest.mark.parametrize("path", GOLD, ids=lambda p: p.stem)
def test_golden_streams_all_layouts(path):
    data = np.load(path)["data"].tobytes()
    print(f"pdlt golden {path.stem}", flush=True)
    Vo, To = PO.decode_v5(data)
    dec = decoder(data)
    assert (dec.get_tune()["tok_chains"], dec.get_tune()["tok_group"]) == (16, 4)   # the default
    assert_same(*dec.decode_to_host(), Vo, To)
    for tune in LAYOUTS + CHAIN_LAYOUTS:
        dec = decoder(data, **tune)
        assert dec.version == 5
        assert dec.get_tune()["tok_chains"] == tune["tok_chains"]
        assert_same(*dec.decode_to_host(), Vo, To)
    V32, _ = PO.decode_v5(data, chain="f32")
    assert_same(*decoder(data, chain="f32").decode_to_host(), V32, To)
    assert_same(*decoder(data, chain="f32", **CHAIN_LAYOUTS[0]).decode_to_host(), V32, To)


def test_normalised_decode_matches_reference_semantics():
    import torch
    data = np.load(GOLD[0])["data"].tobytes()
    dec = decoder(data)
    v, t = dec.decode()
    torch.cuda.synchronize()
    Vn, To = PO.decode_v5(data, world=False)
    assert np.array_equal(v.cpu().numpy().view(np.uint32), Vn.view(np.uint32))
    assert np.array_equal(t.cpu().numpy().astype(np.int64), To)


def test_fresh_streams():
    from meshpress_amd import workloads as w
    from meshpress_amd.encoder.paradelta_v5 import encode_v5
    cases = [(m[1], m[2], {}) for m in small_meshes()]
    cases.append(w.heightfield(90, 0.1, 6, 7) + ({},))
    cases.append(w.displaced_icosphere(4, 0.08, 6, 1) +
                 (dict(precision_error=1.0 / 65534.5, precision_mode="bbox_frac"),))
    cases.append(w.displaced_torus(40, 16, 1.0, 0.3, 0.05, 4, 5) + (dict(max_verts=64, max_tris=96),))
    for i, (V, T, kw) in enumerate(cases):
        print(f"pdlt fresh case {i} n_t={len(T)}", flush=True)
        data = encode_v5(V, T, **kw)
        ref = PO.decode_v5(data)
        assert_same(*decoder(data).decode_to_host(), *ref)
        assert_same(*decoder(data, chain="f32").decode_to_host(), *PO.decode_v5(data, chain="f32"))
        for tune in (dict(mode=4, **LANES), CHAIN_LAYOUTS[1], CHAIN_LAYOUTS[3]):
            assert_same(*decoder(data, **tune).decode_to_host(), *ref)


def test_zero_length_strips_on_every_token_pass():
    """Strip length 0 (one triangle, as length 1) through the token lanes,
    the token chains and the single kernel."""
    from meshpress_amd import workloads as w
    from meshpress_amd.encoder.paradelta_v5 import encode_v5
    from tests.test_pdlt_host import strip_lengths
    V, T = w.displaced_torus(40, 16, 1.0, 0.3, 0.05, 4, 5)
    data = bytearray(encode_v5(V, T, max_verts=64, max_tris=96))
    ref = PO.decode_v5(bytes(data))
    for at, L in strip_lengths(bytes(data)):
        if L == 1:
            data[(at + 15) >> 3] &= ~(1 << (7 - ((at + 15) & 7))) & 0xFF
    data = bytes(data)
    assert [L for _, L in strip_lengths(data)].count(0) > 0
    for tune in (dict(mode=3), dict(mode=4, **LANES),
                 dict(mode=4, tok_chains=2, tok_group=8), dict(mode=4, tok_chains=16, tok_group=4)):
        assert_same(*decoder(data, **tune).decode_to_host(), *ref)


def test_long_strip_meshlets():
    """A one-meshlet stream of 8,000 triangles in one strip decodes through
    the token chains as one chain; one of 20,000 needs more LDS for its
    token records than a chain wave has, and runs the token lanes."""
    from tests.test_pdlt_host import long_strip_stream
    for n, chains in ((8000, 16), (20000, 0)):
        print(f"pdlt long strip n_tris={n}", flush=True)
        data = long_strip_stream(n)
        ref = PO.decode_v5(data)
        dec = decoder(data)
        assert (dec.get_tune()["tok_chains"], dec.get_tune()["tok_group"]) == (chains, 4 if chains else 64)
        assert_same(*dec.decode_to_host(), *ref)
        assert_same(*decoder(data, mode=3).decode_to_host(), *ref)


def test_chain_tune_round_trip_and_errors():
    data = np.load(GOLD[-1])["data"].tobytes()
    dec = decoder(data, **CHAIN_LAYOUTS[0])
    t = dec.get_tune()
    assert (t["tok_chains"], t["tok_group"]) == (16, 4)
    with pytest.raises(ValueError, match="tok_chains"):
        dec.set_tune(tok_chains=17)
    assert dec.get_tune() == t            # a refused tune leaves the layout as it was
    dec.set_tune(tok_chains=-1, group_size=8)   # -1 keeps the chains
    assert (dec.get_tune()["tok_chains"], dec.get_tune()["group_size"]) == (16, 8)
    dec.set_tune(tok_chains=0, tok_group=0)
    assert (dec.get_tune()["tok_chains"], dec.get_tune()["tok_group"]) == (0, 64)
    assert_same(*dec.decode_to_host(), *PO.decode_v5(data))


def test_repeated_decode_is_stable():
    import torch
    data = np.load(GOLD[-1])["data"].tobytes()
    dec = decoder(data)
    V0, T0 = dec.decode_to_host()
    for _ in range(3):
        dec.decode()
        V, T = dec.decode_to_host()
        torch.cuda.synchronize()
        assert np.array_equal(V.view(np.uint32), V0.view(np.uint32)) and np.array_equal(T, T0)


def test_decoder_errors():
    data = np.load(GOLD[0])["data"].tobytes()
    bad = bytearray(data)
    bad[4] = 4
    with pytest.raises(ValueError, match="expected v5, got v4"):
        decoder(bytes(bad))
    with pytest.raises(IndexError):
        decoder(data[: len(data) // 2])
    with pytest.raises(IndexError):      # an endless unary run in the boundary table
        decoder(data[:81] + bytes(len(data) - 81))
    h = PO.read_header(data)
    table = (h["meshlets_bit"] - 32 * h["n_meshlets"]) // 8
    bad = bytearray(data)
    bad[table + 3] ^= 8                   # first meshlet offset off by 8 bits
    with pytest.raises(ValueError, match="offsets"):
        decoder(bytes(bad))


@pytest.mark.parametrize("n", [600])
def test_large_mesh_error_bound_and_faces(n):
    """A 718K-triangle mesh: with the encoder's float32 chain every position
    is within the quantisation bound of its source vertex; the float64 chain
    (decode_paradelta_v5's arithmetic) stays within float32 drift of it; the
    face set is the source's; a second layout decodes identically."""
    from meshpress_amd import workloads as w
    from meshpress_amd.encoder.paradelta_v5 import encode_from_prepared_v5
    from meshpress_amd.encoder.prep import prepare
    V, T = w.heightfield(n, 0.1, 6, 7)
    p = prepare(V, T)
    data = encode_from_prepared_v5(p)
    print(f"pdlt large n_t={len(T)} bytes={len(data)}", flush=True)
    dec = decoder(data)
    Vg, Tg = dec.decode_to_host()
    # decoded vertex ids: boundary table, then each meshlet's interior locals
    plans = p["native"].export_plans()
    prep = dict(p)
    prep["plans"] = plans
    pv = PO.prepare_v5(prep)
    ids = np.concatenate([np.asarray(pv["boundary_list"], np.int64)] +
                         [np.asarray(pl["local_to_global"][pl["n_bnd"]:], np.int64) for pl in plans])
    assert len(ids) == len(Vg)
    V32, T32 = decoder(data, chain="f32").decode_to_host()
    assert np.array_equal(T32, Tg)
    step = p["per_coord_err"] * p["scale"]
    err = np.abs(V32.astype(np.float64) - V[ids]).max()
    bound = step + 16 * 2.0 ** -24 * (np.abs(V).max() + 1)
    assert err <= bound, (err, bound)
    drift = np.abs(Vg.astype(np.float64) - V32).max()
    assert drift <= 0.05 * step, (drift, step)
    got = np.sort(ids[Tg.astype(np.int64)], axis=1)
    want = np.sort(T, axis=1)
    assert np.array_equal(got[np.lexsort(got.T[::-1])], want[np.lexsort(want.T[::-1])])
    for tune in (dict(mode=4, group_size=3, lds_bytes=12288, stage_words=2048),
                 dict(mode=3, group_size=3, lds_bytes=12288)):
        V2, T2 = decoder(data, **tune).decode_to_host()
        assert np.array_equal(V2.view(np.uint32), Vg.view(np.uint32)) and np.array_equal(T2, Tg)


def test_sblb_blobs_decode_like_pdlt():
    from meshpress_amd.utils.sblb import to_sblb
    for path in GOLD:
        data = np.load(path)["data"].tobytes()
        Vo, To = PO.decode_v5(data)
        print(f"sblb {path.stem}", flush=True)
        assert_same(*decoder(to_sblb(data)).decode_to_host(), Vo, To)
    blob = bytearray(to_sblb(np.load(GOLD[0])["data"].tobytes()))
    blob[-1] ^= 0x40                               # last boundary coordinate
    with pytest.raises(ValueError, match="SBLB"):
        decoder(bytes(blob))


def test_native_bench_cli_pdlt(tmp_path):
    """The native bench decodes a PDLT v5 stream and its SBLB blob with both
    chains and reports the event-timed rate."""
    import json
    import subprocess
    from meshpress_amd import build
    from meshpress_amd.utils.sblb import to_sblb
    if not build.BENCH.exists():
        pytest.skip("native bench not built")
    data = np.load([p for p in GOLD if p.stem == "pdlt_uv_c1"][0])["data"].tobytes()
    (tmp_path / "c1.pdlt").write_bytes(data)
    (tmp_path / "c1.sblb").write_bytes(to_sblb(data))
    for name, fmt in (("c1.pdlt", "pdlt_v5"), ("c1.sblb", "sblb")):
        for chain in ("64", "32"):
            r = subprocess.run([str(build.BENCH), str(tmp_path / name), "--iters", "5", "--warmup", "1",
                                "--group", "8", "--lds", "24576", "--chain", chain],
                               capture_output=True, text=True, timeout=120)
            assert r.returncode == 0, r.stderr
            out = json.loads(r.stdout)
            assert out["format"] == fmt and out["n_tris"] == 65536 and out["ms"] > 0
            assert out["chain"] == int(chain) and out["tune"]["group_size"] == 8


@pytest.mark.parametrize("case", [258, 260, 400, 509, "tubes"])
def test_strips_past_257_triangles_in_chains(case):
    """Meshlets of up to 511 tokens in one strip are cut into token chains:
    one strip of n triangles, and thin tubes in meshlets of 400 triangles."""
    from meshpress_amd import workloads
    from meshpress_amd.encoder.paradelta_v5 import encode_v5
    from tests.test_pdlt_host import long_strip_stream, strip_lengths
    if case == "tubes":
        data = encode_v5(*workloads.displaced_torus(400, 3, 1.0, 0.1, 0.02, 4, 5), max_verts=256, max_tris=400)
        assert max(L for _, L in strip_lengths(data)) > 257
    else:
        data = long_strip_stream(case)
    print(f"pdlt strips past 257 triangles: {case}", flush=True)
    for chain in ("f64", "f32"):
        ref = PO.decode_v5(data, chain=chain)
        assert_same(*decoder(data, chain).decode_to_host(), *ref)
        for tune in CHAIN_LAYOUTS:
            assert_same(*decoder(data, chain, **tune).decode_to_host(), *ref)
