"""The two-pass decode's residual waves on the GPU, bit for bit against the
oracle, where their routes part: residual runs staged in LDS or read from the
stream, substreams too long for the chunk table, more units than lanes, 16-bit
codes and wider ones, predictors outside 32-bit exactness."""
import numpy as np
import pytest

from tests.conftest import gpu_available, ribbon

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def stream(V, T, bits, k, pred_n=((1, 1, -1),) * 3, pred_K=(0, 0, 0)):
    """DPR4 bytes with every residual stream coded as Rice(k), or as
    Exp-Golomb(-k) for negative k."""
    from meshpress_amd.encoder.prep import header_f32, prepare
    p = prepare(V, T, precision_error=1.0 / ((1 << bits) - 1.5), precision_mode="bbox_frac")
    nat = p["native"]
    pn, pk = np.array(pred_n, np.int64), np.array(pred_K, np.int64)
    nat.residuals(pn, pk, export=False)
    tagk = np.tile(np.array([1, k] if k >= 0 else [2, -k], np.uint8), (p["n_meshlets"], 6))
    return nat.write(header_f32(p), p["g_bits"], pn, pk, tagk)


CASES = {
    # about 150 bits a value: 8,400 words of residuals in a token wave of four
    "long_runs": (16, 0, {}),
    "rice": (16, 7, {}),
    "exp_golomb": (16, -4, {}),
    "12_bits": (12, 2, {}),
    "18_bits": (18, 9, {}),                                    # int32 codes
    "wide_weights": (16, 7, dict(pred_n=((30000, 30000, -30000),) * 3, pred_K=(15, 15, 15))),
    "shifted": (16, 7, dict(pred_n=((33, 32, -33), (31, 34, -33), (32, 32, -32)), pred_K=(5, 5, 5))),
}


@pytest.mark.parametrize("tune", [dict(), dict(mode=4, group_size=21, lds_bytes=65536, tok_chains=2, tok_group=32),
                                  dict(mode=4, group_size=3, lds_bytes=8192, tok_chains=16, tok_group=1)],
                         ids=["default", "wide_waves", "narrow_waves"])
@pytest.mark.parametrize("case", CASES)
def test_residual_waves(coracle, case, tune):
    from meshpress_amd import workloads
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    bits, k, kw = CASES[case]
    V, T = workloads.mesh_with_tris("torus", 6000, 3)
    data = stream(V, T, bits, k, **kw)
    dec = ParaDeltaV5GpuDecoder(data)
    if tune:
        dec.set_tune(**tune)
    Vo, To = coracle.decode(data)
    for _ in range(2):
        Vg, Tg = dec.decode_to_host()
        assert np.array_equal(Tg.astype(np.int64), To)
        assert np.array_equal(Vg.view(np.uint32), Vo.view(np.uint32))


@pytest.mark.parametrize("n", [2, 3, 15, 16, 17, 31, 32, 33, 128, 1000])
def test_chunk_edges(coracle, n):
    """Meshlets of 2 n vertices, around the 32-entry chunks and the
    8-entry groups of the chain (256 vertices: all eight chunks)."""
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    V, T = ribbon(n)
    data = stream(V, T, 12, 3)
    Vo, To = coracle.decode(data)
    Vg, Tg = ParaDeltaV5GpuDecoder(data).decode_to_host()
    assert np.array_equal(Tg.astype(np.int64), To)
    assert np.array_equal(Vg.view(np.uint32), Vo.view(np.uint32))


def test_substreams_past_the_chunk_table(coracle):
    """Residuals of thousands in unary: substreams past 65,535 bits."""
    from meshpress_amd import workloads
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    V, T = workloads.mesh_with_tris("torus", 600, 3)
    V = V + np.random.default_rng(0).normal(0, 0.02, V.shape)
    data = stream(V, T, 16, 0)
    assert len(data) > 3 * 65535 // 8
    Vo, To = coracle.decode(data)
    Vg, Tg = ParaDeltaV5GpuDecoder(data).decode_to_host()
    assert np.array_equal(Tg.astype(np.int64), To)
    assert np.array_equal(Vg.view(np.uint32), Vo.view(np.uint32))


@pytest.mark.parametrize("meshlets", [4095, 4096, 4097])
def test_scan_by_waves_and_by_lanes(coracle, meshlets):
    """The pre-pass of a batch on both sides of the line between a wave and a
    lane per meshlet: one mesh of many meshlets, then streams of one, so that
    runs of one mesh and runs across meshes both occur."""
    import torch
    from meshpress_amd import workloads
    from meshpress_amd.batch import BatchDecoder
    big = stream(*workloads.mesh_with_tris("torus", 300000, 1), 12, 3)
    one = stream(*ribbon(9), 12, 3)
    n_big = BatchDecoder([big]).n_meshlets
    bd = BatchDecoder([big] + [one] * (meshlets - n_big))
    assert bd.n_meshlets == meshlets
    v, t = bd.decode()
    torch.cuda.synchronize()
    got = bd.split(v.cpu().numpy(), t.cpu().numpy())
    for i, data in ((0, big), (1, one), (len(got) - 1, one)):
        Vo, To = coracle.decode(data)
        assert np.array_equal(got[i][1].astype(np.int64), To)
        assert np.array_equal(got[i][0].view(np.uint32), Vo.view(np.uint32))
    assert all(np.array_equal(g[0].view(np.uint32), got[1][0].view(np.uint32)) for g in got[2:])


@pytest.mark.parametrize("meshlets", [1, 511, 512, 1023, 1024])
def test_default_shape_by_size(coracle, meshlets):
    """The default shape's waves on both sides of their lines, against a named
    shape (which the reported default is), single streams and batches."""
    import torch
    from meshpress_amd.batch import BatchDecoder
    one = stream(*ribbon(40), 12, 3)
    Vo, To = coracle.decode(one)
    bd = BatchDecoder([one] * meshlets)
    assert bd.n_meshlets == meshlets
    shape = bd.get_tune()
    assert (shape["group_size"], shape["tok_group"], shape["tok_chains"]) == (21, 4, 16)
    for tune in (None, shape):
        if tune:
            bd.set_tune(**tune)
        for mode in ("launch", "per_mesh", "graph"):
            bd.d_verts.fill_(-1)
            bd.d_tris.fill_(-1)
            v, t = bd.decode(mode)
            torch.cuda.synchronize()
            v, t = v.cpu().numpy(), t.cpu().numpy()
            for i in (0, meshlets // 2, meshlets - 1):
                (Vi, Ti), = [bd.split(v, t)[i]]
                assert np.array_equal(Ti.astype(np.int64), To)
                assert np.array_equal(Vi.view(np.uint32), Vo.view(np.uint32))


@pytest.mark.parametrize("chain", ["f64", "f32"])
@pytest.mark.parametrize("tris", [2304, 230000, 360000])
def test_pdlt_code_waves_match_one_kernel(tris, chain):
    """PDLT v5 with code waves in the default shape and in named ones, against
    the one-kernel decode of the same stream."""
    from meshpress_amd import workloads
    from meshpress_amd.encoder.paradelta_v5 import encode_from_prepared_v5
    from meshpress_amd.encoder.prep import prepare
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    V, T = workloads.mesh_with_tris("torus", tris, 5)
    data = encode_from_prepared_v5(prepare(V, T, precision_error=1.0 / 4094.5, precision_mode="bbox_frac"))
    dec = ParaDeltaV5GpuDecoder(data, chain=chain)
    got = [dec.decode_to_host()]
    for tune in (dict(mode=4, group_size=16, tok_group=4, tok_chains=16), dict(group_size=1, tok_group=64),
                 dict(tok_chains=0, tok_group=64), dict(mode=3)):
        dec.set_tune(**tune)
        got.append(dec.decode_to_host())
    for Vg, Tg in got[:-1]:
        assert np.array_equal(Tg, got[-1][1])
        assert np.array_equal(Vg.view(np.uint32), got[-1][0].view(np.uint32))


@pytest.mark.parametrize("name", ["pdlt_hf_24_tags", "pdlt_torus_q16_tags", "pdlt_fan_parts", "pdlt_one_tri"])
def test_pdlt_code_waves_on_every_coder(name):
    """Golden streams of the three residual coders, and of meshlets without
    interior or boundary vertices."""
    import hashlib
    from pathlib import Path
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    z = np.load(Path(__file__).resolve().parent / "golden" / f"{name}.npz")
    dec = ParaDeltaV5GpuDecoder(z["data"].tobytes())
    for tune in (dict(), dict(mode=4, group_size=16, tok_group=64, tok_chains=1)):
        if tune:
            dec.set_tune(**tune)
        V, T = dec.decode_to_host()
        for a, key in ((V, "V_sha"), (T.astype(np.int64), "T_sha")):
            assert hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest() == z[key].tobytes().hex()
