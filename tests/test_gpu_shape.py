"""The default launch shape, which goes by the number of meshlets: that a tune
read, saved and set again keeps it, and that decodes are bit for bit the same
on both sides of each of its lines."""
import numpy as np
import pytest

from tests.conftest import gpu_available, ribbon
from tests.test_gpu_resid import stream

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def v5_stream(tris):
    from meshpress_amd import workloads
    from meshpress_amd.encoder.paradelta_v5 import encode_v5
    V, T = workloads.mesh_with_tris("torus", tris, 5)
    return encode_v5(V, T, precision_error=1.0 / 4094.5, precision_mode="bbox_frac")


def side_bytes(dec):
    """Bytes of the tables a decode reads: the groups of both passes are among
    them, so a decoder whose waves take other meshlets reports another number."""
    import ctypes as C
    b = C.c_uint64()
    call = "stride_batch_bytes" if hasattr(dec, "n_meshes") else "stride_decoder_bytes"
    assert getattr(dec._L, call)(dec._h, None, C.byref(b)) == 0
    return int(b.value)


@pytest.mark.parametrize("kind", ["dpr4", "batch", "v5_f64", "v5_f32"])
def test_a_tune_read_and_set_again_keeps_the_shape(kind):
    from meshpress_amd import workloads
    from meshpress_amd.batch import BatchDecoder
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    if kind.startswith("v5"):
        dec = ParaDeltaV5GpuDecoder(v5_stream(60000), chain=kind[3:])
        other = dict(group_size=8, tok_group=2)
    else:
        data = stream(*workloads.mesh_with_tris("torus", 60000, 1), 12, 3)
        dec = BatchDecoder([data]) if kind == "batch" else ParaDeltaV5GpuDecoder(data)
        other = dict(group_size=8, tok_group=2, waves=1)
    base, fresh = dec.get_tune(), side_bytes(dec)
    dec.set_tune(**base)                     # as it was read
    assert dec.get_tune() == base and side_bytes(dec) == fresh
    dec.set_tune(**({} if kind.startswith("v5") else dict(waves=2, stage_words=512)))   # another field
    assert side_bytes(dec) == fresh
    dec.set_tune(**other)
    assert side_bytes(dec) != fresh
    dec.set_tune(**base)                     # saved, then restored
    assert dec.get_tune() == base and side_bytes(dec) == fresh


def test_autotune_times_the_decoders_own_shape():
    """The searches hold the default shape, so that the fastest is never slower
    than not tuning, and a search without a usable candidate restores it."""
    from meshpress_amd.autotune import BENCH_CANDIDATES, candidates, tune
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    dec = ParaDeltaV5GpuDecoder(stream(*ribbon(400), 12, 3))
    base, fresh = dec.get_tune(), side_bytes(dec)
    for cands in (candidates(), BENCH_CANDIDATES):
        assert any(all(base[k] == v for k, v in c.items()) for c in cands)
    best, results = tune(dec, steps=1, cands=[dict(mode=9)])
    assert not results and best == base and side_bytes(dec) == fresh


def ribbon_stream(meshlets, bits=12, v5=False):
    """A ribbon of exactly so many meshlets of eight triangles, ten vertices."""
    from meshpress_amd.encoder.paradelta_v5 import encode_from_prepared_v5
    from meshpress_amd.encoder.prep import header_f32, prepare
    V, T = ribbon(4 * meshlets + 1)
    p = prepare(V, T, max_tris=8, precision_error=1.0 / ((1 << bits) - 1.5), precision_mode="bbox_frac")
    assert p["n_meshlets"] == meshlets
    if v5:
        return encode_from_prepared_v5(p)
    nat, pn, pk = p["native"], np.array([[1, 1, -1]] * 3, np.int64), np.zeros(3, np.int64)
    nat.residuals(pn, pk, export=False)
    return nat.write(header_f32(p), p["g_bits"], pn, pk, np.tile(np.array([1, 3], np.uint8), (meshlets, 6)))


@pytest.mark.parametrize("bits", [12, 18])
@pytest.mark.parametrize("meshlets", [511, 512, 1023, 1024, 4095, 4096, 8191, 8192])
def test_lines_of_the_default_shape(coracle, meshlets, bits):
    """Both sides of the lines between 2, 6 and 12 meshlets an axis group and
    1, 2 and 4 a token wave, with residual waves (12 bits) and without (18)."""
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    data = ribbon_stream(meshlets, bits)
    Vo, To = coracle.decode(data)
    dec = ParaDeltaV5GpuDecoder(data)
    for tune in ({}, dict(group_size=20)):   # by size, and a named shape
        dec.set_tune(**tune)
        Vg, Tg = dec.decode_to_host()
        assert np.array_equal(Tg.astype(np.int64), To)
        assert np.array_equal(Vg.view(np.uint32), Vo.view(np.uint32))


@pytest.mark.parametrize("chain", ["f64", "f32"])
@pytest.mark.parametrize("meshlets", [1023, 1024, 1535, 1536, 4095, 4096, 24575, 24576])
def test_lines_of_the_default_v5_shape(meshlets, chain):
    """PDLT v5: 2, 3, 4 and 6 meshlets a chain group, 1, 2 and 4 a token wave,
    against the one-kernel decode."""
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    dec = ParaDeltaV5GpuDecoder(ribbon_stream(meshlets, v5=True), chain=chain)
    Vg, Tg = dec.decode_to_host()
    dec.set_tune(mode=3)
    V3, T3 = dec.decode_to_host()
    assert np.array_equal(Tg, T3) and np.array_equal(Vg.view(np.uint32), V3.view(np.uint32))


def test_noalloc_without_room_for_the_residuals(coracle):
    """12,914 meshlets of 256 vertices: the walk fits the 32 MiB of static
    scratch, walk and residuals do not.  The axis lanes then decode the
    codewords in groups of their own; named shapes and the decoder's own
    scratch between, a default shape set again after."""
    import torch
    from meshpress_amd import _lib
    from meshpress_amd.utils.paradelta_v5_cuda import ParaDeltaV5GpuDecoder
    data = stream(*ribbon(1640001), 12, 2)
    Vo, To = coracle.decode(data, n_threads=8)
    dec = ParaDeltaV5GpuDecoder(data)
    walk = dec.n_v_total + 4 * dec.n_meshlets + 8
    assert dec.n_meshlets >= 8192 and walk + 64 <= 8 << 20 < 64 + 5 * walk // 2
    base = dec.get_tune()
    V, T = torch.empty_like(dec.d_verts), torch.empty_like(dec.d_tris)
    for tune in ({}, dict(group_size=20), base):
        dec.set_tune(**tune)
        for call in ("noalloc", "own", "noalloc"):
            V.fill_(float("nan"))
            T.fill_(-1)
            if call == "own":
                dec.decode_into(V, T)
            else:
                _lib.check(dec._L.stride_decode_noalloc(dec._h, _lib.ptr(V), _lib.ptr(T), _lib.stream_ptr()))
            assert np.array_equal(T.cpu().numpy(), To)
            assert np.array_equal(V.cpu().numpy().view(np.uint32), Vo.view(np.uint32))
