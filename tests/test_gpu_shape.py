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
