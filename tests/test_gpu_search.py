"""The search kernels' forms against exact integer arithmetic: every split of
a wave over candidates, sample slices and meshlets, the 32-bit and the 64-bit
path, empty and long meshlets and streams."""
import numpy as np
import pytest

from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a ROCm GPU")]


def coder_costs(u, off):
    """Body bits of the 20 coders per stream, exact (u: object integers)."""
    out = np.zeros((len(off) - 1, 20), object)
    for i in range(len(off) - 1):
        x = [int(t) for t in u[off[i]:off[i + 1]]]
        for k in range(12):
            out[i, k] = sum((t >> k) + 1 + k for t in x)
        for k in range(8):
            out[i, 12 + k] = sum(2 * (((t >> k) + 1).bit_length() - 1) + 1 + k for t in x)
    return out


def zigzag(r):
    return np.array([-2 * int(t) - 1 if t < 0 else 2 * int(t) for t in r], object)


def samples(rng, counts, bits):
    off = np.concatenate(([0], np.cumsum(counts))).astype(np.int64)
    c = rng.integers(0, 1 << bits, int(off[-1]))
    step = 1 << max(0, bits - 6)
    a, b = c + rng.integers(-step, step + 1, c.size), c + rng.integers(-step, step + 1, c.size)
    v = a + b - c + rng.integers(-step, step + 1, c.size)
    top = (1 << min(bits, 31)) - 1
    return [np.clip(x, -top, top).astype(np.int32) for x in (a, b, c, v)], off


@pytest.mark.parametrize("n_m", [1, 3, 30, 1100])
@pytest.mark.parametrize("S", [1, 2, 3, 5, 9, 17, 33, 64, 65])
def test_irlp_costs(S, n_m):
    from meshpress_amd import _lib
    from meshpress_amd.encoder import search
    import torch
    rng = np.random.default_rng(1000 * S + n_m)
    K = int(rng.integers(0, 10))
    # few samples where there are many meshlets: the oracle is Python integers
    counts = rng.integers(0, 4 if n_m > 100 else 70, n_m)
    for bits in (12, 16, 28):     # 28: past the 24-bit factors, the 64-bit path
        cols, off = samples(rng, counts, bits)
        D = 1 << K
        cand = (np.array([D, D, -D]) + rng.integers(-D, D + 1, (S, 3))).astype(np.int32)
        got = search.IrlpCost(*cols, off)(cand, K)
        a, b, c, v = (x.astype(object) for x in cols)
        per = np.zeros((n_m, S), object)
        for s in range(S):
            p = int(cand[s, 0]) * a + int(cand[s, 1]) * b + int(cand[s, 2]) * c
            p = np.array([(int(t) + (D >> 1)) >> K for t in p], object) if K else p
            per[:, s] = coder_costs(zigzag(v - p), off).min(1)
        assert [int(x) for x in got] == [int(x) for x in per.sum(0)], bits
        d = [search._dev(x if len(x) else np.zeros(1, np.int32), torch.int32) for x in (*cols, cand)]
        out = torch.full((n_m, S), -1, dtype=torch.int64, device="cuda")
        _lib.check(_lib.lib().stride_irlp_cost_meshlets(
            *[_lib.ptr(x) for x in d[:4]], _lib.ptr(search._dev(off, torch.int64)), n_m, _lib.ptr(d[4]), S, K,
            _lib.ptr(out), _lib.stream_ptr()))
        assert np.array_equal(out.cpu().numpy(), per.astype(np.int64)), bits


def test_irlp_long_meshlet():
    """One meshlet of many samples: sums past 32 bits take the 64-bit path."""
    from meshpress_amd.encoder import search
    n = 70000
    a = np.full(n, 65535, np.int32)
    z = np.zeros(n, np.int32)
    off = np.array([0, n, n + 0], np.int64)
    got = search.IrlpCost(a, a, z, z, off)(np.array([[256, 256, -256], [0, 0, 0]], np.int32), 8)
    want = [coder_costs(zigzag([-131070]), np.array([0, 1])).min() * n, n]
    assert [int(x) for x in got] == [int(x) for x in want]


@pytest.mark.parametrize("kind", ["small", "extreme"])
def test_stream_costs(kind):
    from meshpress_amd.encoder import search
    rng = np.random.default_rng(5)
    lens = np.array([0, 1, 2, 15, 16, 17, 31, 32, 33, 0, 63, 64, 65, 200, 1000, 3, 0, 7, 8], np.int64)
    off = np.concatenate(([0], np.cumsum(lens))).astype(np.int64)
    vals = np.rint(rng.laplace(0, 20, off[-1])).astype(np.int32)
    if kind == "extreme":
        vals[::7] = -(1 << 31)
        vals[3::11] = (1 << 31) - 1
    want = coder_costs(zigzag(vals), off)
    assert np.array_equal(search.stream_costs(vals, off), want.astype(np.int64))
    tagk, bits = search.select_codes(vals, off)
    for i in range(len(lens)):
        r, e = list(want[i, :12]), list(want[i, 12:])
        rice = min(r) <= min(e)
        exp = (1, r.index(min(r))) if rice else (2, e.index(min(e)))
        if lens[i] == 0:
            exp, rb = (1, 0), 0
        else:
            rb = min(min(r), min(e))
        assert (tuple(int(x) for x in tagk[i]), int(bits[i])) == (exp, rb), i


@pytest.mark.parametrize("n", [3, 64, 511, 513, 5000, 140001])
@pytest.mark.parametrize("bits", [12, 16, 24])
def test_irls_matches_the_host(n, bits):
    """The GPU's L1 fit against the numpy one: both solve in float64, the
    host from columns of condition about 2^bits / step."""
    from meshpress_amd.encoder import search
    rng = np.random.default_rng(n + bits)
    top, step = (1 << bits) - 1, (1 << bits) / 200.0
    c = rng.uniform(0, top, n)
    a, b = c + rng.normal(0, step, n), c + rng.normal(0, step, n)
    v = 0.9 * a + 0.8 * b - 0.7 * c + rng.laplace(0, 0.2 * step, n)
    cols = [np.rint(np.clip(x, 0, top)).astype(np.int32) for x in (a, b, c, v)]
    w = search.IrlpCost(*cols, np.array([0, n])).irls_l1()
    X = np.stack(cols[:3], 1).astype(np.float64)
    host = search.irls_l1(X, cols[3].astype(np.float64))
    assert w is not None and np.abs(w - host).max() < 1e-9


def test_irls_leaves_degenerate_fits_to_the_host():
    from meshpress_amd.encoder import search
    n = 1000
    rng = np.random.default_rng(0)
    c = rng.integers(0, 4096, n).astype(np.int32)
    z = np.zeros(n, np.int32)
    off = np.array([0, n])
    assert search.IrlpCost(c, c, c, c, off).irls_l1() is None        # a = b = c
    assert search.IrlpCost(z, z, z, z, off).irls_l1() is None        # all zero
    assert search.IrlpCost(c + 7, c + 7, c, c, off).irls_l1() is None   # a = b
    assert search.IrlpCost(z[:0], z[:0], z[:0], z[:0], np.array([0, 0])).irls_l1() is None


@pytest.mark.parametrize("n_streams", [1, 4, 5, 6145, 12287, 12288, 12289])
@pytest.mark.parametrize("kind", ["small", "extreme"])
def test_long_streams_among_short_ones(n_streams, kind):
    """Streams on both sides of the 1,024 values from which a whole wave takes
    one, anywhere among a wave's four, and of the line from which no workgroup
    waits for them."""
    from meshpress_amd.encoder import search
    rng = np.random.default_rng(n_streams)
    lens = rng.integers(0, 4, n_streams)
    for i, n in ((0, 1024), (1, 1025), (n_streams // 2, 5000), (n_streams - 1, 1100)):
        lens[min(i, n_streams - 1)] = n
    off = np.concatenate(([0], np.cumsum(lens))).astype(np.int64)
    vals = np.rint(rng.laplace(0, 20, off[-1])).astype(np.int32)
    if kind == "extreme":
        vals[::17] = -(1 << 31)
        vals[3::29] = (1 << 31) - 1
    want = coder_costs(zigzag(vals), off).astype(np.int64)
    assert np.array_equal(search.stream_costs(vals, off), want)
    tagk, bits = search.select_codes(vals, off)
    rk, ek = want[:, :12].argmin(1), want[:, 12:].argmin(1)
    rb, eb = want[:, :12].min(1), want[:, 12:].min(1)
    rice = rb <= eb
    assert np.array_equal(bits, np.where(rice, rb, eb))
    assert np.array_equal(tagk, np.stack([np.where(rice, 1, 2), np.where(rice, rk, ek)], 1).astype(np.uint8))
