"""Own keys of a many-row attention call (no or few cached keys) at the edges of the tiled kernel and of its plan: the
rows where it takes over from the few-row kernel, ragged tiles and runs, windows shorter than the call, groups that do
not fill a row block, and every head size, against FP64.

Bar: max |err| / RMS <= 3e-5. A score of magnitude 8 (in powers of two) is off by at most about 8 * 2^-22 after D
FP32 additions of products good to 2^-24, so a weight by 1.4e-6 of itself; an output adds up as many of those as keys
carry weight, and its own rounding, against an RMS that falls with the number of keys averaged: 1e-5 was the largest
measured at 1500 rows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [  # heads, kv_heads, head_dim, rows, cached, window
    (32, 8, 128, 48, 0, 0), (32, 8, 128, 49, 0, 0), (32, 8, 128, 129, 0, 0), (32, 8, 128, 700, 0, 0),
    (16, 4, 256, 32, 0, 0), (16, 4, 256, 33, 0, 0), (16, 4, 256, 188, 0, 0), (16, 4, 256, 390, 0, 0),
    (16, 8, 64, 2, 0, 0), (16, 8, 64, 9, 0, 0), (16, 8, 64, 65, 0, 0), (16, 8, 64, 1100, 0, 0),
    (8, 8, 128, 97, 0, 0),       # one head per KV head: 32-row blocks
    (8, 1, 64, 67, 0, 0),        # eight: 4-row blocks
    (6, 2, 128, 75, 0, 0),       # three: 10-row blocks of 30 columns
    (10, 2, 256, 61, 0, 0),      # five: 6-row blocks of 30 columns
    # the rows on either side of the few-row kernel, at each size of group
    (16, 8, 64, 48, 0, 0), (16, 8, 64, 49, 0, 0), (8, 1, 64, 48, 20, 30), (8, 8, 128, 48, 0, 0), (8, 8, 128, 49, 0, 0),
    (32, 8, 128, 52, 0, 0), (32, 8, 128, 53, 0, 0), (4, 4, 256, 20, 0, 0), (4, 4, 256, 21, 0, 0), (8, 4, 256, 28, 0, 0),
    (8, 4, 256, 29, 0, 0), (16, 4, 256, 36, 0, 0), (16, 4, 256, 37, 0, 0), (8, 1, 256, 33, 0, 0), (8, 1, 256, 34, 0, 0),
    (32, 8, 128, 300, 0, 100), (16, 4, 256, 200, 0, 33), (16, 8, 64, 400, 0, 1), (32, 8, 128, 530, 40, 500),
]


# The tiled scan of many rows: odd and even tile counts (two key halves), splits, a last tile that is half empty, windows
# that end inside a tile, rings not full and overwritten, row blocks that are not filled
SCANS = [  # heads, kv_heads, head_dim, rows, cached, window, ring slots
    (32, 8, 128, 128, 1000, 0, 0), (32, 8, 128, 131, 1057, 0, 0), (32, 8, 128, 200, 1500, 300, 0),
    (32, 8, 128, 140, 700, 500, 1040), (32, 8, 128, 160, 2600, 1024, 1088), (16, 4, 256, 128, 1, 0, 0),
    (16, 4, 256, 150, 333, 0, 0), (16, 4, 256, 190, 1400, 1024, 1040), (16, 8, 64, 129, 31, 0, 0),
    (16, 8, 64, 257, 992, 0, 0), (8, 8, 128, 161, 1056, 0, 0), (6, 2, 128, 135, 1100, 0, 0), (10, 2, 256, 128, 95, 64, 0),
    (8, 1, 64, 130, 200, 0, 0),
    # rings about to wrap and just wrapped, below the rows that share tiles too
    (32, 8, 128, 20, 700, 500, 1040), (16, 4, 256, 40, 1040, 1024, 1040), (16, 4, 256, 40, 1041, 1000, 1040),
    (16, 8, 64, 130, 1088, 1024, 1088), (16, 8, 64, 130, 1089, 1024, 1088),
]


def run(hip, pkg, heads, kv, d, n, cached, window, ring=0, fp8=False, call=None):
    """The largest error over the RMS of one call against FP64."""
    rng = np.random.default_rng(heads * n + d + window + cached)

    def unit(*shape):
        x = rng.standard_normal(shape).astype(np.float32)
        return x / np.linalg.norm(x, axis=-1, keepdims=True)

    q, k = (unit(n, heads, d) * d).astype(np.float32), unit(n, kv, d)
    v = rng.standard_normal((n, kv, d)).astype(np.float32)
    # cached rows exact in BF16 and in E4M3 with a scale: one magnitude, either sign
    ck = np.sign(rng.standard_normal((cached, kv, d))).astype(np.float32) / np.float32(2.0 ** np.ceil(np.log2(d) / 2))
    cv = np.sign(rng.standard_normal((cached, kv, d))).astype(np.float32)
    cache = hip.kv_cache(kv, d, cached + n, ring, pkg.KV_FP8 if fp8 else pkg.KV_BF16)
    for at in range(0, cached, 500):   # in pieces: a ring's later rows overwrite its first
        e = min(cached, at + 500)
        cache.store(at, e - at, hip.array(ck[at:e]), hip.array(cv[at:e]))
    dq, dk, dv, out = hip.array(q), hip.array(k), hip.array(v), hip.array(np.full((n, heads, d), 7, np.float32))
    (call or hip.attention)(cache, dq, dk, dv, out, n, cached, heads, window)
    got = out.numpy().reshape(n, heads, d)
    cache.destroy()

    keys, vals = np.concatenate([ck, k]).astype(np.float64), np.concatenate([cv, v]).astype(np.float64)
    at, mine = np.arange(cached + n), np.arange(cached, cached + n)[:, None]
    hide = (at[None, :] > mine) | ((mine - at[None, :] >= window) if window else False)
    if ring:
        hide = hide | (at[None, :] < cached - ring)   # overwritten
    exact = np.empty((n, heads, d))
    for h in range(heads):
        s = q[:, h].astype(np.float64) @ keys[:, h // (heads // kv)].T / np.sqrt(d)
        s[hide] = -np.inf
        p = np.exp(s - s.max(axis=1, keepdims=True))
        exact[:, h] = (p / p.sum(axis=1, keepdims=True)) @ vals[:, h // (heads // kv)]
    return np.max(np.abs(got - exact)) / np.sqrt(np.mean(exact ** 2))


@pytest.mark.parametrize("heads,kv,d,n,cached,window", CASES)
def test_own_keys_at_the_edges(hip, pkg, heads, kv, d, n, cached, window):
    err = run(hip, pkg, heads, kv, d, n, cached, window)
    assert err <= 3e-5, err


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,kv,d,n,cached,window,ring", SCANS)
def test_many_row_scan_at_the_edges(hip, pkg, heads, kv, d, n, cached, window, ring, fp8):
    """Bar 6e-5: a cached key's weight is off by up to 2^-17 (two BF16 terms), 8e-6 of an output that one key makes,
    against an RMS over outputs that average hundreds of them (about a seventh of a value)."""
    err = run(hip, pkg, heads, kv, d, n, cached, window, ring, fp8)
    assert err <= 6e-5, err


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("heads,kv,d,n,cached,window,ring", SCANS)
def test_shared_tiles_at_the_edges(hip, pkg, monkeypatch, heads, kv, d, n, cached, window, ring, fp8):
    """The same calls with their tiles shared, also where each block's own tiles are faster; one and several splits."""
    monkeypatch.setenv("XTG_ATTN_SHARED", "1")
    err = run(hip, pkg, heads, kv, d, n, cached, window, ring, fp8)
    assert err <= 6e-5, err
    monkeypatch.setenv("XTG_ATTN_SPLITS", "3")
    err = run(hip, pkg, heads, kv, d, n, cached, window, ring, fp8)
    assert err <= 6e-5, err


def test_an_infinite_value_stays_infinite(hip):
    """A visible infinity of V gives an infinity (the split of a value into terms would make it NaN), and rows before
    its 32-row tile do not see it."""
    n, heads, d, at = 160, 4, 128, 100
    rng = np.random.default_rng(5)
    q, k, v = (rng.standard_normal((n, heads, d)).astype(np.float32) * 0.1 for _ in range(3))
    v[at, 0, 3] = np.inf
    cache = hip.kv_cache(heads, d, n)
    out = hip.array(np.zeros((n, heads, d), np.float32))
    hip.attention(cache, hip.array(q), hip.array(k), hip.array(v), out, n, 0, heads, 0)
    got = out.numpy().reshape(n, heads, d)
    cache.destroy()
    assert (got[at:, 0, 3] == np.inf).all()
    assert np.isfinite(got[:at // 32 * 32]).all() and np.isfinite(got[:, 1:]).all()


@pytest.mark.parametrize("heads,kv,d,n,window,ats", [
    (4, 4, 128, 160, 0, (100, 159)), (32, 8, 128, 150, 0, (31, 32, 149)), (16, 4, 256, 70, 20, (0, 40, 69)),
    (8, 1, 64, 131, 50, (64, 65, 130))])
def test_rows_that_do_not_see_a_value_stay_finite(hip, heads, kv, d, n, window, ats):
    """Infinities and a NaN in V: the rows that see their key have them, every other row and dim is bit for bit what it
    is with zeros in their place."""
    rng = np.random.default_rng(n)
    q, k, v = (rng.standard_normal((n, h, d)).astype(np.float32) * 0.1 for h in (heads, kv, kv))
    odd = [(at, i % kv, 3 + 29 * i, x) for i, at in enumerate(ats) for x in ((np.inf, -np.inf, np.nan)[i],)]
    cache = hip.kv_cache(kv, d, n)
    out = hip.array(np.zeros((n, heads, d), np.float32))

    def call(v):
        hip.attention(cache, hip.array(q), hip.array(k), hip.array(v), out, n, 0, heads, window)
        return out.numpy().reshape(n, heads, d).copy()

    for at, h, dim, _ in odd:
        v[at, h, dim] = 0
    want = call(v)
    assert np.isfinite(want).all()
    for at, h, dim, x in odd:
        v[at, h, dim] = x
        for row in range(at, min(n, at + window) if window else n):
            want[row, h * (heads // kv):(h + 1) * (heads // kv), dim] = x
    got = call(v)
    cache.destroy()
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("bits", [0x3f80ffff, 0x3f807fc0, 0x3fd5a5a5])
@pytest.mark.parametrize("heads,kv,d,n", [(4, 4, 64, 70), (2, 2, 128, 100), (2, 2, 256, 70)])
def test_products_of_scores_keep_their_bits(hip, heads, kv, d, n, bits):
    """Scores that are sums of d products of 64 which cancel, so that the sums' roundings vanish and what is left out of
    the products shows: half of them of two values with full mantissas, half of one and its BF16 rounding (whose products
    are whole). Bar: d / 2 products of |x y| each short of at most 2^-24 + 2^-34 of it, times ln 2, and 1e-5 of the
    weight for the other roundings."""
    scale = next(s for s in np.nextafter(np.float32(np.log(2)), np.float32([0, 1, 0.69314718])) if
                 np.float32(s) * np.float32(1.44269504088896341) == 1)   # scores in powers of two, as they are
    x = np.uint32(bits).view(np.float32)
    xb = np.uint32((bits + 0x7fff + ((bits >> 16) & 1)) & 0xffff0000).view(np.float32)
    q = np.full((n, heads, d), x * 64 / np.exp2(np.floor(np.log2(x * x))), np.float32)
    k, v = np.zeros((n, kv, d), np.float32), np.zeros((n, kv, d), np.float32)
    k[0, :, 0::2], k[0, :, 1::2] = x, -xb
    k[1, :, 0::2] = ((x - xb).view(np.uint32) & np.uint32(0xffff0000)).view(np.float32)   # about its score, whole
    v[0] = 1
    w = np.exp2(q[0, 0].astype(np.float64) @ k[:, 0].T.astype(np.float64))
    exact = w[0] / np.cumsum(w)
    cache = hip.kv_cache(kv, d, n)
    out = hip.array(np.zeros((n, heads, d), np.float32))
    hip.attention(cache, hip.array(q), hip.array(k), hip.array(v), out, n, 0, heads, 0, float(scale))
    got = out.numpy().reshape(n, heads, d).astype(np.float64)
    cache.destroy()
    short = d / 2 * float(q[0, 0, 0]) * float(x) * (2.0 ** -24 + 2.0 ** -34)
    err = np.max(np.abs(got - exact[:, None, None]) / exact[:, None, None])
    assert err <= short * np.log(2) + 1e-5, (err, short)


@pytest.mark.parametrize("d,n", [(64, 70), (128, 70), (256, 70)])
def test_values_at_the_ends_of_the_range(hip, d, n):
    """FP32's largest value in V (BF16 would round it to infinity), minus infinity in K (a weight of 0 for these q, all
    above 0), and a NaN whose bits are all in the lower half, which its row and the later ones show. Bar: 3e-5 of the
    value, as above (6 keys' worth of relative weight errors at most)."""
    heads = 2
    rng = np.random.default_rng(d)
    q = rng.uniform(0.5, 1, (n, heads, d)).astype(np.float32)
    k, v = (rng.standard_normal((n, heads, d)).astype(np.float32) * 0.1 for _ in range(2))
    k[10, :, 5] = -np.inf
    k[60, 1, 7] = np.uint32(0x7f800001).view(np.float32)
    v[30, 0, 2] = np.finfo(np.float32).max
    cache = hip.kv_cache(heads, d, n)
    out = hip.array(np.zeros((n, heads, d), np.float32))
    hip.attention(cache, hip.array(q), hip.array(k), hip.array(v), out, n, 0, heads, 0)
    got = out.numpy().reshape(n, heads, d).astype(np.float64)
    cache.destroy()
    assert np.isnan(got[60:, 1]).all()
    k[60, 1] = 0   # of no row below
    for h in range(heads):
        s = q[:, h].astype(np.float64) @ k[:, h].astype(np.float64).T / np.sqrt(d)
        s[np.arange(n)[None, :] > np.arange(n)[:, None]] = -np.inf
        s[:, 10] = -np.inf
        rows = n if h == 0 else 60
        p = np.exp(s[:rows] - s[:rows].max(axis=1, keepdims=True))
        exact = (p / p.sum(axis=1, keepdims=True)) @ v[:, h].astype(np.float64)
        assert np.isfinite(got[:rows, h]).all()
        scale = np.where(np.abs(exact) > 1, np.abs(exact), 0.02)   # the other values' size
        assert np.max(np.abs(got[:rows, h] - exact) / scale) <= 3e-5
