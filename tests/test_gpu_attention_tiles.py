"""Attention with many query rows, where 64 (row, head) pairs share a workgroup's keys: pairs around 64, key counts
around 64, windows, padded head sizes, the keys in one part and in several.  Against the oracle, and against the rows'
kernels (the same call sixteen rows at a time) where the cache or the queries hold infinities or NaN."""
import numpy as np
import pytest

from tessera_amd import synth
from test_gpu_attention import KINDS, attend, cache, expected

pytestmark = pytest.mark.gpu

# too little work for it: the rows' kernels
FEW = [
    (410, 410, 2, 1, 64, 0, 0), (101, 449, 4, 4, 128, 348, 0), (203, 300, 6, 2, 256, 97, 70), (137, 140, 9, 3, 96, 3, 0),
    (401, 200, 1, 1, 64, 100, 0),
]
ONE_PART = [
    # m, n, heads, kv_heads, head_dim, q_base, window
    (410, 410, 8, 4, 64, 0, 0),          # 820 pairs a key head: the last workgroup has 52
    (101, 449, 16, 16, 128, 348, 0),     # a pair a row; one key more than seven tiles
    (203, 300, 24, 8, 256, 97, 70),      # a window shorter than two tiles
    (137, 140, 27, 9, 96, 3, 0),         # padded to 128; rows across workgroups
    (401, 200, 4, 4, 64, 100, 0),        # rows past the last key
]
PARTS = [
    (33, 2100, 24, 4, 256, 2067, 0),     # parts of the keys
    (40, 1100, 8, 8, 128, 1060, 0),
    (70, 1300, 8, 8, 64, 1230, 820),     # parts of which early rows see none of the last, late rows little of the first
    (20, 1537, 16, 4, 160, 1517, 0),     # padded to 256
]


@pytest.mark.parametrize("kind", ["f16", "q8", "q4", "fp8"])
@pytest.mark.parametrize("case", FEW + ONE_PART + PARTS)
def test_attention_tiles(backend, kind, case):
    m, n, heads, kv_heads, head_dim, q_base, window = case
    g = synth.rng(n + head_dim + KINDS[kind])
    width = kv_heads * head_dim
    q = g.standard_normal((m + 3, heads * head_dim)).astype(np.float32)
    k, ks = cache(g, kind, n, width)
    v, vs = cache(g, kind, n, width)
    want = expected(kind, q[2:2 + m], k, v, ks, vs, m, n, heads, kv_heads, head_dim, q_base, window)
    got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, q_base, window, row_base=2)
    # sums in another order, as test_gpu_attention.py (twice it where parts are merged)
    assert np.max(np.abs(got[2:2 + m] - want)) <= 4e-6 * max(1.0, np.max(np.abs(want)))
    assert np.all(got[:2] == 7.0) and np.all(got[2 + m:] == 7.0)


SPECIAL = [(101, 449, 16, 16, 128), (33, 2100, 24, 4, 256), (410, 410, 8, 4, 64)]


@pytest.mark.parametrize("heads", [4, 16])
def test_attention_tiles_not_causal(backend, heads):
    m, n, kv_heads, head_dim = 101, 203, heads, 128
    g = synth.rng(5)
    q = g.standard_normal((m, heads * head_dim)).astype(np.float32)
    k, v = (cache(g, "f16", n, kv_heads * head_dim)[0] for _ in range(2))
    want = expected("f16", q, k, v, None, None, m, n, heads, kv_heads, head_dim, 0, 0, causal=0)
    got = attend(backend, "f16", q, k, v, None, None, m, n, heads, kv_heads, head_dim, 0, 0, causal=0)
    assert np.max(np.abs(got - want)) <= 2e-6 * max(1.0, np.max(np.abs(want)))


@pytest.mark.parametrize("shape", [*SPECIAL, (101, 449, 4, 4, 128), (410, 410, 2, 1, 64)])
@pytest.mark.parametrize("what", ["key", "key-", "value", "value nan", "query", "key scale", "value scale", "zeros"])
def test_attention_tiles_special_values(backend, shape, what):
    m, n, heads, kv_heads, head_dim = shape
    kind = "q8" if "scale" in what else "f16"
    g = synth.rng(n)
    q = g.standard_normal((m, heads * head_dim)).astype(np.float32)
    k, ks = cache(g, kind, n, kv_heads * head_dim)
    v, vs = cache(g, kind, n, kv_heads * head_dim)
    at = n - m // 2                       # some rows see it, some do not
    if what == "key":
        k[at, 3] = np.inf
    elif what == "key-":
        k[at, :head_dim] = -np.inf
    elif what == "value":
        v[at, 5] = np.inf
    elif what == "value nan":
        v[at, 5] = np.nan
    elif what == "query":
        q[m // 2, 7] = np.inf
    elif what == "key scale":
        ks[at] = np.inf
    elif what == "value scale":
        vs[at] = np.inf
    else:
        q[m // 3] = 0.0
        k[:] = 0
    got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, 0)
    want = np.empty_like(got)
    for r in range(0, m, 16):
        rows = min(16, m - r)
        want[r:r + rows] = attend(backend, kind, np.ascontiguousarray(q[r:r + rows]), k, v, ks, vs, rows, n, heads, kv_heads,
                                  head_dim, n - m + r, 0)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got), np.isinf(want))
    fine = np.isfinite(want)
    assert np.array_equal(got[~fine & ~np.isnan(want)], want[~fine & ~np.isnan(want)])
    assert np.max(np.abs(got[fine] - want[fine]), initial=0.0) <= 4e-6 * max(1.0, np.max(np.abs(want[fine]), initial=0.0))


def softmax_rows(q, k, v, heads, kv_heads, head_dim, q_base):
    """Causal attention in float64 over keys and values as the cache stands for them."""
    m, n = q.shape[0], k.shape[0]
    out = np.empty((m, heads * head_dim))
    q, k, v = (x.astype(np.float64).reshape(x.shape[0], -1, head_dim) for x in (q, k, v))
    for h in range(heads):
        s = q[:, h] @ k[:, h * kv_heads // heads].T / np.sqrt(head_dim)
        s[np.arange(n)[None, :] > q_base + np.arange(m)[:, None]] = -np.inf
        w = np.exp(s - s.max(1, keepdims=True))
        out[:, h * head_dim:(h + 1) * head_dim] = w @ v[:, h * kv_heads // heads] / w.sum(1, keepdims=True)
    return out


@pytest.mark.parametrize("kind", ["f16", "q8"])
@pytest.mark.parametrize("shape", SPECIAL)
def test_attention_tiles_key_of_nearly_all_weight_and_no_value(backend, kind, shape):
    """The first key takes all but some e^-20 = 2^-29 of every row's weight and its values are zero, so that the result is
    made of the small weights alone.  They are off by 2^-50 of the largest over an fp16 cache and by 2^-45 of the largest
    contribution over a quantized one: 2^-16 of themselves at most; a score of 20 in fp32 moves them by 20 * 2^-24 < 2^-19.
    The values' signs are random, so a row's sum has its weights' relative error.  (Measured: 1.3e-6.)"""
    m, n, heads, kv_heads, head_dim = shape
    g = synth.rng(n + 1)
    q = g.standard_normal((m, heads, head_dim)).astype(np.float32)
    q[:, :, 0] = 5.0
    k, ks = cache(g, kind, n, kv_heads * head_dim)
    v, vs = cache(g, kind, n, kv_heads * head_dim)
    k, v = (x.copy() if kind == "f16" else x.reshape(n, -1).view(np.int8).copy() for x in (k, v))
    by_head = k.reshape(n, kv_heads, head_dim)
    by_head[:, :, 0] = 0
    by_head[0] = 0
    v[0] = 0
    top = 4.0 * np.sqrt(head_dim)                           # score 20
    by_head[0, :, 0] = top if kind == "f16" else 127
    if kind == "q8":
        ks[0] = top / 127
    keys, values = (x.astype(np.float64) * (1.0 if s is None else s[:, None].astype(np.float64)) for x, s in ((k, ks), (v, vs)))
    q = q.reshape(m, heads * head_dim)
    want = softmax_rows(q, keys, values, heads, kv_heads, head_dim, n - m)
    got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, 0)
    rows = slice(1, None) if n == m else slice(None)        # (the first row of a cache that starts with it sees that key alone)
    err = np.linalg.norm(got[rows] - want[rows]) / np.linalg.norm(want[rows])
    assert err <= 2.0 ** -16, err
