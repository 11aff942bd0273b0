"""Attention over every kind of cache at the edges of its dispatch: head sizes around the padded sizes of
the matrix kernels (64, 128, 256) and ones their loads do not divide, query heads per key head around the
columns of a matrix instruction, key counts around the tiles, a value scale of zero, rising and falling
scales.  Against the oracle's restatements; bound as in test_gpu_trunk.py (sums in another order)."""
import numpy as np
import pytest
import torch

import oracle
from tessera_amd import synth
from util import run

pytestmark = pytest.mark.gpu

KINDS = {"f32": 0, "f16": 1, "q8": 2, "q4": 3, "fp8": 4}


def cache(g, kind, n, width, gain=None):
    """Keys or values as the cache holds them: (elements or codes, scales or None)."""
    x = g.standard_normal((n, width)).astype(np.float32)
    if gain is not None:
        x *= gain[:, None].astype(np.float32)
    if kind == "f32":
        return x, None
    if kind == "f16":
        return x.astype(np.float16), None
    if kind == "fp8":
        return oracle.quantize_fp8_pack(x, n, width)
    return oracle.quantize_kv(x, n, width, 8 if kind == "q8" else 4)


def attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, q_base, window, row_base=0, causal=1, split=0):
    """The attention id of the cache kind, or its split form and the merge; rows of the whole batch buffer."""
    total = q.shape[0]
    dq, dk, dv = backend.Upload(q), backend.Upload(k), backend.Upload(v)
    scales = [] if ks is None else [backend.Upload(ks), backend.Upload(vs)]
    dout = backend.Upload(np.full((total, heads * head_dim), 7.0, np.float32))
    tail = [window, int(kind == "f16"), causal] if ks is None else [window, KINDS[kind] - 2]
    base = "attention" if ks is None else f"attention_{kind}"
    if not split:
        run(backend, base, [dq, dk, dv, *scales, dout], [m, n, heads, kv_heads, head_dim, q_base, row_base, *tail], grid=(m * heads, 1, 1))
    else:
        parts = [backend.AllocateBuffer(4 * m * heads * split * w) for w in (head_dim, 1, 1)]
        run(backend, base + "_split", [dq, dk, dv, *scales, *parts], [m, n, heads, kv_heads, head_dim, q_base, *tail, split],
            grid=(m * heads * split, 1, 1))
        run(backend, "attention_combine", [*parts, dout], [m, heads, head_dim, split], grid=(m * heads, 1, 1))
    backend.Synchronize()
    return backend.CopyD2H(dout, dtype=np.float32).reshape(total, heads * head_dim)


def expected(kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, q_base, window, causal=1):
    if ks is None:
        return oracle.attention(q, k, v, m, n, heads, kv_heads, head_dim, q_base, window, kind == "f16", bool(causal))
    return oracle.attention_quant(q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, kind, q_base, window)


CASES = [
    # m, n, heads, kv_heads, head_dim, q_base, window
    (1, 1, 1, 1, 64, 0, 0),
    (1, 31, 4, 4, 64, 30, 0),            # one head a key head, a tile less one key
    (1, 33, 8, 1, 128, 32, 0),           # all eight columns
    (2, 128, 9, 1, 128, 126, 0),         # nine heads: a second block of one
    (1, 129, 17, 1, 64, 128, 0),         # three blocks; over fp32 two of sixteen
    (1, 300, 16, 4, 64, 299, 0),
    (3, 517, 24, 4, 256, 514, 0),
    (1, 700, 6, 2, 256, 699, 250),       # window
    (2, 90, 6, 3, 96, 88, 0),            # padded to 128
    (2, 90, 4, 2, 80, 88, 0),            # divides the runs of some kinds only
    (2, 70, 4, 2, 160, 60, 0),           # padded to 256
    (1, 45, 2, 1, 16, 44, 0),
    (2, 50, 2, 1, 24, 48, 0),
    (2, 50, 8, 4, 34, 48, 0),            # no kind's runs
]


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("case", CASES)
def test_attention_edges(backend, kind, case):
    m, n, heads, kv_heads, head_dim, q_base, window = case
    g = synth.rng(n * 7 + head_dim + KINDS[kind])
    width = kv_heads * head_dim
    q = g.standard_normal((m + 3, heads * head_dim)).astype(np.float32)
    k, ks = cache(g, kind, n, width)
    v, vs = cache(g, kind, n, width)
    want = expected(kind, q[2:2 + m], k, v, ks, vs, m, n, heads, kv_heads, head_dim, q_base, window)
    bound = 2e-6 * max(1.0, np.max(np.abs(want)))
    got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, q_base, window, row_base=2)
    assert np.max(np.abs(got[2:2 + m] - want)) <= bound
    assert np.all(got[:2] == 7.0) and np.all(got[2 + m:] == 7.0)
    for split in (1, 3, 7):
        got = attend(backend, kind, np.ascontiguousarray(q[2:2 + m]), k, v, ks, vs, m, n, heads, kv_heads, head_dim, q_base, window,
                     split=split)
        assert np.max(np.abs(got - want)) <= 2 * bound, split


@pytest.mark.parametrize("kind", ["q8", "q4", "fp8"])
@pytest.mark.parametrize("shape", ["rising", "falling", "zeros", "tiny"])
def test_attention_value_scales_over_many_binades(backend, kind, shape):
    """The values' scales enter the weights under a power of two that follows the largest so far."""
    m, n, heads, kv_heads, head_dim = 2, 400, 6, 2, 128
    g = synth.rng(900 + len(shape))
    gain = {"rising": np.exp2(np.linspace(-40, 10, n)), "falling": np.exp2(np.linspace(10, -40, n)),
            "zeros": np.where(np.arange(n) < 200, 0.0, 1.0), "tiny": np.full(n, 1e-30)}[shape]
    q = g.standard_normal((m, heads * head_dim)).astype(np.float32)
    k, ks = cache(g, kind, n, kv_heads * head_dim)
    v, vs = cache(g, kind, n, kv_heads * head_dim, gain)
    want = expected(kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, 0)
    got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, 0)
    assert np.max(np.abs(got - want)) <= 4e-6 * np.max(np.abs(want))


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("gain", [2.0 ** -60, 2.0 ** 40])
def test_attention_query_magnitudes(backend, kind, gain):
    """Queries far from 1 (their keys far the other way where the cache can hold that, else scores near zero
    or a one-hot softmax): the power of two under which they enter is undone exactly."""
    m, n, heads, kv_heads, head_dim = 1, 150, 4, 2, 64
    g = synth.rng(77)
    q = (g.standard_normal((m, heads * head_dim)) * gain).astype(np.float32)
    k, ks = cache(g, kind, n, kv_heads * head_dim)
    if kind == "f32":
        k = (k / np.float32(gain)).astype(np.float32)
    v, vs = cache(g, kind, n, kv_heads * head_dim)
    want = expected(kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - 1, 0)
    got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - 1, 0)
    assert np.max(np.abs(got - want)) <= 4e-6 * max(1.0, np.max(np.abs(want)))


# spans of keys of score -inf: one, the last one, whole tiles of every kernel, the first 64 and more, a whole part
@pytest.mark.parametrize("kind", ["f32", "f16"])
@pytest.mark.parametrize("head_dim", [64, 128, 256, 34])
@pytest.mark.parametrize("spans", [[(7, 8)], [(299, 300)], [(0, 40), (64, 96)], [(0, 100)], [(150, 300)]])
def test_attention_keys_of_infinite_score(backend, kind, head_dim, spans):
    """A key with an infinite element whose score is -inf has the weight 0: the rest of the row is as without it."""
    m, n, heads, kv_heads = 2, 301, 6, 2
    g = synth.rng(1200 + head_dim)
    q = g.standard_normal((m, heads * head_dim)).astype(np.float32)
    k, _ = cache(g, kind, n, kv_heads * head_dim)
    v, _ = cache(g, kind, n, kv_heads * head_dim)
    q, k = q.reshape(m, heads, head_dim), k.reshape(n, kv_heads, head_dim)
    q[:, :, 3] = np.abs(q[:, :, 3]) + np.float32(0.1)
    q[0, 0, 3] = 1.0                                   # (no second term)
    q[0, 1, 3] = 0.1                                   # (a negative one)
    q[:, :, 5] = -q[:, :, 3]
    out = np.zeros(n, bool)
    for lo, hi in spans:
        out[lo:hi] = True
    k[out, :, 3] = -np.inf
    k[out[:, None] & (np.arange(kv_heads) == 1), 5] = np.inf
    q, k = q.reshape(m, -1), k.reshape(n, -1)
    want = expected(kind, q, k, v, None, None, m, n, heads, kv_heads, head_dim, n - m, 0)
    assert np.isfinite(want).all()
    bound = 2e-6 * max(1.0, np.max(np.abs(want)))
    for split in (0, 1, 4):
        got = attend(backend, kind, q, k, v, None, None, m, n, heads, kv_heads, head_dim, n - m, 0, split=split)
        assert np.max(np.abs(got - want)) <= 2 * bound, split


@pytest.mark.parametrize("kind", ["f32", "f16"])
@pytest.mark.parametrize("head_dim", [64, 256, 34])
@pytest.mark.parametrize("n", [1, 33, 290])
def test_attention_infinite_values(backend, kind, head_dim, n):
    """An infinite value makes its own element of the rows that see it infinite, with its sign, and no other;
    also as the last key, whose row stands in for the keys past the end."""
    heads, kv_heads, m = 6, 2, min(2, n)
    g = synth.rng(1300 + n + head_dim)
    q = (0.1 * g.standard_normal((m, heads * head_dim))).astype(np.float32)
    k, _ = cache(g, kind, n, kv_heads * head_dim)
    v, _ = cache(g, kind, n, kv_heads * head_dim)
    v = v.reshape(n, kv_heads, head_dim)
    v[n // 2, 0, 1] = np.inf
    v[n - 1, 1, 9] = -np.inf
    v = v.reshape(n, -1)
    want = expected(kind, q, k, v, None, None, m, n, heads, kv_heads, head_dim, n - m, 0)
    assert not np.isnan(want).any() and np.isinf(want).any()
    for split in (0, 3):
        got = attend(backend, kind, q, k, v, None, None, m, n, heads, kv_heads, head_dim, n - m, 0, split=split)
        inf = np.isinf(want)
        assert np.array_equal(got[inf], want[inf]), split
        assert np.max(np.abs(got[~inf] - want[~inf])) <= 4e-6, split


@pytest.mark.parametrize("kind", ["f32", "f16"])
def test_attention_nan_stays_in_its_rows(backend, kind):
    """A NaN in a query spoils that row's head, one in a key the rows that see it, one in a value their element."""
    m, n, heads, kv_heads, head_dim = 4, 90, 4, 2, 64
    g = synth.rng(1400)
    q = g.standard_normal((m, heads * head_dim)).astype(np.float32)
    k, _ = cache(g, kind, n, kv_heads * head_dim)
    v, _ = cache(g, kind, n, kv_heads * head_dim)
    q[0, 70] = np.nan                       # row 0, head 1
    k[88, 5] = np.nan                       # rows 2 and 3, heads 0 and 1
    v[87, 64 + 6] = np.nan                  # rows 1 to 3, heads 2 and 3, element 6
    got = attend(backend, kind, q, k, v, None, None, m, n, heads, kv_heads, head_dim, n - m, 0).reshape(m, heads, head_dim)
    bad = np.zeros(got.shape, bool)
    bad[0, 1] = True
    bad[2:, :2] = True
    bad[1:, 2:, 6] = True
    assert np.array_equal(np.isnan(got), bad)


def attention_f64(kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, q_base):
    """softmax(Q K^T / sqrt(head_dim)) V in float64, causal, over the numbers that the cache holds."""
    if ks is not None:
        k, v = (oracle.dequant_kv(c, np.ones(n, np.float32), n, kv_heads * head_dim, kind).astype(np.float64) *
                np.asarray(s, np.float64)[:, None] for c, s in ((k, ks), (v, vs)))
    k, v = (np.asarray(x, np.float64).reshape(n, kv_heads, head_dim) for x in (k, v))
    q, out = q.astype(np.float64).reshape(m, heads, head_dim), np.empty((m, heads, head_dim))
    for i in range(m):
        for h in range(heads):
            s = k[:q_base + i + 1, h // (heads // kv_heads)] @ q[i, h] / np.sqrt(head_dim)
            p = np.exp(s - s.max())
            out[i, h] = p @ v[:q_base + i + 1, h // (heads // kv_heads)] / p.sum()
    return out.reshape(m, heads * head_dim)


@pytest.mark.parametrize("kind", ["q8", "q4", "fp8"])
@pytest.mark.parametrize("at", [3, 200, 399])
@pytest.mark.parametrize("binades", [12, 20, 30, 45, 60])
def test_attention_weight_on_a_small_value_scale(backend, kind, at, binades):
    """All the weight on one key whose value scale is 2^-binades of the others', which have none: the result keeps
    its precision however large the scales of what does not contribute."""
    m, n, heads, kv_heads, head_dim = 1, 400, 6, 2, 128
    g = synth.rng(1500 + binades)
    q = g.standard_normal((m, heads * head_dim)).astype(np.float32)
    k = (0.01 * g.standard_normal((n, kv_heads, head_dim))).astype(np.float32)
    for h in range(kv_heads):                                    # along every head of the group
        k[at, h] = q.reshape(heads, head_dim)[h * 3:h * 3 + 3].mean(axis=0) * 150.0
    k = k.reshape(n, -1)
    k, ks = (oracle.quantize_fp8_pack(k, n, kv_heads * head_dim) if kind == "fp8" else
             oracle.quantize_kv(k, n, kv_heads * head_dim, 8 if kind == "q8" else 4))
    v, vs = cache(g, kind, n, kv_heads * head_dim)
    vs[at] *= np.float32(2.0 ** -binades)
    want = attention_f64(kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m)
    assert np.max(np.abs(want)) < 8.0 * 2.0 ** -binades         # (the others' weights vanish)
    for split in (0, 4):
        got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, 0, split=split)
        assert np.max(np.abs(got - want)) <= 1e-6 * np.max(np.abs(want)), split


@pytest.mark.parametrize("kind", list(KINDS))
def test_attention_query_range_inside_a_head(backend, kind):
    """One query element 2^18 times the others, on a dimension where every key is zero: the scores come from the
    small ones alone and keep their precision."""
    m, n, heads, kv_heads, head_dim = 2, 400, 6, 2, 128
    g = synth.rng(1600)
    q = g.standard_normal((m, heads, head_dim)).astype(np.float32)
    q[:, :, 17] = 2.0 ** 18
    q = q.reshape(m, -1)
    k = g.standard_normal((n, kv_heads, head_dim)).astype(np.float32)
    k[:, :, 17] = 0.0
    k, ks = {"f32": lambda x: (x, None), "f16": lambda x: (x.astype(np.float16), None),
             "fp8": lambda x: oracle.quantize_fp8_pack(x, n, kv_heads * head_dim)}.get(
                 kind, lambda x: oracle.quantize_kv(x, n, kv_heads * head_dim, 8 if kind == "q8" else 4))(k.reshape(n, -1))
    v, vs = cache(g, kind, n, kv_heads * head_dim)
    want = attention_f64(kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m)
    got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, 0)
    assert np.max(np.abs(got - want)) <= 2e-6 * max(1.0, np.max(np.abs(want)))


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("split", [0, 8])
def test_attention_rounding_of_long_heads(backend, kind, split):
    """Scores of standard deviation 4 over head_dim 256.  A weight's relative error is its score's error.  Sums of
    at most 64 products and pairwise sums of those round like a chain of about 14 terms, each step by
    2^-24 * 0.42 of the score in the root mean square: sqrt(14) * 0.42 * 2^-24 * 4 = 3.7e-7; one running sum over the
    head, or two, are at 8e-7 and more.  The sums over the keys add 2e-7."""
    m, n, heads, kv_heads, head_dim = 1, 1200, 24, 4, 256
    errors = []
    for seed in range(6):
        g = synth.rng(1700 + seed)
        q = (4.0 * g.standard_normal((m, heads * head_dim))).astype(np.float32)
        k, ks = cache(g, kind, n, kv_heads * head_dim)
        v, vs = cache(g, kind, n, kv_heads * head_dim)
        want = attention_f64(kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m)
        got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, 0, split=split)
        errors.append(np.linalg.norm(got - want) / np.linalg.norm(want))
    assert np.sqrt(np.mean(np.square(errors))) <= 1.3 * np.hypot(3.7e-7, 2e-7)


@pytest.mark.parametrize("kind", ["f32", "f16"])
def test_attention_parts_of_large_scores(backend, kind):
    """Scores near 400, exact in fp32 and in natural units (one element a query, head_dim 64): what is left is the
    rounding of differences up to 6, 6 * 2^-23, and of the weights.  A part's largest score rounded apart from its
    sums would cost 400 * 2^-25 = 1.2e-5."""
    m, n, heads, kv_heads, head_dim = 1, 640, 4, 2, 64
    g = synth.rng(1800)
    q = np.zeros((m, heads, head_dim), np.float32)
    q[:, :, 11] = 1.0
    k = g.standard_normal((n, kv_heads, head_dim)).astype(np.float32)
    k[:, :, 11] = 2.0 * np.round(8.0 * 200.0 + 12.0 * g.uniform(-1.0, 1.0, (n, kv_heads)))   # (exact in fp16)
    k = k.reshape(n, -1)
    k = k.astype(np.float16) if kind == "f16" else k
    v, _ = cache(g, kind, n, kv_heads * head_dim)
    q = q.reshape(m, -1)
    want = attention_f64(kind, q, k, v, None, None, m, n, heads, kv_heads, head_dim, n - m)
    for split in (1, 5, 40):
        got = attend(backend, kind, q, k, v, None, None, m, n, heads, kv_heads, head_dim, n - m, 0, split=split)
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert err <= 1.2e-6, (split, err)


def test_attention_more_workgroups_than_one_grid_of_wide_ones(backend):
    """2^23 workgroups of eight wavefronts are 2^32 threads, which one launch may not have: four wavefronts each."""
    heads, head_dim, n = 32, 16, 200
    m = (1 << 23) // heads + 3
    g = synth.rng(1900)
    k, _ = cache(g, "f16", n, heads * head_dim)
    v, _ = cache(g, "f16", n, heads * head_dim)
    q = torch.empty(m, heads * head_dim, device="cuda")
    q.normal_(generator=torch.Generator(device="cuda").manual_seed(7))
    out = torch.full((m, heads * head_dim), float("nan"), device="cuda")
    torch.cuda.synchronize()
    wrap = lambda t: backend.WrapBuffer(t.data_ptr(), t.numel() * t.element_size())
    run(backend, "attention", [wrap(q), backend.Upload(k), backend.Upload(v), wrap(out)],
        [m, n, heads, heads, head_dim, n, 0, 0, 1, 1], grid=(m * heads, 1, 1))
    backend.Synchronize()
    assert torch.isfinite(out).all()
    rows = [0, 1, m // 2, m - 1]
    want = expected("f16", q[rows].cpu().numpy(), k, v, None, None, len(rows), n, heads, heads, head_dim, n, 0)
    assert np.max(np.abs(out[rows].cpu().numpy() - want)) <= 2e-6 * max(1.0, np.max(np.abs(want)))


@pytest.mark.parametrize("kind", ["q8", "q4", "fp8"])
@pytest.mark.parametrize("head_dim", [64, 256, 36])
@pytest.mark.parametrize("at", [5, 200, 299])
def test_attention_infinite_scales(backend, kind, head_dim, at):
    """A key row with an infinite scale holds NaN wherever its code is 0 (what the quantizer leaves of a row with an
    infinity), and spoils the rows that see it, whatever the sign of the codes' score; a value row's makes the elements
    of its codes infinite or, for code 0, NaN, and no others.  Key 299 is the last, whose row also stands in for the
    keys past the end."""
    m, n, heads, kv_heads = 2, 300, 6, 2
    g = synth.rng(1950 + head_dim)
    q = (0.1 * g.standard_normal((m, heads * head_dim))).astype(np.float32)
    k, ks = cache(g, kind, n, kv_heads * head_dim)
    v, vs = cache(g, kind, n, kv_heads * head_dim)
    k, v = (np.asarray(x).reshape(n, -1).copy() for x in (k, v))
    k[at], v[at] = 0, 0
    for h in range(kv_heads):                      # one code other than 0 in each head
        byte = h * head_dim // (2 if kind == "q4" else 1) + 4
        k[at, byte] = 0xF1 if kind == "fp8" else 0x09 if kind == "q4" else 0x81
        v[at, byte] = k[at, byte]
    bad = ks.copy()
    bad[at] = np.inf
    last = np.arange(m) + n - m
    got = attend(backend, kind, q, k, v, bad, vs, m, n, heads, kv_heads, head_dim, n - m, 0).reshape(m, heads, head_dim)
    assert np.array_equal(np.isnan(got), np.broadcast_to((last >= at)[:, None, None], got.shape))
    bad = vs.copy()
    bad[at] = np.inf
    with np.errstate(invalid="ignore"):
        want = expected(kind, q, k, v, ks, bad, m, n, heads, kv_heads, head_dim, n - m, 0)
    for split in (0, 3):
        got = attend(backend, kind, q, k, v, ks, bad, m, n, heads, kv_heads, head_dim, n - m, 0, split=split)
        assert np.array_equal(np.isnan(got), np.isnan(want)), split
        assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]), split
        some = np.isfinite(want)
        assert np.max(np.abs(got[some] - want[some]), initial=0.0) <= 4e-6, split
