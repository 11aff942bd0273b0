"""The largest logits of long rows that workgroups share (top_k_rows: the shares' edges, ties, NaN) and the merge of
more parts of attention than a wavefront has lanes."""
import numpy as np
import pytest

from tessera_amd import synth
from util import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [24577, 32768, 32769, 8192 * 16, 8192 * 16 + 5, 8192 * 33 + 31])
@pytest.mark.parametrize("rows,top_k", [(1, 8), (3, 32), (16, 1), (17, 5)])
@pytest.mark.parametrize("kind", ["normal", "ties", "nan"])
def test_top_k_shared_rows(backend, vocab, rows, top_k, kind):
    g = synth.rng(vocab + rows)
    x = g.standard_normal((rows + 1, vocab)).astype(np.float32)
    if kind == "ties":
        x = np.round(x).astype(np.float32)
    if kind == "nan":
        x[:, ::3] = np.nan
        x[-1, 3:] = np.nan
    dx = backend.Upload(x)
    ids, vals = backend.AllocateBuffer(4 * rows * top_k), backend.AllocateBuffer(4 * rows * top_k)
    run(backend, "top_k_rows", [dx, ids, vals], [rows, vocab, top_k, 1], grid=(rows, 1, 1))
    backend.Synchronize()
    got = backend.CopyD2H(ids, dtype=np.uint32).reshape(rows, top_k)
    got_v = backend.CopyD2H(vals, dtype=np.float32).reshape(rows, top_k)
    col = np.arange(vocab)
    for r in range(rows):
        v = np.where(np.isnan(x[1 + r]), -np.inf, x[1 + r].astype(np.float64))
        order = np.lexsort((col // 256, col % 256, np.isnan(x[1 + r]), -v))[:top_k]
        assert np.array_equal(got[r], order), r
        assert np.array_equal(got_v[r], x[1 + r][order], equal_nan=True)


@pytest.mark.parametrize("split", [1, 16, 17, 63, 64, 65, 130, 1000])
@pytest.mark.parametrize("head_dim", [34, 64, 100, 256])
def test_attention_combine_parts(backend, split, head_dim):
    m, heads = 2, 3
    g = synth.rng(split + head_dim)
    acc = g.standard_normal((m * heads, split, head_dim)).astype(np.float32)
    most = (g.standard_normal((m * heads, split)) * 4).astype(np.float32)
    total = (g.random((m * heads, split)) + 0.5).astype(np.float32)
    most[:, ::5], acc[:, ::5], total[:, ::5] = -1e30, 0.0, 0.0           # empty parts
    if split == 1:
        most[:], total[:] = 0.5, 1.5
    bufs = [backend.Upload(t) for t in (acc, most, total)] + [backend.AllocateBuffer(4 * m * heads * head_dim)]
    run(backend, "attention_combine", bufs, [m, heads, head_dim, split], grid=(m * heads, 1, 1))
    backend.Synchronize()
    got = backend.CopyD2H(bufs[3], dtype=np.float32).reshape(m * heads, head_dim)
    w = np.exp(most.astype(np.float64) - most.max(1, keepdims=True))
    num = np.einsum("rs,rsd->rd", w, acc.astype(np.float64))
    den = (w * total).sum(1, keepdims=True)
    size = np.einsum("rs,rsd->rd", w, np.abs(acc).astype(np.float64)) / den
    # rounding of a weight (2^-22: expf and its argument) and of sums of no more than split / 16 + 20 terms
    assert np.all(np.abs(got - num / den) <= size * (2.0 ** -21 + (split / 16 + 20) * 2.0 ** -24))


# one, four and sixteen wavefronts a row; more rows than a launch has threads for with sixteen each
@pytest.mark.parametrize("rows,heads,head_dim,parts", [
    (1500, 3, 64, 2), (2, 4, 256, 4), (700, 4, 256, 3), (5, 2, 130, 1), (3, 5, 100, 9), (300, 1, 256, 20), (4, 6, 36, 17), (1, 2, 64, 33),
    (65537, 64, 2, 1), (65537, 64, 1, 6)])
def test_attention_combine_rows_and_parts(backend, rows, heads, head_dim, parts):
    """Against the merge in float64; weights of some parts vanish and some parts are empty (0, -1e30, 0)."""
    g = synth.rng(rows + parts)
    count = rows * heads
    acc = g.standard_normal((count, parts, head_dim)).astype(np.float32)
    most = (g.standard_normal((count, parts)) * 20).astype(np.float32)
    total = (1 + g.random((count, parts))).astype(np.float32)
    if parts > 2:
        acc[::3, 1], most[::3, 1], total[::3, 1] = 0.0, -1e30, 0.0
    bufs = [backend.Upload(x) for x in (acc, most, total)]
    out = backend.AllocateBuffer(4 * count * head_dim)
    run(backend, "attention_combine", [*bufs, out], [rows, heads, head_dim, parts], grid=(count, 1, 1))
    backend.Synchronize()
    got = backend.CopyD2H(out, dtype=np.float32).reshape(count, head_dim)
    w = np.exp(most.astype(np.float64) - most.max(1, keepdims=True))
    want = np.einsum("rp,rpd->rd", w, acc) / np.sum(w * total, axis=1, keepdims=True)
    # an exponential of a difference of up to 100 in fp32 (2^-17), the largest terms' alone: 2^-22; sums of parts terms
    assert np.max(np.abs(got - want)) <= (parts + 8) * 2.0 ** -23 * max(1.0, np.max(np.abs(want)))
