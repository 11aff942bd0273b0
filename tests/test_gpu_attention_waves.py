"""Attention with few query rows where a workgroup's part is a little over 128 keys: five wavefronts take 129 to 160 keys at
once (144 over an fp32 cache), four the 128 below, eight (or four) the 161 above, and more workgroups than CUs four.  Against the oracle's
restatements; the bounds are test_gpu_attention.py's (sums in another order, twice that after a merge of parts)."""
import numpy as np
import pytest

from tessera_amd import synth
from test_gpu_attention import KINDS, attend, cache, expected

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("head_dim", [64, 96, 128, 256])
@pytest.mark.parametrize("each", [128, 129, 144, 145, 160, 161])
def test_attention_parts_around_five_wavefronts(backend, kind, head_dim, each):
    g = synth.rng(each * 5 + head_dim + KINDS[kind])
    m, heads, kv_heads = 2, 6, 2
    for n, window, split in ((each, 0, 0), (each, 37, 0), (each * 3 - 2, 0, 3), (each * 3, 150, 3)):
        width = kv_heads * head_dim
        q = g.standard_normal((m, heads * head_dim)).astype(np.float32)
        k, ks = cache(g, kind, n, width)
        v, vs = cache(g, kind, n, width)
        want = expected(kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, window)
        got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, window, split=split)
        assert np.max(np.abs(got - want)) <= (2 if split else 1) * 2e-6 * max(1.0, np.max(np.abs(want))), (n, window, split)


@pytest.mark.parametrize("kind", ["f16", "q8"])
def test_more_workgroups_than_cus(backend, kind):
    """Just as many workgroups as the chip has CUs, and one key head's worth more."""
    g = synth.rng(77)
    n, head_dim = 130, 64
    for m in (128, 129):
        heads = kv_heads = 2
        q = g.standard_normal((m, heads * head_dim)).astype(np.float32)
        k, ks = cache(g, kind, n, kv_heads * head_dim)
        v, vs = cache(g, kind, n, kv_heads * head_dim)
        want = expected(kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, 0)
        got = attend(backend, kind, q, k, v, ks, vs, m, n, heads, kv_heads, head_dim, n - m, 0)
        assert np.max(np.abs(got - want)) <= 2e-6 * max(1.0, np.max(np.abs(want)))
