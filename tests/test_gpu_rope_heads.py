"""Rotary embedding where a thread takes several heads (many rows): the same bits as the same rows a few at a time, heads
around eight, a rotated part shorter than the head, the multimodal form."""
import numpy as np
import pytest

from tessera_amd import synth
from util import run, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads", [1, 7, 8, 9, 24])
@pytest.mark.parametrize("head_dim,rope_dim", [(64, 64), (256, 64), (96, 96)])
@pytest.mark.parametrize("multimodal", [False, True])
def test_rope_heads_share(backend, heads, head_dim, rope_dim, multimodal):
    g = synth.rng(heads + head_dim)
    rows = 65536 // (heads * rope_dim // 2) + 3
    few = max(1, 4096 // (heads * rope_dim // 2))
    x = g.standard_normal((rows, heads, head_dim)).astype(np.float32)
    theta = int(np.float32(1e6).view(np.uint32))
    pos = g.integers(0, 5000, (rows, 3)).astype(np.uint64)

    def rotate(part, first):
        d = backend.Upload(part)
        if multimodal:
            run(backend, "mrope", [d, backend.Upload(pos[first:first + len(part)])], [len(part), heads, head_dim, rope_dim, theta, 11, 10, 9])
        else:
            run(backend, "rope", [d], [len(part), heads, head_dim, rope_dim, 77 + first, theta])
        backend.Synchronize()
        return backend.CopyD2H(d, dtype=np.float32).reshape(part.shape)

    whole = rotate(x, 0)
    for first in (0, few, rows - few):
        assert same_bits(whole[first:first + few], rotate(np.ascontiguousarray(x[first:first + few]), first))
    assert same_bits(whole[..., rope_dim:], x[..., rope_dim:])
