"""The fp16 copy of the activation rows around the lengths up to which a row is held in registers (2048, 6144, 18432):
one-hot rows bring back the fp16 weights of a column, rows with one large element keep their scale."""
import numpy as np
import pytest

import oracle
from tessera_amd import synth
from util import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [256, 2048, 2304, 6144, 6400, 18432, 18688])
def test_one_hot_rows(backend, k):
    m, n = 65, 64
    g = synth.rng(k)
    w = synth.q4k_weights(g, n, k)
    at = np.append(g.integers(0, k, m - 1), k - 1)
    a = np.zeros((m, k), np.float32)
    a[np.arange(m), at] = np.exp2(g.integers(-20, 20, m)).astype(np.float32)
    da, dw, dc = backend.Upload(a), backend.Upload(w), backend.AllocateBuffer(4 * m * n)
    run(backend, "gemm_q4k_wmma", [da, dw, dc], [m, n, k])
    backend.Synchronize()
    got = backend.CopyD2H(dc, dtype=np.float32).reshape(m, n)
    deq = oracle.dequantize_q4k(w).reshape(n, k).astype(np.float16).astype(np.float32)
    assert np.array_equal(got, deq[:, at].T * a[np.arange(m), at][:, None])
