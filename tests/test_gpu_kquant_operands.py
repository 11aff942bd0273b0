"""Q5_K and Q6_K from 17 rows, whose two operands become fp16 in one launch or two: rows of each length a thread's registers are
laid out for, row and column counts on both sides of the lines between these, and counts of blocks that leave the last
workgroup's share short.  One element a row other than zero gives the products of an fp16 activation and an fp16 weight,
which fp32 holds, times the row's power of two."""
import numpy as np
import pytest

import oracle
from tessera_amd import synth
from util import run

pytestmark = pytest.mark.gpu

DECODE = {"q5k": (synth.q5k_weights, oracle.dequantize_q5k), "q6k": (synth.q6k_weights, oracle.dequantize_q6k)}


@pytest.mark.parametrize("kind", list(DECODE))
@pytest.mark.parametrize("k", [256, 2048, 2304, 6144, 6400, 8192, 8448, 18432, 18688])
@pytest.mark.parametrize("m,n", [(17, 33), (17, 409), (41, 7), (512, 9), (513, 9)])
def test_one_element_a_row_gives_the_weights(backend, kind, k, m, n):
    g = synth.rng(k + m)
    w = DECODE[kind][0](g, n, k)
    a = np.zeros((m, k), np.float32)
    at = g.integers(0, k, m)
    at[:3] = 0, k - 1, k // 2
    x = (g.standard_normal(m) * np.exp2(g.integers(-20, 20, m))).astype(np.float32)
    a[np.arange(m), at] = x
    c = backend.AllocateBuffer(4 * m * n)
    run(backend, f"gemm_{kind}_batched", [backend.Upload(a), backend.Upload(w), c], [m, n, k])
    backend.Synchronize()
    got = backend.CopyD2H(c, dtype=np.float32).reshape(m, n)
    scale = np.exp2(np.floor(np.log2(np.abs(x))) - 10.0)
    x16 = ((x / scale).astype(np.float16).astype(np.float64) * scale)[:, None]
    deq = DECODE[kind][1](w).reshape(n, k)[:, at].T
    want = x16 * deq.astype(np.float16).astype(np.float64)
    # Q5_K's decode rounds a multiply-add once, the oracle a product and a difference: one fp16 unit in the last place apart
    ulp = 0.0 if kind == "q6k" else np.abs(x16) * np.maximum(np.abs(deq) * 2.0 ** -10, 2.0 ** -24)
    assert np.all(np.abs(got - want) <= ulp)
