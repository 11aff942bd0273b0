"""MXFP4 weights times 17 and more fp32 rows where workgroups share a tile's steps of K: row counts around the tiles
of 64, 128 and 256 rows, column counts around 256 and off the four-column stores, few and many workgroups a tile, rows
that need two and four terms in one tile.  Against the float64 product of the split rows (bounds of
test_gpu_gemm_mxfp4_f32.py)."""
import numpy as np
import pytest

import oracle
from tessera_amd import synth
from test_gpu_gemm_mxfp4_f32 import ACC_TOL, mx_gemm, split_model
from util import rms_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (17, 256, 2048), (64, 257, 2176), (65, 511, 2048), (128, 1023, 2048), (129, 514, 4096), (255, 256, 2048),
    (257, 300, 2304), (384, 770, 2048), (449, 2306, 2048), (33, 5000, 2048), (100, 40, 16384),
])
def test_shared_tiles(backend, m, n, k):
    g = synth.rng(m + n + k)
    a = g.standard_normal((m, k)).astype(np.float32)
    a[::3] = synth.round_to_bf16(a[::3])                    # two terms
    w = synth.mxfp4_weights(g, n, k)
    got = mx_gemm(backend, "gemm_mxfp4_batched", a, w, m, n, k)
    deq = oracle.dequantize_mxfp4(w, n, k).astype(np.float64)
    rows = sorted({0, 1, 2, 15, 16, m // 2, m - 2, m - 1} & set(range(m)))
    sim = np.stack([split_model(a[r:r + 1], 4)[0] @ deq.T for r in rows])
    assert rms_err(got[rows], sim) <= ACC_TOL
    assert np.array_equal(got, mx_gemm(backend, "gemm_mxfp4", a, w, m, n, k))    # the same bits again
    assert np.all(np.isfinite(got))
