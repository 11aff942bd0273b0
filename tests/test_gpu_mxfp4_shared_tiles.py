"""MXFP4 weights times 17 and more fp32 rows where workgroups share a tile's steps of K: row counts around the tiles
of 64, 128 and 256 rows, column counts around 256 and off the four-column stores, few and many workgroups a tile, rows
that need two and four terms in one tile and in neighbouring ones.  Against the float64 product of the split rows (bounds
of test_gpu_gemm_mxfp4_f32.py).  And the same bits wherever the tiles' pieces lie, or where there is no room for them."""
import numpy as np
import pytest
import torch

import oracle
from tessera_amd import KernelLaunch, StatusCode, StatusError, synth
from test_gpu_gemm_mxfp4_f32 import ACC_TOL, mx_gemm, split_model
from util import rms_err, same_bits

pytestmark = pytest.mark.gpu

WHOLE = [(255, 256, 2048), (384, 770, 2048), (449, 2306, 2048), (300, 16500, 2048)]
SHARED = [
    (17, 256, 2048), (64, 257, 2176), (65, 511, 2048), (128, 1023, 2048), (129, 514, 4096), (257, 300, 2304), (33, 5000, 2048),
    (100, 40, 16384), (128, 1023, 4224), (255, 256, 4096), (384, 770, 4096), (449, 2306, 4096),
]


@pytest.mark.parametrize("m,n,k", WHOLE + SHARED)
@pytest.mark.parametrize("two_terms", ["every third row", "the first 128 rows"])
def test_shared_tiles(backend, m, n, k, two_terms):
    g = synth.rng(m + n + k)
    a = g.standard_normal((m, k)).astype(np.float32)
    short = slice(None, None, 3) if two_terms == "every third row" else slice(0, 128)
    a[short] = synth.round_to_bf16(a[short])                # two terms
    w = synth.mxfp4_weights(g, n, k)
    got = mx_gemm(backend, "gemm_mxfp4_batched", a, w, m, n, k)
    deq = oracle.dequantize_mxfp4(w, n, k).astype(np.float64)
    assert rms_err(got, split_model(a, 4) @ deq.T) <= ACC_TOL
    assert np.array_equal(got, mx_gemm(backend, "gemm_mxfp4", a, w, m, n, k))    # the same bits again
    assert np.all(np.isfinite(got))


# tiles of 64, 128 and 256 rows; pieces that fit the static array, and more than it holds (60 and 98 MB)
@pytest.mark.parametrize("m,n,k", [(17, 700, 2048), (40, 5000, 5120), (100, 520, 4096), (100, 6144, 5120), (200, 2306, 4096),
                                   (300, 3000, 4096), (453, 17408, 5120)])
def test_same_bits_with_and_without_room_for_the_pieces(backend, m, n, k):
    g = synth.rng(m + n)
    dw, da, dc = backend.Upload(synth.mxfp4_weights(g, n, k)), backend.Upload(g.standard_normal((m, k)).astype(np.float32)), backend.AllocateBuffer(4 * m * n)
    kernel, launch = backend.LoadKernel("gemm_mxfp4_batched"), KernelLaunch(grid_x=1, buffers=[da, dw, dc], scalars=[m, n, k])
    nothing = np.full(m * n, np.nan, np.float32)

    def result(**kw):
        backend.CopyH2D(dc, nothing)
        backend.LaunchKernel(kernel, launch, **kw)
        backend.Synchronize()
        return backend.CopyD2H(dc, dtype=np.float32)

    need = backend.WorkspaceBytes(kernel, [m, n, k])
    terms = 4 * m * k + 2 * 256 * 8                         # at least what the rows' terms take
    assert need > terms
    want = result()
    assert np.all(np.isfinite(want)) and same_bits(result(no_alloc=True), want)
    try:
        for size in (need, need - 256, terms):              # all of it, some of it, the rows' terms alone
            ws = torch.empty(size, dtype=torch.uint8, device="cuda")
            backend.SetWorkspace(backend.WrapBuffer(ws.data_ptr(), size))
            assert same_bits(result(), want), size
        backend.SetWorkspace(backend.WrapBuffer(ws.data_ptr(), 4 * m * k))
        with pytest.raises(StatusError) as e:
            result()
        assert e.value.code == StatusCode.InvalidArgument
    finally:
        backend.Synchronize()
        backend.SetWorkspace(None)
