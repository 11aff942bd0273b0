"""FP8 E4M3 weights ("gemm_fp8") times 17 rows and more on the fp16 matrix instruction: the codes are exact in
fp16, an fp32 row goes in as two fp16 terms (2^-23 of every element down to 2^-28 of the row's largest).
Reference kernel src/backends/rocm/rocm_kernels_basic.cpp:1039-1064, CPU GemmFp8Ref.

Bound, in units of an output's root sum of squared products (the size it has before its products cancel): the
terms leave 2^-23 of each product, the fp32 sum of k products rounds partial sums of at most a few units k times
independently, sqrt(k) * 2^-24; (2 + sqrt(k)) * 2^-23 covers both.  Against float64."""
import numpy as np
import pytest

import oracle
from tessera_amd import synth
from util import run

pytestmark = pytest.mark.gpu
LUT = np.array([oracle.fp8_e4m3_to_float(c) for c in range(256)], np.float32)


def fp8_gemm(backend, a, codes, scales, m, n, k):
    da, dw, ds = backend.Upload(a), backend.Upload(codes), backend.Upload(scales)
    guard = np.full(m * n + 64, 7.0, np.float32)
    dc = backend.Upload(guard)
    run(backend, "gemm_fp8", [da, dw, ds, dc], [m, n, k], grid=((m * n + 255) // 256, 1, 1))
    backend.Synchronize()
    out = backend.CopyD2H(dc, dtype=np.float32)
    assert np.all(out[m * n:] == 7.0)
    return out[:m * n].reshape(m, n)


def exact(a, codes, scales, n, k):
    """The float64 result and each output's root sum of squared products."""
    a, w = a.astype(np.float64), LUT[codes].reshape(n, k).astype(np.float64) * scales.astype(np.float64)[:, None]
    return a @ w.T, np.sqrt((a * a) @ (w * w).T)


def within(got, ref, unit, k):
    return bool(np.all(np.abs(got.astype(np.float64) - ref) <= (2.0 + np.sqrt(k)) * 2.0 ** -23 * unit))


# edges of the 32/64/128-row and 128-column tiles, one stage of K and more parts of it than stages in the ring,
# odd n (scalar stores of the last launch), long rows (read twice by the conversion), a k that stays with the
# multiply-add passes
@pytest.mark.parametrize("m,n,k", [(17, 512, 1024), (31, 1, 64), (32, 129, 128), (33, 127, 192), (64, 640, 1088), (65, 1001, 2048),
                                   (127, 385, 2112), (128, 2048, 512), (129, 130, 5120), (300, 1537, 1280), (20, 200, 8256),
                                   (257, 6144, 256), (1030, 4100, 320), (40, 64, 96)])
def test_matches_float64(backend, m, n, k):
    g = synth.rng(6100 * m + n + k)
    codes, scales = synth.fp8_weights(g, n, k)
    a = synth.activations_f32(g, m, k)
    a[m // 2] *= np.float32(2.0 ** 100)      # rows keep scales of their own
    a[m - 1] *= np.float32(2.0 ** -110)
    a[0, : k // 2] *= np.float32(2.0 ** -20)
    assert within(fp8_gemm(backend, a, codes, scales, m, n, k), *exact(a, codes, scales, n, k), k)


def test_zero_and_non_finite_rows_and_weights(backend):
    g = synth.rng(6200)
    m, n, k = 40, 300, 512
    codes, scales = synth.fp8_weights(g, n, k)
    a = synth.activations_f32(g, m, k)
    a[3] = 0.0
    a[5, 100] = np.inf
    a[7, 9] = np.nan
    codes = codes.reshape(n, k).copy()
    codes[11, 4] = 0x7F
    got = fp8_gemm(backend, a, codes.reshape(-1), scales, m, n, k)
    good_cols = np.delete(np.arange(n), 11)
    assert not np.isfinite(got[[5, 7]]).any() and np.isnan(got[:, 11]).all()
    assert np.all(got[3, good_cols] == 0.0)
    rows = [0, 1, 2, 4, 6, 8, 39]
    ref, unit = exact(a[rows], codes.reshape(-1), scales, n, k)
    assert within(got[rows][:, good_cols], ref[:, good_cols], unit[:, good_cols], k)


def test_every_weight_code(backend):
    """Weight row c is code c along its whole length, one-hot activations: the product bit for bit."""
    k, m = 64, 48
    codes = np.repeat(np.arange(256, dtype=np.uint8), k)
    scales = np.ones(256, np.float32)
    a = np.zeros((m, k), np.float32)
    for r in range(m):
        a[r, r] = np.float32(1.0 + r / 64.0)
    got = fp8_gemm(backend, a, codes, scales, m, 256, k)
    finite = np.isfinite(LUT)
    want = np.array([1.0 + r / 64.0 for r in range(m)], np.float32)[:, None] * LUT[None, finite]
    assert np.array_equal(got[:, finite], want) and np.isnan(got[:, ~finite]).all()


def test_small_caller_workspace_still_runs(backend):
    """With less scratch than the matrix-core path asks for the call is carried out all the same."""
    g = synth.rng(6300)
    m, n, k = 1100, 1300, 4096                # terms of 18 MB: more than the library's own decode-sized block
    codes, scales = synth.fp8_weights(g, n, k)
    a = synth.activations_f32(g, m, k)
    block = backend.AllocateBuffer(1 << 20)
    backend.SetWorkspace(block)
    try:
        slow = fp8_gemm(backend, a, codes, scales, m, n, k)
    finally:
        backend.SetWorkspace(None)
    fast = fp8_gemm(backend, a, codes, scales, m, n, k)
    want = exact(a[:64], codes, scales, n, k)
    assert within(slow[:64], *want, k) and within(fast[:64], *want, k)


@pytest.mark.parametrize("m,n,k", [(17, 130, 1024), (64, 300, 5120)])
@pytest.mark.parametrize("binades", [10, 17, 20, 24, 28])
def test_elements_far_below_the_row_s_largest(backend, m, n, k, binades):
    """Weights that are zero on a row's largest elements: the output comes from the others alone, 2^-binades as
    large, and keeps their precision."""
    g = synth.rng(6400 + binades)
    codes, scales = synth.fp8_weights(g, n, k)
    a = synth.activations_f32(g, m, k)
    largest = np.arange(0, k, 16)
    a = np.clip(a, -4.0, 4.0)
    a[:, largest] = 4.0 * np.sign(a[:, largest] + np.float32(0.5))
    rest = np.setdiff1d(np.arange(k), largest)
    small = a[:, rest]
    a[:, rest] = np.sign(small) * np.clip(np.abs(small), 1.0, 4.0) * np.float32(2.0 ** -binades)
    codes = codes.reshape(n, k).copy()
    codes[:, largest] = 0
    codes = codes.reshape(-1)
    assert within(fp8_gemm(backend, a, codes, scales, m, n, k), *exact(a, codes, scales, n, k), k)


@pytest.mark.parametrize("steps", [2, 14, 16, 30, 32, 48])
def test_a_step_of_zeros_changes_nothing(backend, steps):
    """Sums are kept in runs of 2 and of 16 steps of K, and a run that has ended goes on to the next sum also where one more
    step is left: 64 more zeros a row have the bits of the product without them.  (300 x 6144: one part of K.)"""
    m, n, k = 300, 6144, steps * 64
    g = synth.rng(6300 + steps)
    codes, scales = synth.fp8_weights(g, n, k + 64)
    a = synth.activations_f32(g, m, k)
    short = fp8_gemm(backend, a, np.ascontiguousarray(codes.reshape(n, k + 64)[:, :k]).reshape(-1), scales, m, n, k)
    long = fp8_gemm(backend, np.concatenate([a, np.zeros((m, 64), np.float32)], 1), codes, scales, m, n, k + 64)
    assert np.array_equal(short, long)
