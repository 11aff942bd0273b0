"""fp32 rows as E4M3 terms, many rows: row lengths around the thread counts that hold a row and past them, values down to the
terms' subnormal grid, zero rows, a row's largest value just below a power of two, and elements that are not finite.
Against the float64 product of the split rows, row by row
(bound of test_gpu_gemm_mxfp4_f32.py)."""
import numpy as np
import pytest

import oracle
from tessera_amd import KernelLaunch, synth
from test_gpu_gemm_mxfp4_f32 import ACC_TOL, ACC_TOL_OUTLIERS, split_model
from util import rms_err

pytestmark = pytest.mark.gpu


# K: a row of 256, 512 and 1024 threads, the last that fits each and the first past it; and one that no workgroup holds
@pytest.mark.parametrize("m,k", [(65, 1024), (65, 4096), (67, 4224), (65, 8192), (65, 8320), (65, 16384), (65, 16512), (65, 32768), (65, 32896),
                                 (64, 4096), (17, 3968)])
def test_many_rows_as_terms(backend, m, k):
    n = 40
    g = synth.rng(m + k)
    scale = np.where(g.random((m, k)) < 0.25, np.exp2(g.integers(-24, 1, (m, k))), 1.0)    # N(0, 1) rows with small values among them
    a = (g.standard_normal((m, k)) * scale).astype(np.float32)
    a[3] = 0
    # largest values just below a power of two and on one, some twenty times the others as the bound for outliers has it (the
    # matrix instruction's sums lose what lies far below its largest product)
    a[5, 7] = np.nextafter(np.float32(16), np.float32(0))
    a[6] = -a[5]
    a[9, k - 1] = 16
    w = synth.mxfp4_weights(g, n, k)
    bad = {1: np.inf, 4: np.nan, m - 1: -np.inf}
    for row, x in bad.items():
        a[row, (row * 131) % k] = x
    c = backend.AllocateBuffer(4 * m * n)
    backend.LaunchKernel(backend.LoadKernel("gemm_mxfp4_batched"),
                         KernelLaunch(grid_x=1, buffers=[backend.Upload(a), backend.Upload(w), c], scalars=[m, n, k]))
    backend.Synchronize()
    got = backend.CopyD2H(c, dtype=np.float32).reshape(m, n)
    fine = np.array([row not in bad for row in range(m)])
    assert np.all(np.isnan(got[~fine])) and np.all(got[3] == 0)
    want = split_model(np.where(np.isfinite(a), a, 0), 4) @ oracle.dequantize_mxfp4(w, n, k).astype(np.float64).T
    for row in np.flatnonzero(fine):
        assert rms_err(got[row], want[row]) <= (ACC_TOL_OUTLIERS if row in (5, 6, 9) else ACC_TOL), row
