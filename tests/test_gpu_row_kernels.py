"""Row-wise trunk kernels at the edges of their dispatch: the sizes at which another variant, another
number of loads a thread or another loop takes over, against the oracle."""
import numpy as np
import pytest

import oracle
from tessera_amd import synth
from util import run

pytestmark = pytest.mark.gpu


# one float4 a thread up to 4096 columns, then two, four, eight up to 32768; any other length, and longer
# rows, on the scalar loop; 512 rows and more with 256 threads a row
@pytest.mark.parametrize("rows,cols", [(1, 4), (2, 252), (1, 4096), (3, 4100), (1, 8192), (2, 8196), (1, 16388), (1, 32768),
                                       (1, 32772), (3, 4097), (511, 260), (512, 1024), (513, 1028), (515, 5120), (512, 8196)])
def test_rmsnorm_edges(backend, rows, cols):
    g = synth.rng(rows * 7 + cols)
    x = g.standard_normal((rows, cols)).astype(np.float32)
    w = g.uniform(0.5, 1.5, cols).astype(np.float32)
    eps = np.float32(1e-6)
    dx, dw = backend.Upload(x), backend.Upload(w)
    dy = backend.Upload(np.full(rows * cols, np.nan, np.float32))
    run(backend, "rmsnorm", [dx, dw, dy], [rows, cols, int(eps.view(np.uint32))])
    backend.Synchronize()
    got = backend.CopyD2H(dy, dtype=np.float32).reshape(rows, cols)
    want = oracle.rmsnorm(x, w, rows, cols, float(eps))
    # the two sums of cols squares are fp32 chains in different orders: cols * 2^-24 relative at worst,
    # halved by the square root
    bound = max(2e-6, cols * 2.0 ** -25)
    assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 1e-30)) <= bound
