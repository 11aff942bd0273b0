"""The feed forward's front half with more than 64 rows, where one tile takes both products: rows and columns around
its tiles (256 x 128, 128 x 64) and rounds of them, against the library's own two products and silu_mul, bit for bit."""
import numpy as np
import pytest

from tessera_amd import synth
from test_gpu_ffn import ffn
from util import run, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(65, 40, 256), (128, 64, 512), (129, 65, 768), (255, 127, 256), (257, 4224, 256),
                                   (511, 8300, 256), (300, 16385, 512), (1025, 6600, 256)])
def test_gate_up_equals_its_products(backend, m, n, k):
    g = synth.rng(m + n)
    gate, up = synth.q4k_weights(g, n, k), synth.q4k_weights(g, n, k)
    x = synth.activations_f32(g, m, k)
    got = ffn(backend, x, gate, up, m, n, k)
    dx, dg, du = backend.Upload(x), backend.Upload(gate), backend.Upload(up)
    og, ou = backend.AllocateBuffer(4 * m * n), backend.AllocateBuffer(4 * m * n)
    run(backend, "gemm_q4k", [dx, dg, og], [m, n, k])
    run(backend, "gemm_q4k", [dx, du, ou], [m, n, k])
    run(backend, "silu_mul", [og, ou, og], [m * n])
    backend.Synchronize()
    assert same_bits(got.reshape(-1), backend.CopyD2H(og, dtype=np.float32))
