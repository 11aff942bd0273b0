"""Q4_K, Q5_K and Q6_K products on the tensor tile where workgroups share a tile's super-blocks: row and column counts around the
128 x 128 tiles and the 32 x 32 matrix tiles, super-blocks dealt out in pieces of two and of many, tiles with one owner
beside shared ones.  Against the float64 product of the two fp16 operands; and the same bits wherever the pieces lie or find
no room: through the entry point that allocates nothing, with a caller's workspace, on each thread's own stream, and recorded."""
import numpy as np
import pytest
import torch

import oracle
from tessera_amd import KernelLaunch, synth
from test_gpu_gemm_q4k import ACC_TOL, f16_operands_product
from util import rms_err, run, same_bits

pytestmark = pytest.mark.gpu

WEIGHTS = {"q4k": synth.q4k_weights, "q5k": synth.q5k_weights, "q6k": synth.q6k_weights}
NAMES = {"q4k": "gemm_q4k_wmma", "q5k": "gemm_q5k_batched", "q6k": "gemm_q6k_batched"}
# rows, columns, K; all shared with 256 CUs (tests/test_launch_rules.py)
SHARED = [(64, 40, 2048), (65, 127, 2048), (127, 129, 2304), (129, 257, 2048), (257, 384, 3072), (300, 1030, 5120), (100, 33, 17408)]
# Q5_K's decode rounds a multiply-add once, the oracle a product and a difference: where the two lie on either side of an fp16
# midpoint a weight differs by a unit in the last place, which moves a result by up to 5 * 2^-11 * 2 rms(w) against an rms of
# sqrt(k) rms(w): 7e-5 at K = 5120 (1.1e-4 at 2048), and hardly more than one such weight meets a large activation.
TOL = {"q4k": ACC_TOL, "q5k": ACC_TOL + 2 * 1.1e-4, "q6k": ACC_TOL}
SHARED_FEW = {"q4k": [(17, 256, 2560), (32, 130, 5120), (33, 130, 2304), (63, 700, 5120)], "q5k": [(17, 256, 2048), (33, 130, 2304)],
              "q6k": [(17, 256, 2048), (33, 130, 2304)]}


def product(a, kind, w, m, n, k):
    if kind == "q4k":
        return f16_operands_product(a, w, m, n, k)
    deq = (oracle.dequantize_q5k if kind == "q5k" else oracle.dequantize_q6k)(w).reshape(n, k)
    amax = np.max(np.abs(a), axis=1)
    s = np.exp2(np.floor(np.log2(amax)) - 10.0).astype(np.float32)
    a16 = (a / s[:, None]).astype(np.float16).astype(np.float64) * s[:, None].astype(np.float64)
    return a16 @ deq.astype(np.float16).astype(np.float64).T


class Product:
    def __init__(self, backend, kind, m, n, k, seed=1):
        g = synth.rng(seed + m + n + k)
        self.backend, self.shape, self.kind = backend, (m, n), kind
        self.w, self.a = WEIGHTS[kind](g, n, k), g.standard_normal((m, k)).astype(np.float32)
        self.c = backend.AllocateBuffer(4 * m * n)
        self.kernel, self.scalars = backend.LoadKernel(NAMES[kind]), [m, n, k]
        self.launch = KernelLaunch(grid_x=1, buffers=[backend.Upload(self.a), backend.Upload(self.w), self.c], scalars=self.scalars)

    def clear(self):
        self.backend.CopyH2D(self.c, np.full(self.shape, np.nan, np.float32))

    def bits(self):
        self.backend.Synchronize()
        return self.backend.CopyD2H(self.c, dtype=np.float32).reshape(self.shape)

    def result(self, **kw):
        self.clear()
        self.backend.LaunchKernel(self.kernel, self.launch, **kw)
        return self.bits()


@pytest.mark.parametrize("kind,m,n,k", [(kind, *s) for kind in WEIGHTS for s in SHARED] + [(kind, *s) for kind in WEIGHTS for s in SHARED_FEW[kind]])
def test_shared_tiles(backend, kind, m, n, k):
    p = Product(backend, kind, m, n, k)
    got = p.result()
    assert rms_err(got, product(p.a, kind, p.w, m, n, k)) <= TOL[kind]
    assert same_bits(p.result(), got) and same_bits(p.result(no_alloc=True), got)


# (the pieces of the last of each kind do not fit the static array behind the operands)
@pytest.mark.parametrize("kind,m,n,k", [("q4k", 300, 1030, 5120), ("q4k", 1000, 2040, 5120), ("q6k", 100, 1030, 5120), ("q6k", 300, 1400, 5120)])
def test_same_bits_wherever_there_is_scratch(backend, kind, m, n, k):
    p = Product(backend, kind, m, n, k)
    want = p.result()
    assert np.all(np.isfinite(want)) and same_bits(p.result(no_alloc=True), want)
    need = backend.WorkspaceBytes(p.kernel, p.scalars)
    operands = 2 * m * k + 4 * (m + 256) + (0 if kind == "q4k" else 2 * n * k)
    assert need == operands if kind == "q4k" else need > operands
    room = need + (64 << 20)                                # more than any plan's pieces
    ws = torch.empty(room, dtype=torch.uint8, device="cuda")
    try:
        for size in (operands, operands + (1 << 20), need, room):         # the pieces in a block of the stream's, twice; in the workspace
            backend.SetWorkspace(backend.WrapBuffer(ws.data_ptr(), size))
            assert same_bits(p.result(), want), size
    finally:
        backend.SetWorkspace(None)


@pytest.mark.parametrize("kind,m,n,k", [("q4k", 300, 1030, 5120), ("q5k", 100, 1030, 5120), ("q6k", 100, 1030, 5120)])
def test_same_bits_on_each_threads_own_stream(backend, kind, m, n, k):
    """hipStreamPerThread has no block: with a caller's workspace of just the operands there is no room anywhere."""
    p = Product(backend, kind, m, n, k)
    want = p.result()
    operands = 2 * m * k + 4 * (m + 256) + (0 if kind == "q4k" else 2 * n * k)
    ws = torch.empty(operands, dtype=torch.uint8, device="cuda")
    try:
        backend.SetStream(2)
        assert same_bits(p.result(), want)
        backend.SetWorkspace(backend.WrapBuffer(ws.data_ptr(), operands))
        assert same_bits(p.result(), want)
    finally:
        backend.SetWorkspace(None)
        backend.SetStream(0)


def test_feed_forward_keeps_its_products_apart(backend):
    """64 rows: gate and up as two products in one workspace, the pieces behind the up product's result."""
    m, n, k = 64, 1030, 5120
    g = synth.rng(31)
    gate, up, x = synth.q4k_weights(g, n, k), synth.q4k_weights(g, n, k), g.standard_normal((m, k)).astype(np.float32)
    bufs = [backend.Upload(x), backend.Upload(gate), backend.Upload(up), backend.AllocateBuffer(4 * m * n)]
    kernel = backend.LoadKernel("ffn_gate_up_silu_q4k")
    launch = KernelLaunch(grid_x=1, buffers=bufs, scalars=[m, n, k])

    def result(**kw):
        backend.CopyH2D(bufs[3], np.full((m, n), np.nan, np.float32))
        backend.LaunchKernel(kernel, launch, **kw)
        backend.Synchronize()
        return backend.CopyD2H(bufs[3], dtype=np.float32).reshape(m, n)
    products = [backend.AllocateBuffer(4 * m * n) for _ in range(2)]
    for weights, out in zip(bufs[1:3], products):
        run(backend, "gemm_q4k_wmma", [bufs[0], weights, out], [m, n, k])
    run(backend, "silu_mul", [*products, bufs[3]], [m * n])
    backend.Synchronize()
    want = backend.CopyD2H(bufs[3], dtype=np.float32).reshape(m, n)
    assert np.all(np.isfinite(want)) and same_bits(result(), want)
    need = backend.WorkspaceBytes(kernel, [m, n, k])
    ws = torch.empty(need + (64 << 20), dtype=torch.uint8, device="cuda")
    try:
        for size in (need, need + (64 << 20)):
            backend.SetWorkspace(backend.WrapBuffer(ws.data_ptr(), size))
            assert same_bits(result(), want), size
    finally:
        backend.SetWorkspace(None)
    assert same_bits(result(no_alloc=True), want)


@pytest.mark.parametrize("tight", [False, True])
def test_recorded(backend, tight):
    """Two products recorded together, replayed with eager work of other sizes between the replays; with the library's workspace
    and with a caller's that holds no more than the operands."""
    calls = [Product(backend, "q4k", 300, 1030, 5120), Product(backend, "q6k", 100, 1030, 5120)]
    other = Product(backend, "q4k", 129, 257, 2048, 9)
    want, want_other = [p.result() for p in calls], other.result()
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    ws = torch.empty(2 * 100 * 5120 + 4 * 356 + 2 * 1030 * 5120, dtype=torch.uint8, device="cuda")     # the second product's
    try:
        if tight:
            backend.SetWorkspace(backend.WrapBuffer(ws.data_ptr(), ws.numel()))
        with torch.cuda.graph(graph, stream=stream):
            backend.SetStream(torch.cuda.current_stream().cuda_stream)
            for p in calls:
                backend.LaunchKernel(p.kernel, p.launch)
        backend.SetStream(torch.cuda.current_stream().cuda_stream)
        for _ in range(3):
            for p in calls:
                p.clear()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert all(same_bits(p.bits(), w) for p, w in zip(calls, want))
            assert same_bits(other.result(), want_other)
    finally:
        backend.SetWorkspace(None)
        backend.SetStream(0)
