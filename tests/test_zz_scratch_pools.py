"""A program that records its step again and again: each recording keeps a scratch block for good.  Those of attention in
parts of its keys, whose calls do without one, must leave the blocks of "gemm_fp8" alone, which then runs other kernels.
(Named to run last: the parts' blocks are used up afterwards.)"""
import numpy as np
import pytest
import torch

from tessera_amd import KernelLaunch, synth
from test_gpu_streams import Call, home, record     # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu


def test_recorded_attention_leaves_fp8_its_scratch(backend, home):     # noqa: F811
    m, n, heads, kv_heads, head_dim = 40, 4200, 24, 4, 256
    dev = torch.device("cuda:0")
    wrap = lambda t: backend.WrapBuffer(t.data_ptr(), t.numel() * t.element_size())
    q, k, v = (torch.randn(rows, width, device=dev) for rows, width in ((m, heads * head_dim), (n, kv_heads * head_dim), (n, kv_heads * head_dim)))
    k, v, out = k.half(), v.half(), torch.empty_like(q)
    kernel = backend.LoadKernel("attention")
    launch = KernelLaunch(grid_x=m * heads, buffers=[wrap(q), wrap(k), wrap(v), wrap(out)], scalars=[m, n, heads, kv_heads, head_dim, n - m, 0, 0, 1, 1])

    def attend():
        backend.SetStream(torch.cuda.current_stream().cuda_stream)
        backend.LaunchKernel(kernel, launch)

    attend()
    torch.cuda.synchronize()
    want, graphs = out.clone(), []
    for _ in range(140):                                    # 16 MB of parts each
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            attend()
    call = Call(backend, "gemm_fp8", 300, 512, 5120, 9900)
    alone = call.alone(home)
    graph = record([call])
    for g in (graph, graphs[0], graphs[-1], graph):
        call.y.fill_(float("nan")), out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        if g is graph:
            assert np.array_equal(call.bits(), alone)
        else:                                               # with a block of its own, and without one
            assert torch.max(torch.abs(out - want)).item() <= 4e-6 * torch.max(torch.abs(want)).item()
