"""The calls whose parts lie in a stream's scratch block, attention over parts of its keys and top_k_rows over shared rows, on
several streams at once, recorded beside eager ones, through the entry point that allocates nothing, with a caller's
workspace set, and without a block.  And MXFP4 with shared tiles, whose pieces lie in the workspace, recorded."""
import numpy as np
import pytest
import torch

from tessera_amd import KernelLaunch, synth
from test_gpu_streams import Call, home, record     # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu


class Parts(Call):
    """Call with its buffers made here: "attention" (fp16 or int8 cache) or "top_k_rows"; m rows, n keys or columns."""

    def __init__(self, backend, kind, m, n, seed):
        dev = torch.device("cuda:0")
        g = torch.Generator(device="cuda").manual_seed(seed)
        randn = lambda *s: torch.randn(*s, device=dev, generator=g)
        wrap = lambda t: backend.WrapBuffer(t.data_ptr(), t.numel() * t.element_size())
        self.backend, self.m, self.n, self.k = backend, m, n, kind
        if kind == "top_k_rows":
            self.held, self.ids, self.y = [randn(m, n)], torch.zeros(m, 7, dtype=torch.int32, device=dev), torch.empty(m * 7, device=dev)
            buffers, scalars = [*self.held, self.ids, self.y], [m, n, 7, 0]
        else:
            heads, kv_heads, d = 24, 4, 256
            q, k, v = randn(m, heads * d), randn(n, kv_heads * d), randn(n, kv_heads * d)
            self.y = torch.empty(m * heads * d, device=dev)
            if kind == "attention":
                self.held, tail = [q, k.half(), v.half()], [0, 1, 1]
            else:
                codes = [(x * 40).round().clamp(-127, 127).to(torch.int8) for x in (k, v)]
                self.held, tail = [q, *codes, *((torch.rand(n, device=dev, generator=g) + 0.5) / 40 for _ in range(2))], [0, 0]
            buffers, scalars = [*self.held, self.y], [m, n, heads, kv_heads, d, n - m, 0, *tail]
        self.kernel = backend.LoadKernel(kind)
        self.launch = KernelLaunch(grid_x=m, buffers=[wrap(t) for t in buffers], scalars=scalars)

    def bits(self):
        own = super().bits()
        return np.concatenate([own, self.ids.cpu().numpy().view(np.uint32).ravel()]) if self.k == "top_k_rows" else own


CALLS = [("attention", 33, 2100), ("attention_q8", 40, 3000), ("top_k_rows", 1, 131072), ("top_k_rows", 16, 40000)]


@pytest.mark.parametrize("spec", CALLS)
def test_two_streams_at_once(backend, home, spec):      # noqa: F811
    one, two = Parts(backend, *spec, 1), Parts(backend, *spec, 2)
    want = one.alone(home), two.alone(home)
    assert not np.array_equal(*want)
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        one.y.fill_(float("nan")), two.y.fill_(float("nan"))
        torch.cuda.synchronize()
        for _ in range(40):
            one.go(s)
            two.go(t)
        torch.cuda.synchronize()
        assert np.array_equal(one.bits(), want[0]) and np.array_equal(two.bits(), want[1])


def test_recorded_calls_beside_eager_ones(backend, home):       # noqa: F811
    first, second, eager = ([Parts(backend, *s, seed + i) for i, s in enumerate(CALLS)] for seed in (10, 20, 30))
    want = [[c.alone(home) for c in group] for group in (first, second, eager)]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    graphs = record(first, side), record(second, side)
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        for c in (*first, *second, *eager):
            c.y.fill_(float("nan"))
        torch.cuda.synchronize()
        for _ in range(10):
            with torch.cuda.stream(s):
                graphs[0].replay()
            with torch.cuda.stream(t):
                graphs[1].replay()
            for c in eager:
                c.go(side)
        torch.cuda.synchronize()
        for group, bits in zip((first, second, eager), want):
            for c, b in zip(group, bits):
                assert np.array_equal(c.bits(), b), (c.k, c.m, c.n)


@pytest.mark.parametrize("spec", CALLS)
def test_same_kernels_whatever_ran_before(backend, home, spec):     # noqa: F811
    call = Parts(backend, *spec, 40)
    assert backend.WorkspaceBytes(call.kernel, call.launch.scalars) == 0
    graph = record([call])
    call.y.fill_(float("nan"))
    graph.replay()
    torch.cuda.synchronize()
    recorded = call.bits()
    eager = call.alone(home)
    assert np.isfinite(eager[:call.y.numel()].view(np.float32)).all() and np.array_equal(recorded, eager)
    small = torch.empty(256, dtype=torch.uint8, device="cuda")
    backend.SetWorkspace(backend.WrapBuffer(small.data_ptr(), 256))
    assert np.array_equal(call.alone(home), eager)
    backend.SetWorkspace(None)
    call.y.fill_(float("nan"))
    call.go(home, no_alloc=True)
    torch.cuda.synchronize()
    assert np.array_equal(call.bits(), eager)
    # without a block (the per-thread stream): the same candidates, the same attention to fp32 rounding
    call.y.fill_(float("nan"))
    torch.cuda.synchronize()
    backend.SetStream(2)
    backend.LaunchKernel(call.kernel, call.launch)
    torch.cuda.synchronize()
    plain = call.bits()
    if spec[0] == "top_k_rows":
        assert np.array_equal(plain, eager)
    else:
        plain, got = (b.view(np.float32).astype(np.float64) for b in (plain, eager))
        assert np.linalg.norm(plain - got) <= 1e-6 * np.linalg.norm(plain)


def test_recorded_mxfp4_with_shared_tiles(backend, home):       # noqa: F811
    """Recorded after one eager call and replayed between eager calls of another size, in order: they share the workspace."""
    dev = torch.device("cuda:0")
    g = synth.rng(50)
    wrap = lambda t: backend.WrapBuffer(t.data_ptr(), t.numel() * t.element_size())

    class Mxfp4(Call):
        def __init__(self, m, n, k):
            self.backend, self.kernel = backend, backend.LoadKernel("gemm_mxfp4_batched")
            self.held = [torch.from_numpy(x).to(dev) for x in (synth.activations_f32(g, m, k), synth.mxfp4_weights(g, n, k))]
            self.y = torch.empty(m * n, device=dev)
            self.launch = KernelLaunch(grid_x=1, buffers=[*map(wrap, self.held), wrap(self.y)], scalars=[m, n, k])

    recorded, other = Mxfp4(100, 1030, 4096), Mxfp4(300, 520, 4352)
    want = recorded.alone(home), other.alone(home)
    graph = record([recorded])
    for _ in range(4):
        recorded.y.fill_(float("nan")), other.y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        other.go(home)
        torch.cuda.synchronize()
        assert np.array_equal(recorded.bits(), want[0]) and np.array_equal(other.bits(), want[1])
