"""Calls on several streams at once, and recorded calls beside eager ones, for the ids that hand intermediate
results from one kernel to the next without a caller's scratch: "gemm_fp8" from 17 rows, Q5_K and Q6_K with a
few rows.  Every result must have the bits of the call made alone, and the same whatever ran before it."""
import threading

import numpy as np
import pytest
import torch

from tessera_amd import KernelLaunch, synth

pytestmark = pytest.mark.gpu

# (id, rows, n, k): K split into parts in each; FP8 with 1000 rows in one go, Q6_K in two passes of rows
CALLS = [("gemm_fp8", 17, 1030, 2048), ("gemm_fp8", 300, 512, 5120), ("gemm_q6k_batched", 5, 2050, 4096),
         ("gemm_q6k_batched", 16, 1030, 8704), ("gemm_q5k_batched", 8, 1026, 5120)]


class Call:
    """One launch with its own buffers."""

    def __init__(self, backend, name, m, n, k, seed):
        dev = torch.device("cuda:0")
        g = synth.rng(seed)
        self.backend, self.kernel, self.m, self.n, self.k = backend, backend.LoadKernel(name), m, n, k
        to_dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
        if name == "gemm_fp8":
            self.w = [to_dev(x) for x in synth.fp8_weights(g, n, k)]
        else:
            self.w = [to_dev({"q5k": synth.q5k_weights, "q6k": synth.q6k_weights}[name.split("_")[1]](g, n, k))]
        self.x = to_dev(synth.activations_f32(g, m, k))
        self.y = torch.empty(m * n, device=dev)
        wrap = lambda t: backend.WrapBuffer(t.data_ptr(), t.numel() * t.element_size())
        self.launch = KernelLaunch(grid_x=(m * n + 255) // 256, buffers=[wrap(self.x), *map(wrap, self.w), wrap(self.y)], scalars=[m, n, k])

    def go(self, stream, no_alloc=False):
        self.backend.SetStream(stream.cuda_stream)
        self.backend.LaunchKernel(self.kernel, self.launch, no_alloc=no_alloc)

    def bits(self):
        return self.y.cpu().numpy().view(np.uint32).copy()

    def alone(self, stream):
        self.y.fill_(float("nan"))
        torch.cuda.synchronize()
        self.go(stream)
        torch.cuda.synchronize()
        return self.bits()


@pytest.fixture
def home(backend):
    cur = torch.cuda.current_stream()
    yield cur
    torch.cuda.synchronize()
    backend.SetWorkspace(None)
    backend.SetStream(cur.cuda_stream)


@pytest.mark.parametrize("spec", CALLS)
def test_two_streams_at_once(backend, home, spec):
    one, two = Call(backend, *spec, 9000), Call(backend, *spec, 9001)
    want = one.alone(home), two.alone(home)
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    for _ in range(3):
        one.y.fill_(float("nan")), two.y.fill_(float("nan"))
        torch.cuda.synchronize()
        for _ in range(40):
            one.go(s)
            two.go(t)
        torch.cuda.synchronize()
        assert np.array_equal(one.bits(), want[0]) and np.array_equal(two.bits(), want[1])


def record(calls, stream=None):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for c in calls:
            c.go(torch.cuda.current_stream())
    return graph


def test_recorded_calls_beside_eager_ones(backend, home):
    """Two graphs from the same capture stream replayed on two streams, eager calls on a third and on the capture
    stream itself; the graphs replay several times with the eager work between."""
    specs = CALLS[1:4]
    first, second, eager = ([Call(backend, *s, seed + i) for i, s in enumerate(specs)] for seed in (9100, 9200, 9300))
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
                assert np.array_equal(c.bits(), b), (c.m, c.n, c.k)


def test_branches_of_one_capture(backend, home):
    """Two streams of the same capture run side by side in the graph."""
    one, two = Call(backend, *CALLS[1], 9400), Call(backend, *CALLS[1], 9401)
    want = one.alone(home), two.alone(home)
    fork = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        main = torch.cuda.current_stream()
        fork.wait_stream(main)
        one.go(main)
        with torch.cuda.stream(fork):
            two.go(fork)
        main.wait_stream(fork)
    for _ in range(4):
        one.y.fill_(float("nan")), two.y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(one.bits(), want[0]) and np.array_equal(two.bits(), want[1])


def test_two_threads_on_one_stream(backend, home):
    """A call's kernels stay together: two threads' calls on one stream follow one another."""
    one, two = Call(backend, *CALLS[1], 9500), Call(backend, *CALLS[1], 9501)
    want = one.alone(home), two.alone(home)
    s = torch.cuda.Stream()
    backend.SetStream(s.cuda_stream)
    failed = []

    def repeat(call):
        try:
            for _ in range(50):
                backend.LaunchKernel(call.kernel, call.launch)
        except Exception as e:        # noqa: BLE001 (reported by the test's thread)
            failed.append(e)

    threads = [threading.Thread(target=repeat, args=(c,)) for c in (one, two)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed
    assert np.array_equal(one.bits(), want[0]) and np.array_equal(two.bits(), want[1])


# terms of 18 and of 181 MB (several goes and a rest), and calls that need little
@pytest.mark.parametrize("spec", [("gemm_fp8", 1100, 200, 4096), ("gemm_fp8", 2600, 130, 17408), CALLS[0], CALLS[2], CALLS[3]])
def test_same_kernels_whatever_ran_before(backend, home, spec):
    """No workspace is asked for, none set is too small, and a call recorded before any eager call of its size
    runs what the eager call runs: the same bits recorded, eagerly, with a caller's workspace, and through the
    entry point that allocates nothing."""
    call = Call(backend, *spec, 9600)
    assert backend.WorkspaceBytes(call.kernel, call.launch.scalars) == 0
    graph = record([call])
    call.y.fill_(float("nan"))
    graph.replay()
    torch.cuda.synchronize()
    recorded = call.bits()
    eager = call.alone(home)
    assert np.isfinite(eager.view(np.float32)).all()
    assert np.array_equal(recorded, eager)
    small = torch.empty(256, dtype=torch.uint8, device="cuda")
    backend.SetWorkspace(backend.WrapBuffer(small.data_ptr(), 256))
    assert np.array_equal(call.alone(home), eager)
    backend.SetWorkspace(None)
    call.y.fill_(float("nan"))
    call.go(home, no_alloc=True)
    torch.cuda.synchronize()
    still = call.bits()
    if spec[1] < 2600:                           # (32 MB of static scratch: other goes)
        assert np.array_equal(still, eager)
    # and right: sums in the order of the kernels without scratch (the per-thread stream's), to fp32 rounding
    call.y.fill_(float("nan"))
    torch.cuda.synchronize()
    backend.SetStream(2)
    backend.LaunchKernel(call.kernel, call.launch)
    torch.cuda.synchronize()
    plain, got, still = (b.view(np.float32).astype(np.float64) for b in (call.bits(), eager, still))
    assert max(np.linalg.norm(plain - got), np.linalg.norm(plain - still)) <= 1e-6 * np.linalg.norm(plain)
