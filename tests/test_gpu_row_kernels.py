"""Row-wise trunk kernels at the edges of their dispatch: the sizes at which another variant, another
number of loads a thread or another loop takes over, against the oracle."""
import numpy as np
import pytest
import torch

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
    exact = x.astype(np.float64) / np.sqrt(np.mean(x.astype(np.float64) ** 2, axis=1, keepdims=True) + float(eps)) * w
    # float64: the sum of squares rounds once a term of a thread's chain (32 at most, cols / 256 on the scalar loop),
    # of the butterfly (6) and of the wavefronts' sums (16; 4), all terms positive, halved by the square root; then
    # the mean, the root, the reciprocal and two products
    steps = cols / 256 + 6 + 4 if cols % 4 or cols > 32768 else 32 + 6 + 16
    assert np.max(np.abs(got - exact) / np.maximum(np.abs(exact), 1e-30)) <= (steps / 2 + 5) * 2.0 ** -24
    # the oracle's sum is one chain of cols: within that of it
    want = oracle.rmsnorm(x, w, rows, cols, float(eps))
    assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 1e-30)) <= max(2e-6, cols * 2.0 ** -25)


def top_k_want(row, top_k):
    """Descending; ties to the lower share (column mod 256), inside a share to the earlier column."""
    c = np.arange(row.size)
    order = np.lexsort((c // 256, c % 256, -row.astype(np.float64)))[:top_k]
    return order.astype(np.uint32), row[order]


# a wavefront a row up to 256 and up to 512 columns, then a workgroup a row: less than a tile of 8192, one
# tile, one column more, many tiles with a remainder.  Sorted rows and rows of few different values are the
# ones whose candidates outgrow the list.
@pytest.mark.parametrize("kind", ["normal", "rising", "falling", "ties", "equal", "infinite", "nan"])
@pytest.mark.parametrize("rows,vocab,top_k", [(1, 1, 1), (5, 64, 8), (3, 256, 32), (6, 257, 3), (2, 512, 32), (2, 513, 32), (3, 1000, 1),
                                              (2, 8192, 8), (1, 8193, 32), (2, 70001, 32), (1, 131072, 8), (1, 151936, 17)])
def test_top_k_edges(backend, rows, vocab, top_k, kind):
    g = synth.rng(vocab + top_k)
    x = g.standard_normal((rows + 1, vocab)).astype(np.float32)
    if kind in ("rising", "falling"):
        x = np.sort(x, axis=1)
        x = x if kind == "rising" else x[:, ::-1].copy()
    elif kind == "ties":
        x = np.round(x * 2) / 2          # holds -0.0 and 0.0, which tie
    elif kind == "equal":
        x[:] = -1.25
    elif kind == "infinite":
        x[:, ::3] = -np.inf
        x[:, vocab // 2] = np.inf
    elif kind == "nan":
        x[:, ::5] = np.nan               # below everything
    dx = backend.Upload(x)
    di, dv = backend.Upload(np.full(rows * top_k, 0xFFFFFFFF, np.uint32)), backend.AllocateBuffer(4 * rows * top_k)
    if kind == "infinite" and np.isfinite(x[0]).sum() + 1 < top_k:
        top_k = 1
    run(backend, "top_k_rows", [dx, di, dv], [rows, vocab, top_k, 1])   # rows 1.. of the buffer
    backend.Synchronize()
    ids = backend.CopyD2H(di, dtype=np.uint32)[:rows * top_k].reshape(rows, top_k)
    vals = backend.CopyD2H(dv, dtype=np.float32)[:rows * top_k].reshape(rows, top_k)
    for r in range(rows):
        want_ids, want_vals = top_k_want(x[r + 1], top_k)
        assert np.array_equal(ids[r], want_ids), r
        assert np.array_equal(vals[r].view(np.uint32), want_vals.view(np.uint32)), r


def test_top_k_more_rows_than_one_grid(backend):
    """2^22 rows of a workgroup of 1024 are 2^32 threads, which one launch may not have: two launches."""
    rows, vocab, top_k = (1 << 22) + 5, 513, 3
    x = torch.empty(rows, vocab, device="cuda")
    x.normal_(generator=torch.Generator(device="cuda").manual_seed(5))
    ids = torch.full((rows, top_k), -1, dtype=torch.int32, device="cuda")
    vals = torch.empty(rows, top_k, device="cuda")
    torch.cuda.synchronize()
    wrap = lambda t: backend.WrapBuffer(t.data_ptr(), t.numel() * t.element_size())
    run(backend, "top_k_rows", [wrap(x), wrap(ids), wrap(vals)], [rows, vocab, top_k, 0])
    backend.Synchronize()
    assert (ids >= 0).all()
    some = list(range(4)) + list(range((1 << 22) - 6, rows))
    for r in some:
        want_ids, want_vals = top_k_want(x[r].cpu().numpy(), top_k)
        assert np.array_equal(ids[r].cpu().numpy().astype(np.uint32), want_ids), r
        assert np.array_equal(vals[r].cpu().numpy(), want_vals), r


def test_rmsnorm_more_rows_than_one_grid_of_wide_workgroups(backend):
    """2^22 rows too long for a workgroup of 256 to hold, in place: 138 GB, on the loop that reads a row twice."""
    rows, cols = (1 << 22) + 1, 8196
    if torch.cuda.mem_get_info()[0] < 150 << 30:
        pytest.skip("needs 150 GB")
    x = torch.empty(rows * cols, device="cuda")
    x.normal_(generator=torch.Generator(device="cuda").manual_seed(6))
    w = torch.ones(cols, device="cuda")
    some = [0, 1 << 21, rows - 1]
    before = {r: x[r * cols:(r + 1) * cols].cpu().numpy() for r in some}
    torch.cuda.synchronize()
    wrap = lambda t: backend.WrapBuffer(t.data_ptr(), t.numel() * t.element_size())
    eps = np.float32(1e-6)
    run(backend, "rmsnorm", [wrap(x), wrap(w), wrap(x)], [rows, cols, int(eps.view(np.uint32))])
    backend.Synchronize()
    for r in some:
        want = oracle.rmsnorm(before[r][None], np.ones(cols, np.float32), 1, cols, float(eps))[0]
        assert np.max(np.abs(x[r * cols:(r + 1) * cols].cpu().numpy() - want)) <= 2e-5, r
    del x
    torch.cuda.empty_cache()
