"""W8A16 for few rows of A, for unaligned operands, and with K split over
workgroups.

Against the float64 oracle on the fp16 activations.  Products of f16 and int8
are exact in f32 and every sum is f32, so an element is within
(K + 16) * 2^-24 * sum_k |a_k b_k| of the exact result (K additions in any
order, the scale's rounding, the partial sums'), far inside the bar used
here: 1e-5 of max|ref|, as for the tiled kernel's 1e-4.
"""
from __future__ import annotations

import json

import pytest
import torch

import neso_amd
from neso_amd import _lib
from oracle import qmatmul as Q

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(m, n, k, seed, lda=None, ldb=None):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(m, lda or k, generator=g).half()
    b = torch.randint(-128, 128, (k, ldb or n), generator=g, dtype=torch.int8)
    s = (torch.rand(n, generator=g) * 0.1 + 0.001).half()
    return a, b, s


def _ref(a, b, s, k, n):
    ref = Q.w8a16_matmul(a[:, :k].double().numpy(), b[:, :n].double().numpy())
    return ref if s is None else ref * s.double().numpy()


# Row tiles of 16, 32 and 64; strips of 128 columns with 8-column tails; K
# below one 32-row step, not a multiple of it, shorter than a step per wave,
# and split over workgroups (K = 4096 at N <= 4096) or not (N = 40000).
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 8, 8), (3, 136, 40), (16, 128, 256), (17, 120, 520), (8, 4096, 4096),
                                   (32, 1000, 1048), (33, 2056, 2048), (64, 264, 4104), (5, 40000, 264),
                                   (64, 4096, 11008)])
def test_matches_oracle(gpu, m, n, k, scaled):
    a, b, s = _inputs(m, n, k, m + n + k)
    c = torch.full((m, n), float("nan"), device=DEV)
    if scaled:
        neso_amd.w8a16_scaled_matmul(a.to(DEV), b.to(DEV), c, s.to(DEV), k, k, n, n, M=m, N=n)
    else:
        neso_amd.w8a16_matmul(a.to(DEV), b.to(DEV), c, k, k, n, n, M=m, N=n)
    assert Q.rel_err(c.cpu().numpy(), _ref(a, b, s if scaled else None, k, n)) < 1e-5


def test_strides_and_nonfinite_neighbours(gpu):
    """Padded rows of A, B and C: the padding of A (NaN) is not read into
    the result and the padding of C keeps its contents."""
    m, n, k = 9, 200, 296
    a, b, s = _inputs(m, n, k, 5, lda=k + 24, ldb=n + 56)
    a[:, k:] = float("nan")
    c = torch.full((m, n + 7), 5.0, device=DEV)
    neso_amd.w8a16_scaled_matmul(a.to(DEV), b.to(DEV), c, s.to(DEV), k, k + 24, n + 56, n + 7, M=m, N=n)
    c = c.cpu()
    assert Q.rel_err(c[:, :n].numpy(), _ref(a, b, s, k, n)) < 1e-5
    assert torch.all(c[:, n:] == 5.0)


def test_workspace_or_not(gpu):
    """The same call through the C ABI with the workspace it asks for, with
    one byte less, and without one: the split runs only with the whole
    workspace (two launches), and all results agree with the oracle."""
    lib = _lib.load()
    m, n, k = 8, 1024, 4096
    a, b, s = _inputs(m, n, k, 11)
    ad, bd, sd = a.to(DEV), b.to(DEV), s.to(DEV)
    ref = _ref(a, b, s, k, n)
    need = lib.neso_w8a16_workspace_bytes(ad.data_ptr(), bd.data_ptr(), k, k, n, m, n)
    assert need > 0 and need % (4 * m * n) == 0
    ws = torch.full((need // 4,), float("nan"), device=DEV)
    for ptr, size, launches in ((ws.data_ptr(), need, 2), (ws.data_ptr(), need - 1, 1), (None, need, 1),
                                (None, 0, 1)):
        c = torch.full((m, n), float("nan"), device=DEV)
        args = [ad.data_ptr(), bd.data_ptr(), c.data_ptr(), sd.data_ptr(), k, k, n, n, m, n, ptr, size, None]
        assert lib.neso_plan_begin(0) == _lib.NESO_OK
        assert lib.neso_w8a16_matmul_ws(*args) == _lib.NESO_OK
        plan = json.loads(lib.neso_plan_end().decode())["launches"]
        assert len(plan) == launches and plan[0]["device_kernel"] == "w8a16_skinny_kernel"
        assert lib.neso_w8a16_matmul_ws(*args) == _lib.NESO_OK
        torch.cuda.synchronize()
        assert Q.rel_err(c.cpu().numpy(), ref) < 1e-5


def test_graph_replays(gpu):
    """Captured with its workspace in the graph's pool: replays match the
    eager result bit for bit, with other work in between."""
    m, n, k = 4, 1024, 4096
    a, b, s = (t.to(DEV) for t in _inputs(m, n, k, 3))
    c = torch.empty(m, n, device=DEV)

    def launch():
        neso_amd.w8a16_scaled_matmul(a, b, c, s, k, k, n, n, M=m, N=n)

    launch()
    eager = c.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch()
    for _ in range(4):
        c.fill_(float("nan"))
        torch.randn(1 << 20, device=DEV)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, eager)


# Every boundary of the unaligned 128 x 128-tile kernel: odd K, N and row
# strides, bases of A on 2 bytes and of B on any byte, single elements, K one
# short of and one past a step, ragged tiles in both directions; NaN in every
# element of A outside its rows.
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("m,n,k,lda,ldb,da,db", [
    (1, 1, 1, 1, 1, 0, 0), (1, 1, 1, 3, 5, 1, 3), (3, 7, 63, 64, 8, 0, 1), (5, 130, 65, 65, 131, 1, 2),
    (128, 128, 64, 65, 129, 0, 0), (129, 127, 127, 127, 127, 1, 1), (70, 256, 129, 136, 256, 4, 5),
    (200, 257, 640, 641, 259, 3, 3), (65, 301, 1999, 2001, 301, 0, 2)])
def test_unaligned(gpu, m, n, k, lda, ldb, da, db, scaled):
    a, b, s = _inputs(m, n, k, m + n + k, lda=lda, ldb=ldb)
    a[:, k:] = float("nan")
    abuf = torch.full((da + m * lda + 8,), float("nan"), dtype=torch.float16)
    abuf[da:da + m * lda] = a.reshape(-1)
    bbuf = torch.full((db + k * ldb,), 77, dtype=torch.int8)
    bbuf[db:] = b.reshape(-1)
    c = torch.full((m, n + 3), 5.0, device=DEV)
    ad, bd = abuf.to(DEV)[da:], bbuf.to(DEV)[db:]
    if scaled:
        neso_amd.w8a16_scaled_matmul(ad, bd, c, s.to(DEV), k, lda, ldb, n + 3, M=m, N=n)
    else:
        neso_amd.w8a16_matmul(ad, bd, c, k, lda, ldb, n + 3, M=m, N=n)
    c = c.cpu()
    assert Q.rel_err(c[:, :n].numpy(), _ref(a, b, s if scaled else None, k, n)) < 1e-5
    assert torch.all(c[:, n:] == 5.0)


# Split tiles: the last range short, more ranges than steps allow, and a
# result whose rows are no multiple of four.
@pytest.mark.parametrize("m,n,k", [(128, 1024, 1032), (100, 304, 4000), (300, 501, 2001), (65, 128, 8192)])
def test_split_tiles(gpu, m, n, k):
    a, b, s = _inputs(m, n, k, m + n + k)
    ad, bd, sd = a.to(DEV), b.to(DEV), s.to(DEV)
    c = torch.full((m, n), float("nan"), device=DEV)
    plan = neso_amd.launch_plan("w8a16_scaled_matmul", ad, bd, c, sd, k, k, n, n, M=m, N=n, cu_count=256)
    assert [p["device_kernel"] for p in plan] == ["w8a16_gemm_kernel", "w8a16_reduce_kernel"]
    assert plan[0]["grid"][2] > 1
    neso_amd.w8a16_scaled_matmul(ad, bd, c, sd, k, k, n, n, M=m, N=n)
    assert Q.rel_err(c.cpu().numpy(), _ref(a, b, s, k, n)) < 1e-5
