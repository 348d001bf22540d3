"""The magnitude check of the split-precision calls: one kernel that gives
the largest |x| of up to three fp32 tensors, exactly as torch does."""
from __future__ import annotations

import math

import pytest
import torch

import neso_amd
from neso_amd import kernels as KN

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _maxima(views, add=None):
    check = KN._RangeCheck(views, torch.cuda.current_stream().cuda_stream, add)
    assert check.each > 0
    return check.wait()


# One quad, fewer quads than a workgroup's threads, ragged grids, more work
# than one pass of the largest grid.
@pytest.mark.parametrize("b,n,d", [(1, 1, 4), (1, 1, 32), (3, 7, 32), (2, 129, 64), (8, 1000, 128), (64, 4099, 64)])
@pytest.mark.parametrize("where", ["first", "last"])
def test_contiguous(gpu, b, n, d, where):
    g = torch.Generator(device=DEV).manual_seed(b * n + d)
    xs = [torch.randn(b, n, d, generator=g, device=DEV) for _ in range(3)]
    for i, x in enumerate(xs):
        x.view(-1)[0 if where == "first" else -1] = (-1) ** i * (100.0 + i)
    assert _maxima([(x, b, n, d, d, n * d) for x in xs]) == [x.abs().max().item() for x in xs] == [100.0, 101.0, 102.0]


def test_strided_and_added(gpu):
    """Rows of a wider tensor (the rest must not count), and the bias_v of
    the precompute added to the first tensor."""
    b, n, d = 3, 50, 64
    g = torch.Generator(device=DEV).manual_seed(5)
    big = torch.full((b, n + 2, 2 * d), 1e9, device=DEV)
    big[:, :n, :d] = torch.randn(b, n, d, generator=g, device=DEV)
    other = torch.randn(b, 2 * n - 1, d, generator=g, device=DEV)
    add = torch.randn(b, d, generator=g, device=DEV)
    views = [(big, b, n, d, 2 * d, (n + 2) * 2 * d), (other, b, 2 * n - 1, d, d, (2 * n - 1) * d)]
    assert _maxima(views) == [big[:, :n, :d].abs().max().item(), other.abs().max().item()]
    assert _maxima(views, add) == [(big[:, :n, :d] + add[:, None]).abs().max().item(), other.abs().max().item()]


def test_nonfinite_and_zero(gpu):
    n = 777
    z = torch.zeros(1, n, 32, device=DEV)
    inf, nan = z.clone(), z.clone()
    inf[0, 500, 3] = -math.inf
    nan[0, 20, 1], nan[0, 700, 9] = math.nan, math.inf
    m = _maxima([(x, 1, n, 32, 32, n * 32) for x in (z, inf, nan)])
    assert m[0] == 0.0 and math.isinf(m[1]) and math.isnan(m[2])


def test_rescaled_call_after_a_queued_one(gpu):
    """attention() queues its kernel behind the check: tiny and huge inputs
    are run again rescaled, an infinite one is refused, and the next plain
    call is not disturbed."""
    g = torch.Generator(device=DEV).manual_seed(1)
    q, k, v = (torch.randn(2, 300, 64, generator=g, device=DEV) for _ in range(3))
    ref = neso_amd.attention(q, k, v)
    out = neso_amd.attention(q, k, v * 1e-5)
    assert (out * 1e5 - ref).abs().max().item() < 1e-4
    assert (neso_amd.attention(q, k, v * 1e6) * 1e-6 - ref).abs().max().item() < 1e-4
    bad = k.clone()
    bad[1, 5, 5] = math.inf
    with pytest.raises(neso_amd.NesoArgumentError, match="K: infinite"):
        neso_amd.attention(q, bad, v)
    assert torch.equal(neso_amd.attention(q, k, v), ref)


def test_side_stream_and_out(gpu):
    """An explicit O (checked before the launch) on a side stream."""
    g = torch.Generator(device=DEV).manual_seed(2)
    q, k, v = (torch.randn(2, 200, 64, generator=g, device=DEV) for _ in range(3))
    ref = neso_amd.attention(q, k, v)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    o = torch.empty_like(ref)
    neso_amd.flash_attention_fwd(q, k, v, o, 200, 64, 64, 0.125, batch_heads=2, stride_bh_qo=200 * 64,
                                 stride_bh_kv=200 * 64, stream=s)
    s.synchronize()
    assert torch.equal(o, ref)


def test_precompute_limit(gpu):
    q = torch.zeros(2, 40, 64, device=DEV)
    k_rel = torch.zeros(2, 79, 64, device=DEV)
    u = v = torch.zeros(2, 64, device=DEV)
    k_rel[1, 78, 63] = 65503.0
    neso_amd.precompute_bias_and_qu(q, k_rel, u, v)
    k_rel[1, 78, 63] = 65504.0
    with pytest.raises(neso_amd.NesoArgumentError, match="K_rel"):
        neso_amd.precompute_bias_and_qu(q, k_rel, u, v)
