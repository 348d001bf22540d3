"""Workgroup shapes that the cost model picks, on both sides of its lines:
tiny and ragged N, causal rows below 1024, windows narrower than a block and
wider than the sequence, with and without a rest round, fp16 and fp32 output.
The bar is the 2e-3 of the other FA2 tests."""
from __future__ import annotations

import math

import pytest
import torch

import neso_amd
from oracle import attention as A

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _qkv(bh, n, d, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(bh, n, d, generator=g).half() for _ in range(3))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("bh,n,d", [
    (1, 1, 64), (3, 17, 128), (2, 64, 64), (5, 65, 128), (8, 127, 64), (9, 129, 64), (30, 300, 128), (2, 511, 64),
    (70, 250, 64), (33, 900, 128), (20, 1000, 64), (5, 1025, 128), (7, 1300, 64), (40, 520, 128)])
def test_attention(gpu, bh, n, d, causal):
    q, k, v = _qkv(bh, n, d, bh + n)
    out = neso_amd.attention(q.to(DEV), k.to(DEV), v.to(DEV), causal=causal).cpu()
    ref = A.attention(q[None], k[None], v[None], 1 / math.sqrt(d), causal=causal)[0]
    assert (out - ref).abs().max().item() <= 2e-3


@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n,h,d,wl,wr", [
    (1, 2, 64, 3, 0), (63, 3, 128, 8, 8), (300, 10, 64, 40, 0), (400, 4, 64, 500, 0), (400, 4, 64, 399, 1),
    (1000, 8, 64, 64, 64), (1100, 6, 128, 0, 0), (1500, 5, 128, 100, 30), (2050, 3, 64, 1024, 1024)])
def test_window(gpu, n, h, d, wl, wr, out_dtype):
    q, k, v = (x.transpose(0, 1).contiguous() for x in _qkv(h, n, d, n + wl))
    out = neso_amd.window_attention(q.to(DEV), k.to(DEV), v.to(DEV), wl, wr, out_dtype=out_dtype).float().cpu()
    i = torch.arange(n)[:, None] - torch.arange(n)[None, :]
    s = torch.einsum("ihd,jhd->hij", q.float(), k.float()) / math.sqrt(d)
    s = s.masked_fill((i > wl) | (i < -wr), -math.inf)
    ref = torch.einsum("hij,jhd->ihd", torch.softmax(s, -1), v.float())
    assert (out - ref).abs().max().item() <= 2e-3
