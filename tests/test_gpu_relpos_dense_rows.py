"""Dense f16 rel-pos bias on every row alignment: even T (rows on 4-byte
boundaries), odd T, an odd head stride and an odd base address, ragged last
blocks included, against the fp32 oracle at the attention bar of 2e-3 (fp16
probabilities and inputs, the bar of the other FA2 tests)."""
from __future__ import annotations

import math

import pytest
import torch

import neso_amd

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(h, t, d, pad=0, shift=0, neg=False, out=torch.float32, seed=0):
    """Bias rows contiguous; `pad` elements between heads, `shift` elements
    before the first; the elements outside the bias are NaN."""
    g = torch.Generator().manual_seed(seed + t)
    q, k, v = (torch.randn(h, t, d, generator=g).half() for _ in range(3))
    bias = torch.randn(h, t, t, generator=g).half()
    scale = (-1 if neg else 1) / math.sqrt(d)
    stride = t * t + pad
    buf = torch.full((shift + h * stride + 16,), float("nan"), dtype=torch.float16)
    for i in range(h):
        buf[shift + i * stride:shift + i * stride + t * t] = bias[i].reshape(-1)
    bd = buf.to(DEV)[shift:]
    o = torch.full((h, t, d), float("nan"), dtype=out, device=DEV)
    neso_amd.rel_pos_fa2_fwd(q.to(DEV), k.to(DEV), v.to(DEV), bd, o, t, d, scale, t * d, stride, num_heads=h)
    s = (q.float() @ k.float().transpose(1, 2) + bias.float()) * scale
    ref = torch.softmax(s, dim=-1) @ v.float()
    assert torch.isfinite(o).all()
    assert (o.float().cpu() - ref).abs().max().item() <= 2e-3


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("t", [1, 2, 3, 31, 62, 63, 65, 100, 129, 254, 511, 1026])
def test_rows(gpu, t, d):
    _run(2, t, d)


@pytest.mark.parametrize("t,pad,shift", [(64, 1, 0), (64, 0, 1), (66, 2, 2), (65, 1, 1), (65, 0, 1), (130, 3, 0)])
def test_strides_and_base(gpu, t, pad, shift):
    _run(3, t, 64, pad, shift)


@pytest.mark.parametrize("qw,ks", [("2", "1"), ("2", "4"), ("4", "1"), ("4", "3")])
@pytest.mark.parametrize("t", [253, 254])
def test_every_split(gpu, monkeypatch, t, qw, ks):
    monkeypatch.setenv("NESO_AMD_FA2_QW", qw)
    monkeypatch.setenv("NESO_AMD_FA2_KSPLIT", ks)
    _run(2, t, 64, neg=True, seed=3)
    _run(2, t, 128, seed=4, out=torch.float32)
