"""int4 tile GEMM with the weights staged through LDS four steps at a time:
step counts that do not divide by four or by the K-groups, scales of every
power-of-two group, rows past N, and K ranges that end inside a batch, for
all seven tile forms.  Against the float64 oracle at the bar of the other
int4 tests, 2e-3 of max|ref|."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import neso_amd
from oracle import inputs as I
from oracle import qmatmul as Q

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("form", ["1", "2", "3", "4", "5", "6", "7"])
@pytest.mark.parametrize("m,n,k,group", [
    (17, 16, 64, 32), (33, 40, 128, 64), (40, 33, 192, 32), (130, 100, 320, 64), (65, 129, 384, 128),
    (48, 70, 2112, 32), (129, 65, 4160, 32), (50, 200, 4224, 128), (20, 31, 11008, 256), (64, 90, 1280, 64),
    (70, 40, 4128, 32), (35, 50, 192, 192)])
def test_forms(gpu, monkeypatch, form, m, n, k, group):
    monkeypatch.setenv("NESO_AMD_W4_TILE_GEMM", form)
    x, codes, scales = I.qmatmul_inputs(m, k, n, group=group, seed=m + n + k)
    words = Q.pack_int4(codes.numpy())
    y = neso_amd.w4a16_linear(x.to(DEV), torch.as_tensor(words).to(DEV), scales.to(DEV), group_size=group)
    ref = Q.w4a16_matmul(x.numpy(), words, scales.numpy(), group, dtype=np.float64)
    assert Q.rel_err(y.float().cpu().numpy(), ref) <= 2e-3


@pytest.mark.parametrize("form", ["1", "2", "3", "5", "6", "7"])
@pytest.mark.parametrize("k,group", [(192, 32), (320, 32), (384, 64), (640, 128)])
def test_neighbour_scales_stay_out(gpu, monkeypatch, form, k, group):
    """A batch past the end of a row reads the next row's scales: infinite
    and NaN ones there must not reach this row."""
    monkeypatch.setenv("NESO_AMD_W4_TILE_GEMM", form)
    m, n = 40, 66
    x, codes, scales = I.qmatmul_inputs(m, k, n, group=group, seed=k)
    words = Q.pack_int4(codes.numpy())
    ref = Q.w4a16_matmul(x.numpy(), words, scales.numpy(), group, dtype=np.float64)
    scales[1::2] = float("inf")
    scales[3::4] = float("nan")
    y = neso_amd.w4a16_linear(x.to(DEV), torch.as_tensor(words).to(DEV), scales.to(DEV), group_size=group)
    assert Q.rel_err(y[:, ::2].float().cpu().numpy(), ref[:, ::2]) <= 2e-3
