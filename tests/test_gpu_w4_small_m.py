"""int4 small-M routes: X in LDS for every power-of-two group, long K in
phases, M up to 32, and the GEMV past K = 8192, against the float64 oracle.

Bar: max|err| / max|ref| <= 2e-3 as in the other int4 tests (weights rounded
to fp16 once, 2^-11 relative each, and the fp16 result).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import neso_amd
from oracle import inputs as I
from oracle import qmatmul as Q

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(m, n, k, group, kernel, targs=None, zero=8):
    x, codes, scales = I.qmatmul_inputs(m, k, n, group=group, seed=m + n + k + group)
    words = Q.pack_int4(codes.numpy())
    xd, wd, sd = x.to(DEV), torch.as_tensor(words).to(DEV), scales.to(DEV)
    y = torch.full((m, n), float("nan"), dtype=torch.float16, device=DEV)
    plan = neso_amd.launch_plan("w4a16_matmul", xd, wd, sd, y, m, n, k, k, n, group, zero, cu_count=256)
    assert [p["device_kernel"] for p in plan] == [kernel], plan
    for at, want in (targs or {}).items():
        assert plan[0]["template_args"][at] == want, plan
    neso_amd.w4a16_linear(xd, wd, sd, group_size=group, zero_point=zero, out=y)
    ref = Q.w4a16_matmul(x.numpy(), words, scales.numpy(), group, zero, dtype=np.float64)
    assert Q.rel_err(y.float().cpu().numpy(), ref) <= 2e-3


# QWMAX (index 2), scales per quad (3), phases (4): one quad, a ragged tile,
# fewer quads than waves, several tiles per workgroup, and phases with a
# short last one (4224 = 17 + 16 quads, 11008 = 3 x 29 - 1).
@pytest.mark.parametrize("m,n,k,group,qw,gs,mp", [
    (3, 7, 128, 128, 4, 1, 0), (16, 100, 256, 64, 4, 2, 0), (5, 4100, 4096, 64, 4, 2, 0),
    (16, 13000, 1024, 1024, 4, 1, 0), (16, 300, 4096, 4096, 4, 1, 0), (16, 200, 4224, 128, 4, 1, 1),
    (9, 16, 11008, 256, 4, 1, 1), (8, 1024, 11008, 32, 4, 4, 1), (16, 1040, 8192, 32, 4, 4, 1),
    (15, 4120, 5120, 64, 4, 2, 1),
    (17, 1024, 1024, 32, 2, 4, 1), (32, 1030, 2048, 64, 2, 2, 1), (31, 4104, 2176, 128, 2, 1, 1),
    (18, 12300, 4224, 32, 2, 4, 1)])
def test_x_in_lds(gpu, m, n, k, group, qw, gs, mp):
    _check(m, n, k, group, "w4a16_skinny_lds_kernel", {2: qw, 3: gs, 4: mp})


# The other side of each line of the rule.
@pytest.mark.parametrize("m,n,k,group,kernel", [
    (16, 100, 480, 96, "w4a16_skinny_kernel"), (16, 100, 160, 32, "w4a16_skinny_kernel"),
    (16, 100, 1152, 384, "w4a16_skinny_kernel"), (17, 1023, 1024, 32, "w4a16_tile_gemm_kernel"),
    (32, 1024, 896, 128, "w4a16_tile_gemm_kernel"), (32, 8200, 1024, 32, "w4a16_tile_gemm_kernel"),
    (33, 1024, 1024, 32, "w4a16_tile_gemm_kernel"), (17, 1024, 1056, 32, "w4a16_tile_gemm_kernel")])
def test_rule_lines(gpu, m, n, k, group, kernel):
    _check(m, n, k, group, kernel)


# Six and eight chunks per lane (GI, index 1), ragged chunk counts, 2, 4 and
# 8 rows per wave; M = 2 only while two rows per wave fill the chip.
@pytest.mark.parametrize("m,n,k,group,gi,r", [
    (1, 1024, 8224, 32, 6, 2), (1, 1030, 12288, 128, 6, 2), (1, 1100, 12320, 32, 8, 2),
    (1, 1024, 16384, 64, 8, 2), (1, 4099, 11008, 32, 6, 4), (1, 6150, 8448, 32, 6, 8),
    (2, 1024, 11008, 32, 6, 2), (2, 4095, 16384, 128, 8, 2)])
def test_gemv_long_k(gpu, m, n, k, group, gi, r):
    _check(m, n, k, group, "w4a16_gemv_kernel", {0: m, 1: gi, 2: r}, zero=7)


def test_wide_rows_of_x(gpu):
    """Padded rows of X (NaN past K) and of Y on the phase path."""
    m, n, k, group = 20, 1032, 2304, 128
    x, codes, scales = I.qmatmul_inputs(m, k, n, group=group, seed=1)
    words = torch.from_numpy(Q.pack_int4(codes.numpy())).to(DEV)
    xp = torch.full((m, k + 40), float("nan"), dtype=torch.float16, device=DEV)
    xp[:, :k] = x.to(DEV)
    y = torch.full((m, n + 3), 5.0, dtype=torch.float16, device=DEV)
    neso_amd.w4a16_matmul(xp, words, scales.to(DEV), y, m, n, k, k + 40, n + 3, group)
    ref = Q.w4a16_matmul(x.numpy(), words.cpu().numpy(), scales.numpy(), group)
    assert Q.rel_err(y[:, :n].float().cpu().numpy(), ref) <= 2e-3
    assert torch.all(y[:, n:].cpu() == 5.0)
