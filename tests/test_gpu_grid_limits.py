"""Full grids at the N where one kernel's launch grid ends and another one still
covers the product: the fp32 shared and tile kernels count 64-column groups in a
grid dimension of 65535, the fp16 column batches 128-column ones.  Integer values
keep every sum exact, so C equals the dense product bit for bit.
"""
from __future__ import annotations

import pytest

import xspmm_amd as X

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need an MI355X (torch.cuda.is_available() is False)")
    X.load()
    return torch


def full_grid(torch, M, K, dtype):
    """Every block of an M x K matrix, and the matrix itself (fp32)."""
    dev = "cuda:0"
    D = (torch.arange(M * K, device=dev) * 7 % 9 - 4).view(M, K).float()
    blocks = D.view(M // 16, 16, K // 16, 16).transpose(1, 2).contiguous()
    Mb, Kb = M // 16, K // 16
    rp = (torch.arange(Mb + 1, device=dev) * Kb).int()
    ci = torch.arange(Kb, device=dev).repeat(Mb).int()
    return X.BCSRMatrix(Mb, Kb, 16, 16, M, K, rp, ci, blocks.view(-1).to(dtype)), D


def check(torch, M, K, N, dtype):
    A, D = full_grid(torch, M, K, dtype)
    B = (torch.arange(K * N, device="cuda:0") % 11 - 5).view(K, N).to(dtype)
    C = X.spmm(A, B, torch.full((M, N), -7.0, device="cuda:0"))
    for n0 in range(0, N, 1 << 20):
        want = D @ B[:, n0:n0 + (1 << 20)].float()
        assert torch.equal(C[:, n0:n0 + (1 << 20)], want), n0


# 64 columns past the last group that a grid of 65535 holds: 65535 * 64 = 4194240
@pytest.mark.parametrize("M,N", [(64, 4194240), (64, 4194300), (64, 4194241), (16, 4194300), (64, 4194304)])
def test_f32_columns_near_the_grid_limit(torch, M, N):
    print(M, N, flush=True)
    check(torch, M, 16, N, torch.float32)


# 65535 * 128 = 8388480
@pytest.mark.parametrize("N", [8388480, 8388488])
def test_f16_columns_near_the_grid_limit(torch, N):
    print(N, flush=True)
    check(torch, 16, 16, N, torch.float16)
