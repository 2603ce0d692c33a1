"""fp16 products with N % 8 != 0: which kernel a grid takes, told by the order of its
sums, and the stores of C rows off 16 bytes.  Short rows of many columns keep panels
of B, in Tier-1, plans and the pipeline alike."""
from __future__ import annotations

import ctypes as C

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


def csr(torch, M, K, per_row, seed=0):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(M + K + seed)
    keys = torch.unique((torch.arange(M, device="cuda:0")[:, None] * K +
                         torch.randint(K, (M, per_row), generator=g, device="cuda:0")).reshape(-1))
    rp = torch.searchsorted(keys, torch.arange(M + 1, device="cuda:0") * K)
    vals = torch.randn(keys.numel(), generator=g, device="cuda:0").half()
    D = torch.zeros(M * K, device="cuda:0", dtype=torch.float64)
    D[keys] = vals.double()
    return X.CSRMatrix(M, K, rp.int(), (keys % K).int(), vals), D.view(M, K)


@pytest.mark.parametrize("cluster", [False, True])
@pytest.mark.parametrize("M,K,per_row", [(8205, 300, 6), (8205, 700, 2), (40000, 300, 3)])
@pytest.mark.parametrize("N", [33, 65, 67, 129, 391, 1023])
def test_short_rows(torch, M, K, per_row, N, cluster):
    A, D = csr(torch, M, K, per_row)
    blocks = X.csr_to_bcsr(A)
    assert blocks.num_blocks < (20 if K == 300 else 32) * blocks.num_block_rows
    B = torch.randn((K, N), device="cuda:0").half()
    guard = torch.full((M * N + 64,), -7.0, device="cuda:0")
    got = X.spmm(blocks, B, guard[:M * N].view(M, N))
    # |sum error| <= n eps sum |a b|, n terms of a row's blocks
    bound = K * 2.0 ** -24 * (D.abs() @ B.abs().double())
    assert bool(((got - D @ B.double()).abs() <= bound).all())
    assert bool((guard[M * N:] == -7.0).all())
    plan = X.SpMMPlan(A, optimize_pattern=cluster)
    assert torch.equal(plan.execute(B), X.spmm_pipeline(A, B, optimize_pattern=cluster)[0])


def test_scratch_tells_panels_from_a_copy(torch):
    """Panels hold 16 columns to a tile and whole blocks of rows, a copy 8 and marks."""
    out = C.c_int64(0)

    def scratch(Mb, nnzb, N, K=8000):
        assert X.load().xspmm_bcsr_spmm_scratch(X.F16, Mb * 16, K, Mb, K // 16, nnzb, 0, 0, N, 1, 0,
                                                C.byref(out)) == X.OK
        return out.value

    for N, panels in ((33, False), (64, False), (65, False), (129, True), (257, True)):
        copy, panel = -(-(256 + 8000 * (-(-N // 8) * 8) * 2) // 256) * 256, 8000 * (-(-N // 16) * 16) * 2
        if N % 8:
            assert scratch(900, 20 * 900 - 1, N) == (panel if panels else copy)
            assert scratch(900, 20 * 900, N) == copy
            assert scratch(300, 20 * 300 - 1, N) == copy  # at most 900 workgroups


@pytest.mark.parametrize("M,K", [(811, 303), (305, 1003)])
@pytest.mark.parametrize("N", [67, 257, 511])
def test_full_grids_of_odd_columns(torch, M, K, N):
    """Small full grids, in batches or tiles on a padded copy, stores guarded."""
    A, D = csr(torch, M, K, K)
    blocks = X.csr_to_bcsr(A)
    assert blocks.num_blocks == blocks.num_block_rows * blocks.num_block_cols
    B = torch.randn((K, N), device="cuda:0").half()
    guard = torch.full((M * N + 64,), -7.0, device="cuda:0")
    got = X.spmm(blocks, B, guard[:M * N].view(M, N))
    bound = K * 2.0 ** -24 * (D.abs() @ B.abs().double())
    assert bool(((got - D @ B.double()).abs() <= bound).all())
    assert bool((guard[M * N:] == -7.0).all())


def test_full_grids_price_the_copy_for_both_kernels():
    """A small full grid of odd columns is multiplied in batches, which take an order
    of a long grid's rows beside the copy; the tiles of a wide one do not."""
    out = C.c_int64(0)
    L = X.load()
    for Mb, Kb, N, batches in ((2100, 30, 9, True), (2100, 30, 1023, False)):
        assert L.xspmm_bcsr_spmm_scratch(X.F16, Mb * 16, Kb * 16, Mb, Kb, Mb * Kb, 0, 0, N, 0, 0, C.byref(out)) == X.OK
        copy = -(-(256 + Kb * 16 * (-(-N // 8) * 8) * 2) // 256) * 256
        assert out.value == copy + (4 * Mb if batches else 0), (Mb, Kb, N)
