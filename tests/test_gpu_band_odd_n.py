"""fp32 bands of more than 64 columns whose rows of B start off 16 bytes: the tile
kernel on small grids, the band kernel on a padded copy of B on large ones.  Which
one ran shows in the order of the sums: C equals the forced tile kernel's bit for
bit, or does not.  Both are checked against fp64.
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


@pytest.mark.parametrize("M,half,N,tile", [(1024, 410, 127, True), (2048, 820, 511, True), (4096, 1024, 67, True),
                                           (4096, 1024, 129, True), (4096, 1024, 511, False), (8192, 410, 129, False),
                                           (8192, 2048, 67, False), (8190, 2048, 127, False)])
def test_kernel_and_result(torch, monkeypatch, M, half, N, tile):
    dev = "cuda:0"
    i = torch.arange(M, device=dev)
    D = torch.randn((M, M), device=dev) * ((i[:, None] - i[None, :]).abs() <= half)
    at = D.nonzero()
    rp = torch.searchsorted(at[:, 0].contiguous(), torch.arange(M + 1, device=dev))
    A = X.csr_to_bcsr(X.CSRMatrix(M, M, rp.int(), at[:, 1].int().contiguous(), D[at[:, 0], at[:, 1]]))
    assert A.band_rows()
    B = torch.randn((M, N), device=dev)
    C = X.spmm(A, B)
    want = D.double() @ B.double()
    # |sum error| <= n eps sum |a b|, n = 2 half + 1 terms; far above what occurs
    bound = (2 * half + 1) * 2.0 ** -24 * (D.abs().double() @ B.abs().double())
    assert bool(((C - want).abs() <= bound).all())
    monkeypatch.setenv("XSPMM_F32_KERNEL", "tile")
    A._band_key = A._order_key = None
    assert torch.equal(C, X.spmm(A, B)) is tile
