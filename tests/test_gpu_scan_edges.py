"""GPU parity at the sizes where the device scan and the band check change
kernels: one workgroup scans up to 32768 values (tiles of 4096), three kernels
above; one workgroup checks up to 4096 groups of four block-rows, atomics above.
"""
from __future__ import annotations

import numpy as np
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


@pytest.mark.parametrize("itype", [np.int32, np.int64])
@pytest.mark.parametrize("M", [1, 3, 63, 255, 4095, 4096, 4097, 20000, 32767, 32768, 32769, 50001])
def test_permuted_row_ptr(torch, M, itype):
    rng = np.random.default_rng(M)
    n = rng.integers(0, 6, size=M)
    rp = np.zeros(M + 1, itype)
    np.cumsum(n, out=rp[1:])
    ci = rng.integers(0, 50, size=int(rp[-1])).astype(itype)
    vals = rng.standard_normal(len(ci)).astype(np.float32)
    perm = rng.permutation(M).astype(itype)
    P = X.apply_permutation(X.CSRMatrix.from_host(M, 50, rp, ci, vals, device="cuda:0"), perm)
    want = np.zeros(M + 1, itype)
    np.cumsum(n[perm], out=want[1:])
    assert np.array_equal(P.row_ptr.cpu().numpy(), want)
    src = np.concatenate([np.arange(rp[o], rp[o + 1]) for o in perm]).astype(np.int64)
    assert np.array_equal(P.col_ind.cpu().numpy(), ci[src])
    assert np.array_equal(P.values.cpu().numpy(), vals[src])


@pytest.mark.parametrize("Mb", [1, 255, 4097, 32768, 32769])
def test_block_row_ptr(torch, Mb):
    """csr_to_bcsr's row pointers and total: block-row b holds b % 5 blocks."""
    K = 16 * 8
    dev = "cuda:0"
    b = torch.arange(Mb, device=dev)
    n = torch.zeros(Mb * 16, dtype=torch.int64, device=dev)
    n[::16] = b % 5  # the first row of each block-row, one entry per block
    rp = torch.zeros(Mb * 16 + 1, dtype=torch.int64, device=dev)
    rp[1:] = torch.cumsum(n, 0)
    first = torch.repeat_interleave(rp[:-1], n)
    ci = (torch.arange(int(rp[-1]), device=dev) - first) * 16
    A = X.CSRMatrix(Mb * 16, K, rp.int(), ci.int(), torch.ones(ci.numel(), device=dev))
    B = X.csr_to_bcsr(A)
    want = torch.zeros(Mb + 1, dtype=torch.int64, device=dev)
    want[1:] = torch.cumsum(b % 5, 0)
    assert torch.equal(B.row_ptr.long(), want) and B.num_blocks == int(want[-1])


@pytest.mark.parametrize("groups", [1, 4096, 4097])
@pytest.mark.parametrize("gap", [False, True])
def test_band_check(torch, groups, gap):
    """Block-rows of three neighbouring blocks (fp16 bands); with `gap` the last
    block-row's middle block is one column further."""
    Mb, dev = 4 * groups, "cuda:0"
    Kb = Mb + 4
    rp = (torch.arange(Mb + 1, device=dev) * 3).int()
    ci = (torch.arange(Mb, device=dev)[:, None] + torch.arange(3, device=dev)[None, :]).int()
    if gap:
        ci[-1, 2] += 1
    vals = torch.ones(Mb * 3 * 256, dtype=torch.float16, device=dev)
    A = X.BCSRMatrix(Mb, Kb, 16, 16, 16 * Mb, 16 * Kb, rp, ci.reshape(-1).contiguous(), vals)
    assert A.band_rows() is (not gap)
