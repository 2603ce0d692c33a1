"""GPU parity of products whose B rows do not start on 16 bytes (N % 8 != 0 in
fp16, N % 4 != 0 in fp32, or fp32 B / C off a 16-byte boundary): Tier-1 and
plans multiply a copy of B with padded rows on the column-batch, band and
full-grid kernels.  Full grids of few columns take the column batches too, for
any N.

Integer-valued A and B keep every fp32 partial sum exact, so C must equal the
fp64 tile product bit for bit.  An Inf or NaN must reach exactly the
entries of C it reaches in the reference's tile product
(src/common/spmm_math.hpp:93-110), which multiplies whole blocks.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import xspmm_amd as X

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need an MI355X (torch.cuda.is_available() is False)")
    X.load()
    return torch


def integer_csr(kind, M, K, dtype, itype, seed):
    """Rows of distinct columns with values in -4 .. 4, no zeros."""
    rng = np.random.default_rng(seed)
    rows = []
    for i in range(M):
        if kind == "full":  # one entry in every block of the block-row, at least
            c = np.arange(i % 16, K, 16) if K % 16 == 0 else np.unique(
                np.minimum(np.arange(0, K + 15, 16) + i % 16, K - 1))
        elif kind == "band":
            c = np.arange(max(0, i - 70), min(K, i + 71))
        elif kind == "wide":
            c = np.arange(max(0, i - 300), min(K, i + 301))
        elif kind == "deep":
            c = np.unique(rng.integers(0, K, 48))
        else:
            c = np.sort(rng.choice(K, size=int(rng.integers(0, min(K, 9))), replace=False))
        rows.append(c)
    rp = np.zeros(M + 1, itype)
    np.cumsum([len(c) for c in rows], out=rp[1:])
    ci = np.concatenate(rows).astype(itype)
    vals = rng.choice([-4, -3, -2, -1, 1, 2, 3, 4], size=len(ci)).astype(dtype)
    return rp, ci, vals


def product(A, B):
    """The tile product of A's BCSR form in fp64: every column of a block,
    zeros included, meets its B row (oracle.bcsr_spmm_f64 skips zeros)."""
    brp, bci, bv = (t.cpu().numpy() for t in (A.row_ptr, A.col_ind, A.values))
    B = B.astype(np.float64)
    C = np.zeros((A.num_block_rows * 16, B.shape[1]))
    blocks = bv.reshape(-1, 16, 16).astype(np.float64)
    with np.errstate(invalid="ignore"):
        for r in range(A.num_block_rows):
            at = slice(int(brp[r]), int(brp[r + 1]))
            cols = (bci[at, None] * 16 + np.arange(16)).reshape(-1)
            inside = cols < A.num_cols
            rows = blocks[at].transpose(1, 0, 2).reshape(16, -1)
            C[16 * r:16 * r + 16] = rows[:, inside] @ B[cols[inside]]
    return C[:A.num_rows]


# fp32 takes the padded copy from 2^18 products of a block with a 16-column tile
# and N > 16 ("deep": 73521 blocks), the tile kernel below; full grids of many
# columns (2050 x 1601 from N = 250) the kernel of banded grids, and bands ("wide")
# of few columns the tile kernel
SHAPES = [("deep", 4099, 5003), ("sparse", 8197, 203), ("sparse", 333, 500), ("band", 1003, 997), ("full", 515, 97),
          ("full", 131, 1601), ("full", 2050, 1601), ("wide", 4003, 3997)]


@pytest.mark.parametrize("itype", [np.int32, np.int64])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("kind,M,K", SHAPES)
def test_odd_n_exact(torch, kind, M, K, dtype, itype):
    rp, ci, vals = integer_csr(kind, M, K, dtype, itype, seed=M)
    A = X.csr_to_bcsr(X.CSRMatrix.from_host(M, K, rp, ci, vals, device="cuda:0"))
    rng = np.random.default_rng(1)
    for N in (1, 2, 7, 8, 15, 17, 33, 63, 65, 72, 127, 129, 256, 257, 301):
        print(kind, M, K, dtype.__name__, itype.__name__, N, flush=True)
        B = rng.integers(-8, 9, size=(K, N)).astype(dtype)
        guard = torch.full((M * N + 64,), -7.0, device="cuda:0")
        C = X.spmm(A, torch.as_tensor(B).cuda(), guard[:M * N].view(M, N))
        assert np.array_equal(C.cpu().numpy(), product(A, B))
        assert bool((guard[M * N:] == -7.0).all())  # nothing stored past C


@pytest.mark.parametrize("itype", [np.int32, np.int64])
def test_f32_off_16_bytes(torch, itype):
    """fp32 B and C may start on any float: N % 4 == 0 with either off 16 bytes."""
    M, K, N = 4099, 5003, 72
    rp, ci, vals = integer_csr("deep", M, K, np.float32, itype, seed=3)
    A = X.csr_to_bcsr(X.CSRMatrix.from_host(M, K, rp, ci, vals, device="cuda:0"))
    B = np.random.default_rng(2).integers(-8, 9, size=(K, N)).astype(np.float32)
    want = product(A, B)
    for db, dc in ((1, 0), (0, 1), (3, 2)):
        b = torch.zeros(K * N + 4, device="cuda:0")[db:db + K * N].view(K, N)
        b.copy_(torch.as_tensor(B))
        c = torch.empty(M * N + 4, device="cuda:0")[dc:dc + M * N].view(M, N)
        assert np.array_equal(X.spmm(A, b, c).cpu().numpy(), want)


@pytest.mark.parametrize("itype", [np.int32, np.int64])
def test_f32_full_grid_in_another_order(torch, itype):
    """A caller's full grid whose rows hold their blocks in any order, and one
    whose block columns lie outside the grid (they contribute nothing)."""
    M, K, N = 2050, 1601, 260
    rp, ci, vals = integer_csr("full", M, K, np.float32, itype, seed=4)
    A = X.csr_to_bcsr(X.CSRMatrix.from_host(M, K, rp, ci, vals, device="cuda:0"))
    assert A.num_blocks == A.num_block_rows * A.num_block_cols
    B = np.random.default_rng(3).integers(-8, 9, size=(K, N)).astype(np.float32)
    want = product(A, B)
    b = torch.as_tensor(B).cuda()
    assert np.array_equal(X.spmm(A, b).cpu().numpy(), want)
    Kb = A.num_block_cols
    at = torch.arange(A.num_blocks, device="cuda:0").view(-1, Kb)
    at[5] = at[5].flip(0)          # one block-row reversed
    at[-1] = at[-1].roll(3)
    flat = at.reshape(-1)
    S = X.BCSRMatrix(A.num_block_rows, Kb, 16, 16, M, K, A.row_ptr, A.col_ind[flat].contiguous(),
                     A.values.view(-1, 256)[flat].reshape(-1).contiguous())
    assert np.array_equal(X.spmm(S, b).cpu().numpy(), want)
    ci2 = A.col_ind.clone()
    ci2[40 * Kb + 7] = Kb + 3      # outside the grid
    S = X.BCSRMatrix(A.num_block_rows, Kb, 16, 16, M, K, A.row_ptr, ci2, A.values)
    v = A.values.clone()
    v.view(-1, 256)[40 * Kb + 7] = 0
    Z = X.BCSRMatrix(A.num_block_rows, Kb, 16, 16, M, K, A.row_ptr, A.col_ind, v)
    assert np.array_equal(X.spmm(S, b).cpu().numpy(), product(Z, B))


@pytest.mark.parametrize("where", ["A", "B"])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("kind,M,K", SHAPES)
def test_nonfinite_reaches_what_the_reference_reaches(torch, kind, M, K, dtype, where):
    rp, ci, vals = integer_csr(kind, M, K, dtype, np.int32, seed=M + 1)
    for N, special in ((5, np.inf), (67, -np.inf), (131, np.nan), (40, np.inf)):
        if N % 8 == 0 and kind not in ("full", "band", "wide"):
            continue  # the column batches of aligned rows skip zero columns
        print(kind, M, K, dtype.__name__, where, N, flush=True)
        v = vals.copy()
        B = np.random.default_rng(N).integers(1, 9, size=(K, N)).astype(dtype)
        if where == "A":
            v[len(v) // 2] = special
        else:
            B[K // 2, N // 2] = special
        A = X.csr_to_bcsr(X.CSRMatrix.from_host(M, K, rp, ci, v, device="cuda:0"))
        C = X.spmm(A, torch.as_tensor(B).cuda()).cpu().numpy()
        assert np.array_equal(C, product(A, B), equal_nan=True)


@pytest.mark.parametrize("cluster", [False, True])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_plan_and_pipeline_odd_n(torch, dtype, cluster):
    M, K = 4099, 5003
    rp, ci, vals = integer_csr("deep", M, K, dtype, np.int32, seed=9)
    A = X.CSRMatrix.from_host(M, K, rp, ci, vals, device="cuda:0")
    plan = X.SpMMPlan(A, optimize_pattern=cluster)
    for N in (3, 67, 130):
        B = np.random.default_rng(N).integers(-8, 9, size=(K, N)).astype(dtype)
        want = oracle.csr_spmm_f64(M, N, rp, ci, vals, B)
        b = torch.as_tensor(B).cuda()
        assert np.array_equal(plan.execute(b).cpu().numpy(), want)
        assert np.array_equal(X.spmm_pipeline(A, b, optimize_pattern=cluster)[0].cpu().numpy(), want)


@pytest.mark.parametrize("where", [None, "A", "B"])
@pytest.mark.parametrize("cluster", [False, True])
@pytest.mark.parametrize("itype", [np.int32, np.int64])
def test_packed_plan_on_padded_b(torch, itype, cluster, where):
    """fp16 plans of sparse blocks ("deep": 73521 of them) multiply their packed
    batches on the padded copy from N = 257; an Inf or NaN takes whole blocks."""
    M, K = 4099, 5003
    rp, ci, vals = integer_csr("deep", M, K, np.float16, itype, seed=11)
    if where == "A":
        vals[len(vals) // 2] = np.inf
    A = X.CSRMatrix.from_host(M, K, rp, ci, vals, device="cuda:0")
    plan = X.SpMMPlan(A, optimize_pattern=cluster)
    assert plan.packed_batches > 0
    # the rows' order decides which blocks cover which rows
    perm = X.jaccard_clustering(A) if cluster else torch.arange(M, dtype=A.row_ptr.dtype, device="cuda:0")
    blocks = X.csr_to_bcsr(X.apply_permutation(A, perm))
    rows = perm.cpu().numpy()
    for N in (129, 257, 260, 391):
        print(itype.__name__, cluster, where, N, flush=True)
        B = np.random.default_rng(N).integers(1, 9, size=(K, N)).astype(np.float16)
        if where == "B":
            B[K // 2, N // 2] = np.nan if N == 260 else -np.inf
        want = np.empty((M, N))
        want[rows] = product(blocks, B)
        guard = torch.full((M * N + 64,), -7.0, device="cuda:0")
        C = plan.execute(torch.as_tensor(B).cuda(), guard[:M * N].view(M, N))
        assert np.array_equal(C.cpu().numpy(), want, equal_nan=True)
        assert bool((guard[M * N:] == -7.0).all())
