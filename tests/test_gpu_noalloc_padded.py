"""The allocation-free Tier-1 call against the allocating ones where rows of B
start off 16 bytes: whether B's padded copy fits the 8 MiB array or not, and on
full grids, each runs the same kernels, so C is equal bit for bit.  Real-valued
inputs, so that another kernel's order of sums would show.
"""
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
    return torch


@pytest.fixture(scope="module")
def lib(torch):
    L = X.load()
    p, i64, i32 = C.c_void_p, C.c_int64, C.c_int
    for fn in (L.xspmm_bcsr_spmm, L.xspmm_bcsr_spmm_noalloc, L.xspmm_bcsr_spmm_band):
        fn.restype = i32
        fn.argtypes = [i32, i32, i64, i64, i64, i64, i64, p, p, p, p, p, i64, p]
    return L


def matrix(torch, M, K, per_row, dtype):
    """per_row entries anywhere in each row; per_row 0: every block present."""
    g = torch.Generator(device="cuda:0")
    g.manual_seed(M + K)
    if per_row == 0:
        cols = torch.arange(0, K, 16, device="cuda:0") + torch.arange(M, device="cuda:0")[:, None] % 16
        cols = cols.clamp(max=K - 1)
    else:
        cols = torch.randint(K, (M, per_row), generator=g, device="cuda:0")
    keys = torch.unique((torch.arange(M, device="cuda:0")[:, None] * K + cols).reshape(-1))
    rp = torch.searchsorted(keys, torch.arange(M + 1, device="cuda:0") * K)
    vals = torch.randn(keys.numel(), generator=g, device="cuda:0").to(dtype)
    return X.csr_to_bcsr(X.CSRMatrix(M, K, rp.int(), (keys % K).int(), vals))


# K = 16384 in fp32: 124 columns of copy are 8 126 464 bytes, 128 are all 8 MiB and
# leave no room for the marks.  K = 32768 in fp16: the panels of N = 127 are all of
# the array, the copy and its marks more.  60000 rows: the marks, the copy and an
# order.
CASES = [("f32", 4099, 16384, 48, (121, 123, 125, 127, 129)), ("f32", 60000, 5003, 8, (33, 129, 397, 419)),
         ("f32", 515, 97, 0, (33, 131)), ("f32", 2050, 1601, 0, (5, 257, 301)),
         ("f16", 3000, 32768, 16, (119, 121, 127)), ("f16", 515, 97, 0, (8, 33, 256)),
         ("f16", 2050, 1601, 0, (5, 8, 257))]


@pytest.mark.parametrize("values,M,K,per_row,columns", CASES)
def test_noalloc_equals_allocating(torch, lib, values, M, K, per_row, columns):
    dtype = torch.float16 if values == "f16" else torch.float32
    A = matrix(torch, M, K, per_row, dtype)
    order = torch.arange(A.num_block_rows, dtype=torch.int32, device="cuda:0")
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for N in columns:
        print(values, M, K, N, A.num_blocks, flush=True)
        B = torch.randn((K, N), device="cuda:0").to(dtype)
        args = [X.vcode(dtype), X.I32, M, K, A.num_block_rows, A.num_block_cols, A.num_blocks] + [
            C.c_void_p(t.data_ptr()) for t in (A.row_ptr, A.col_ind, A.values, B)]
        out = [torch.full((M, N), float("nan"), device="cuda:0") for _ in range(3)]
        calls = [lambda c: lib.xspmm_bcsr_spmm(*args, c, N, s), lambda c: lib.xspmm_bcsr_spmm_noalloc(*args, c, N, s),
                 lambda c: lib.xspmm_bcsr_spmm_ordered(*args, c, N, C.c_void_p(order.data_ptr()), s)]
        for call, c in zip(calls, out):
            assert call(C.c_void_p(c.data_ptr())) == X.OK, lib.xspmm_last_error().decode()
        assert bool(torch.isfinite(out[0]).all())
        assert torch.equal(out[0], out[1])
        assert torch.equal(out[0], out[2])
