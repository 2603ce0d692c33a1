"""xspmm_bcsr_spmm_scratch: what a Tier-1 product takes beside its operands, from
its sizes (no GPU is asked)."""
from __future__ import annotations

import ctypes as C
import threading

import pytest

import xspmm_amd as X

LIMIT = 1 << 31


def scratch(vt, M, K, N, nnzb, ordered=True, b=0, c=0):
    out = C.c_int64(-1)
    rc = X.load().xspmm_bcsr_spmm_scratch(vt, M, K, -(-M // 16), -(-K // 16), nnzb, b, c, N, int(ordered), 0,
                                          C.byref(out))
    assert rc == X.OK, X.load().xspmm_last_error().decode()
    return out.value


def copy(value_bytes, K, N):
    per = 16 // value_bytes
    n = 256 + K * (-(-N // per) * per) * value_bytes
    return -(-n // 256) * 256  # where an order would begin


@pytest.mark.parametrize("vt,M,K,N,nnzb,want", [
    # fp32: aligned rows, the tile kernel (16 columns, few blocks), B beyond 2^31
    # bytes: nothing
    (X.F32, 16384, 16384, 128, 10 ** 6, 0), (X.F32, 16384, 16384, 16, 10 ** 6, 0),
    (X.F32, 16384, 16384, 3, 10 ** 6, 0), (X.F32, 16384, 16384, 33, 10 ** 4, 0),
    (X.F32, 16384, 1 << 20, 513, 10 ** 6, 0),
    # the batches on a padded copy
    (X.F32, 16384, 16384, 17, 10 ** 6, copy(4, 16384, 17)), (X.F32, 16384, 1 << 20, 509, 10 ** 6, copy(4, 1 << 20, 509)),
    # fp16: aligned rows; a padded copy; a full grid's marks; panels beyond 2^31 bytes
    (X.F16, 16384, 16384, 128, 10 ** 6, 0), (X.F16, 5003, 4999, 31, 90000, copy(2, 4999, 31)),
    (X.F16, 4096, 4096, 2048, 65536, 0), (X.F16, 4096, 4096, 8, 65536, 256),
    (X.F16, 16384, 1 << 20, 1031, 10 ** 6, (1 << 20) * 1040 * 2),
])
def test_bytes(vt, M, K, N, nnzb, want):
    assert scratch(vt, M, K, N, nnzb) == want


def test_wide_b():
    """fp32: no copy of a B with more than nine rows to a block, however many columns."""
    for K, nnzb, pads in ((500000, 15987, False), (500000, 236400, True), (2000000, 15996, False),
                          (2000000, 956467, True), (100000, 15922, True), (143298, 15922, True), (143299, 15922, False)):
        assert (scratch(X.F32, 4000, K, 257, nnzb) > 0) is pads, (K, nnzb)


def test_alignment_and_order():
    # B off 16 bytes is copied, C only marked
    assert scratch(X.F32, 16384, 16384, 128, 10 ** 6, b=4) == copy(4, 16384, 128)
    assert scratch(X.F32, 16384, 16384, 128, 10 ** 6, c=4) == 256
    # more than 2048 block-rows without an order
    assert scratch(X.F32, 60000, 4096, 64, 10 ** 6, ordered=False) == 4 * 3750
    assert scratch(X.F16, 60000, 4096, 33, 10 ** 6, ordered=False) == copy(2, 4096, 33) + 4 * 3750


def test_errors():
    # in a thread of its own: the library keeps the last error per thread
    L, codes = X.load(), []

    def calls():
        out = C.c_int64(0)
        codes.append(L.xspmm_bcsr_spmm_scratch(X.F16, 16, 16, 1, 1, 1, 0, 0, 8, 0, 0, None))
        codes.append(L.xspmm_bcsr_spmm_scratch(7, 16, 16, 1, 1, 1, 0, 0, 8, 0, 0, C.byref(out)))
        codes.append(L.xspmm_bcsr_spmm_scratch(X.F16, 17, 16, 1, 1, 1, 0, 0, 8, 0, 0, C.byref(out)))

    t = threading.Thread(target=calls)
    t.start()
    t.join()
    assert codes == [X.ERR_INVALID] * 3
