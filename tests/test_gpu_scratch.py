"""Where Tier-1's temporaries come from: the Python view hands the library scratch
of the bytes that the product uses, so nothing is allocated that no kernel reads
and nothing comes from the library's pool; without memory for a padded copy of B
the product takes a kernel that needs none."""
from __future__ import annotations

import ctypes as C

import pytest

import xspmm_amd as X

pytestmark = pytest.mark.gpu

USED, HIGH = 0x7, 0x8  # hipMemPoolAttrUsedMemCurrent, hipMemPoolAttrUsedMemHigh


@pytest.fixture(scope="module")
def torch():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need an MI355X (torch.cuda.is_available() is False)")
    X.load()
    return torch


@pytest.fixture(scope="module")
def hip(torch):
    return C.CDLL("libamdhip64.so.7")


def matrix(torch, M, K, per_row, dtype):
    """per_row integer-valued entries anywhere in each row; 0: one in every block."""
    g = torch.Generator(device="cuda:0")
    g.manual_seed(M + K)
    if per_row == 0:
        cols = torch.arange(0, K, 16, device="cuda:0") + torch.arange(M, device="cuda:0")[:, None] % 16
        cols = cols.clamp(max=K - 1)
    else:
        cols = torch.randint(K, (M, per_row), generator=g, device="cuda:0")
    keys = torch.unique((torch.arange(M, device="cuda:0")[:, None] * K + cols).reshape(-1))
    rp = torch.searchsorted(keys, torch.arange(M + 1, device="cuda:0") * K)
    vals = torch.randint(1, 5, keys.shape, generator=g, device="cuda:0").to(dtype)
    D = torch.zeros(M * K, device="cuda:0")
    D[keys] = vals.float()
    return X.csr_to_bcsr(X.CSRMatrix(M, K, rp.int(), (keys % K).int(), vals)), D.view(M, K)


def operands(torch, K, N, dtype):
    return (torch.arange(K * N, device="cuda:0") % 13 - 6).view(K, N).to(dtype)


def pool_attribute(hip, torch, attr, set_zero=False):
    pool, v = C.c_void_p(), C.c_uint64(0)
    assert hip.hipDeviceGetDefaultMemPool(C.byref(pool), torch.cuda.current_device()) == 0
    fn = hip.hipMemPoolSetAttribute if set_zero else hip.hipMemPoolGetAttribute
    assert fn(pool, attr, C.byref(v)) == 0
    return v.value


# (values, per_row, N, whether the product takes scratch)
@pytest.mark.parametrize("values,M,K,per_row,N,takes", [
    ("f32", 5003, 4999, 48, 3, False), ("f32", 5003, 4999, 48, 13, False), ("f32", 515, 4999, 8, 33, False),
    ("f32", 5003, 4999, 48, 67, True), ("f16", 5003, 4999, 48, 31, True), ("f16", 515, 1601, 0, 8, True),
    ("f16", 5003, 4999, 48, 64, False), ("f32", 40000, 999, 3, 5, False), ("f16", 40000, 999, 3, 5, True)])
def test_scratch_is_what_the_product_uses(torch, hip, values, M, K, per_row, N, takes):
    dtype = torch.float16 if values == "f16" else torch.float32
    A, D = matrix(torch, M, K, per_row, dtype)
    B = operands(torch, K, N, dtype)
    out = torch.empty((M, N), device="cuda:0")
    X.spmm(A, B, out)
    torch.cuda.synchronize()
    base = pool_attribute(hip, torch, USED)
    pool_attribute(hip, torch, HIGH, set_zero=True)
    torch.cuda.reset_peak_memory_stats()
    held = torch.cuda.memory_allocated()
    X.spmm(A, B, out)
    torch.cuda.synchronize()
    assert (torch.cuda.max_memory_allocated() > held) is takes
    assert pool_attribute(hip, torch, HIGH) <= base
    assert torch.equal(out, D @ B.float())


@pytest.mark.parametrize("values,N", [("f32", 67), ("f16", 31)])
def test_torch_out_of_memory(torch, monkeypatch, values, N):
    """No memory for the scratch in torch's allocator: the library's own serves."""
    dtype = torch.float16 if values == "f16" else torch.float32
    A, D = matrix(torch, 5003, 4999, 48, dtype)
    B = operands(torch, 4999, N, dtype)
    out = torch.empty((5003, N), device="cuda:0")
    empty, refused = torch.empty, []

    def without(*args, **kw):
        if kw.get("dtype") is torch.uint8:
            refused.append(args)
            raise torch.OutOfMemoryError("no memory")
        return empty(*args, **kw)

    monkeypatch.setattr(torch, "empty", without)
    X.spmm(A, B, out)
    monkeypatch.undo()
    assert refused
    assert torch.equal(out, D @ B.float())


class _Location(C.Structure):
    _fields_ = [("type", C.c_int), ("id", C.c_int)]


class _PoolProps(C.Structure):  # hipMemPoolProps
    _fields_ = [("alloc", C.c_int), ("handles", C.c_int), ("location", _Location), ("security", C.c_void_p),
                ("max_size", C.c_size_t), ("reserved", C.c_ubyte * 56)]


@pytest.mark.parametrize("N", [67, 301])
def test_f32_without_memory_for_a_copy(torch, hip, monkeypatch, N):
    """A pool of 256 KB (hipMemPoolProps.maxSize) and no scratch: the tile kernel,
    which reads B itself, makes the product, as the tile kernel forced does."""
    A, D = matrix(torch, 5003, 4999, 48, torch.float32)
    B = operands(torch, 4999, N, torch.float32)
    out = torch.full((5003, N), -7.0, device="cuda:0")
    X.spmm(A, B, out)
    assert torch.equal(out, D @ B)
    R = torch.randn((4999, N), device="cuda:0")
    monkeypatch.setenv("XSPMM_F32_KERNEL", "tile")
    want = X.spmm(A, R)
    monkeypatch.delenv("XSPMM_F32_KERNEL")
    dev = torch.cuda.current_device()
    before, small = C.c_void_p(), C.c_void_p()
    assert hip.hipDeviceGetMemPool(C.byref(before), dev) == 0
    assert hip.hipMemPoolCreate(C.byref(small), C.byref(_PoolProps(1, 0, _Location(1, dev), None, 1 << 18))) == 0
    empty = torch.empty

    def without(*args, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no memory")
        return empty(*args, **kw)

    assert hip.hipDeviceSetMemPool(dev, small) == 0
    try:
        monkeypatch.setattr(torch, "empty", without)
        X.spmm(A, R, out)
        torch.cuda.synchronize()
    finally:
        monkeypatch.undo()
        assert hip.hipDeviceSetMemPool(dev, before) == 0
        assert hip.hipMemPoolDestroy(small) == 0
    assert torch.equal(out, want)
    assert not torch.equal(out, X.spmm(A, R))  # the batches, with memory again
