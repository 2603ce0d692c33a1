"""Prepared products against the pipeline, bit for bit, where the plan multiplies a
padded copy of B or stores into a C off 16 bytes: real-valued operands, so that
another kernel's order of sums would show."""
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


def csr(torch, M, K, keys, dtype):
    rp = torch.searchsorted(keys, torch.arange(M + 1, device="cuda:0") * K)
    vals = torch.randn(keys.numel(), device="cuda:0").to(dtype)
    return X.CSRMatrix(M, K, rp.int(), (keys % K).int(), vals)


def full_blocks(torch, M, K, share):
    Mb, Kb = M // 16, K // 16
    b = (torch.rand(Mb * Kb, device="cuda:0") < share).nonzero().reshape(-1)
    r = torch.arange(16, device="cuda:0")
    keys = ((b // Kb * 16)[:, None, None] + r[None, :, None]) * K + (b % Kb * 16)[:, None, None] + r[None, None, :]
    return keys.reshape(-1).sort().values


@pytest.mark.parametrize("N", [64, 200])
def test_f32_clustered_plan_with_c_off_16_bytes(torch, N):
    """Blocks that the packed form would not shrink: the plan's product goes through
    its workspace, as the pipeline's does, and keeps its kernel."""
    M = K = 9216
    A = csr(torch, M, K, full_blocks(torch, M, K, 0.02), torch.float32)
    plan = X.SpMMPlan(A, optimize_pattern=True)
    assert plan.packed_batches == -1
    B = torch.randn((K, N), device="cuda:0")
    want = X.spmm_pipeline(A, B, optimize_pattern=True)[0]
    for off in (0, 1, 2):
        guard = torch.full((M * N + 8,), -7.0, device="cuda:0")
        C = plan.execute(B, guard[off:off + M * N].view(M, N))
        assert torch.equal(C, want), off
        assert bool((guard[off + M * N:] == -7.0).all())


@pytest.mark.parametrize("cluster", [False, True])
@pytest.mark.parametrize("M,K,per_row,columns", [(4099, 5003, 48, (129, 257, 260, 391)), (20000, 20000, 12, (3, 67, 127))])
def test_packed_f16_plan_on_padded_b_equals_the_pipeline(torch, monkeypatch, M, K, per_row, columns, cluster):
    """fp16, N % 8 != 0, on both sides of the line from which a plan multiplies its
    packed batches on the padded copy (3 * 2^16 products of a block with 128
    columns: 73 thousand blocks from N = 257, 222 thousand from N = 1): the
    pipeline's C and that of a plan without packed batches."""
    keys = torch.unique((torch.arange(M, device="cuda:0")[:, None] * K +
                         torch.randint(K, (M, per_row), device="cuda:0")).reshape(-1))
    A = csr(torch, M, K, keys, torch.float16)
    packed = X.SpMMPlan(A, optimize_pattern=cluster)
    monkeypatch.setenv("XSPMM_PLAN_PACK", "off")
    plain = X.SpMMPlan(A, optimize_pattern=cluster)
    monkeypatch.delenv("XSPMM_PLAN_PACK")
    assert packed.packed_batches > 0 and plain.packed_batches == -1
    for N in columns:
        print(M, cluster, N, packed.num_blocks, flush=True)
        B = torch.randn((K, N), device="cuda:0").half()
        C = packed.execute(B)
        assert torch.equal(C, plain.execute(B)), N
        assert torch.equal(C, X.spmm_pipeline(A, B, optimize_pattern=cluster)[0]), N


@pytest.mark.parametrize("cluster", [False, True])
@pytest.mark.parametrize("values,M,K,per_row,N", [
    ("f32", 4099, 5003, 48, 67), ("f32", 4099, 5003, 48, 5), ("f16", 4099, 5003, 48, 31), ("f16", 4099, 5003, 48, 257),
    ("f16", 515, 97, 0, 8), ("f16", 515, 97, 0, 33), ("f32", 2050, 1601, 0, 257), ("f16", 17000, 300, 2, 129)])
def test_execute_allocates_nothing_again(torch, values, M, K, per_row, N, cluster):
    """The second product of N columns takes nothing from the library's pool, and can
    be captured (which refuses hipMalloc): each replay gives the eager C."""
    import ctypes as C
    hip, pool = C.CDLL("libamdhip64.so.7"), C.c_void_p()
    assert hip.hipDeviceGetDefaultMemPool(C.byref(pool), torch.cuda.current_device()) == 0
    used, high, zero = C.c_uint64(0), C.c_uint64(0), C.c_uint64(0)
    cols = (torch.randint(K, (M, per_row), device="cuda:0") if per_row else
            (torch.arange(0, K, 16, device="cuda:0") + torch.arange(M, device="cuda:0")[:, None] % 16).clamp(max=K - 1))
    keys = torch.unique((torch.arange(M, device="cuda:0")[:, None] * K + cols).reshape(-1))
    dtype = torch.float16 if values == "f16" else torch.float32
    plan = X.SpMMPlan(csr(torch, M, K, keys, dtype), optimize_pattern=cluster)
    B = torch.randn((K, N), device="cuda:0").to(dtype)
    want, out = plan.execute(B), torch.empty((M, N), device="cuda:0")
    torch.cuda.synchronize()
    assert hip.hipMemPoolGetAttribute(pool, 0x7, C.byref(used)) == 0  # hipMemPoolAttrUsedMemCurrent
    assert hip.hipMemPoolSetAttribute(pool, 0x8, C.byref(zero)) == 0  # hipMemPoolAttrUsedMemHigh
    plan.execute(B, out)
    torch.cuda.synchronize()
    assert hip.hipMemPoolGetAttribute(pool, 0x8, C.byref(high)) == 0
    assert high.value <= used.value
    assert torch.equal(out, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.execute(B, out)
    for i in range(3):
        B.mul_(-1)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, plan.execute(B)), i
