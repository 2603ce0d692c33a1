"""The sparse products that programs have this framework do, as timed cases.

A case is one call (or one fixed chain of calls) through the Python view of
the library on matrices made from a seed:

  tier1     C = A_bcsr * B, the blocks laid out once (csr_to_bcsr)
  prepared  SpMMPlan.execute: the Tier-2 pipeline's preparation done once
  pipeline  spmm_pipeline on a CSR matrix, every stage in the call
  staged    the Tier-2 stages called one by one: jaccard_clustering,
            apply_permutation, csr_to_bcsr, spmm, unpermute_dense_matrix

Matrix families (`pattern`) are the benchmark's and the tests': uniform
entries, rows from shared column templates, power-law graphs, whole 16x16
blocks, magnitude-pruned weights, bands, upper triangles.  `cluster` turns
the clustering stage on; for tier1, whose matrix is ready made, it means that
rows of one template lie together, as a clustering leaves them.
"""
import math

import torch

import xspmm_amd as X

DEVICE = "cuda:0"
_VALUES = {"f16": torch.float16, "f32": torch.float32}
_INDEX = {"i32": torch.int32, "i64": torch.int64}


def listed():
    return [
        # a small product inside a larger program (the CPU reference's shape):
        # launch and call latency are most of it
        _case("small_uniform", "tier1", "uniform", "f32", "i32", 1024, 1024, 64, density=0.01),
        # block-structured weights, every stored block full, a batch of 256
        _case("blocks", "tier1", "blocks", "f16", "i32", 8192, 8192, 256, density=0.05),
        # the headline product: row templates in an order the clustering cannot
        # mend, most blocks a column or two full
        _case("templates", "tier1", "templates", "f16", "i32", 16384, 16384, 128, density=0.005),
        # the reference's own value type and default index type, ragged edges,
        # rows in clustered order
        _case("clustered_wide_index", "tier1", "templates", "f32", "i64", 15001, 14999, 100, density=0.005, cluster=True),
        # feature propagation on a power-law graph
        _case("graph", "tier1", "graph", "f16", "i32", 131072, 131072, 64, density=16 / 131072),
        # a pruned projection layer over a long prompt (prefill)
        _case("pruned", "tier1", "pruned", "f16", "i32", 14336, 4096, 2048, density=0.1),
        # the same kind of layer in the reference's value type, a shorter prompt
        _case("pruned_f32", "tier1", "pruned", "f32", "i32", 4096, 4096, 512, density=0.1),
        # the middle of the reference's density sweep, in its value type
        _case("band", "tier1", "band", "f32", "i32", 16384, 16384, 128, density=0.5),
        # odd sizes everywhere: a graph-classifier head's 31 outputs
        _case("ragged", "tier1", "uniform", "f16", "i32", 5003, 4999, 31, density=0.02),
        # a solver or a server that multiplies one matrix again and again
        _case("prepared", "prepared", "templates", "f32", "i32", 16384, 16384, 128, density=0.005),
        # one call on a matrix seen for the first time, all defaults
        # (clustering on the host), the reference's Tier-2 sweep's shape
        _case("pipeline", "pipeline", "triangular", "f32", "i64", 8192, 8192, 256, density=0.01, cluster=True),
        # the same work stage by stage, clustering on the GPU
        _case("staged", "staged", "templates", "f16", "i32", 16384, 16384, 128, density=0.005, cluster=True),
    ]


def draw(rng):
    while True:
        case = _draw_once(rng)
        if _cost(case) <= 1.0:
            return case


def _draw_once(rng):
    kind = rng.choice(["tier1"] * 6 + ["prepared"] * 2 + ["pipeline"] * 2 + ["staged"])
    vt = rng.choice(["f16", "f32"])
    it = rng.choice(["i32", "i32", "i64"])
    N = _size(rng, 1, 512)
    if rng.random() < 0.5:
        N = max(8, N // 8 * 8)
    cluster = kind == "staged" or rng.random() < 0.4
    pattern = rng.choice(["uniform", "templates", "graph", "blocks", "pruned", "band", "triangular"])
    if kind == "tier1" and pattern != "templates":
        cluster = False
    if pattern == "graph":
        M = K = _size(rng, 4096, 24000 if cluster else 131072)
        density = rng.uniform(4, 20) / M
    elif pattern == "pruned":
        M, K = _size(rng, 512, 14336), _size(rng, 512, 8192)
        density = rng.uniform(0.06, 0.3)
        if kind == "tier1" and vt == "f16" and rng.random() < 0.5:
            N = _size(rng, 64, 2048)
    elif pattern == "band":
        M = K = _size(rng, 1024, 16384)
        density = math.exp(rng.uniform(math.log(0.002), math.log(0.8)))
    elif pattern == "blocks":
        M, K = _size(rng, 1024, 12000), _size(rng, 1024, 12000)
        density = rng.uniform(0.01, 0.1)
    else:
        M = _size(rng, 1024, 16384)
        K = M if pattern == "triangular" or rng.random() < 0.5 else _size(rng, 1024, 16384)
        density = math.exp(rng.uniform(math.log(0.003), math.log(0.02)))
    return _case(None, kind, pattern, vt, it, M, K, N, density=density, cluster=cluster)


def _size(rng, lo, hi):
    return round(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def _case(name, kind, pattern, values, index, M, K, N, density, cluster=False):
    case = dict(kind=kind, pattern=pattern, values=values, index=index, M=M, K=K, N=N,
                density=density, cluster=cluster)
    if name:
        case["name"] = name
    return case


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------

def _entries(case):
    """Expected CSR entries."""
    M, K, d = case["M"], case["K"], case["density"]
    if case["pattern"] == "band":
        w = _bandwidth(case)
        return M * (2 * w + 1) - w * (w + 1)
    if case["pattern"] == "triangular":
        return M * (M + 1) / 2 * d + M * (1 - d)
    return M * K * d


def _blocks(case):
    """Expected 16x16 blocks that hold an entry."""
    M, K, d = case["M"], case["K"], case["density"]
    Mb, Kb = -(-M // 16), -(-K // 16)
    if case["pattern"] == "blocks":
        return Mb * Kb * d
    if case["pattern"] == "band":
        w = -(-_bandwidth(case) // 16)
        return min(Mb * Kb, Mb * (2 * w + 1) - w * (w + 1))
    if case["pattern"] == "templates" and _grouped(case):
        columns = (1 + 16 * 0.3) * d * K
        return Mb * Kb * (1 - math.exp(-columns / Kb))
    share = 1 - (1 - d) ** 256
    return Mb * Kb * share * (0.5 if case["pattern"] == "triangular" else 1.0)


def _grouped(case):
    return case["kind"] == "tier1" and case["cluster"]


def _bandwidth(case):
    return max(1, int(case["density"] * case["M"] / 2))


def _cost(case):
    """A case's expense against the largest listed ones' (1: as large)."""
    f16 = case["values"] == "f16"
    block_bytes = _blocks(case) * (512 if f16 else 1024)
    padded = 512.0 * _blocks(case) * case["N"]
    cost = max(block_bytes / 1.0e9, padded / (2.4e11 if f16 else 3.2e10), _entries(case) / 9.0e7)
    if case["cluster"] and case["kind"] != "tier1":
        # host clustering inside the call, or the GPU's
        cost = max(cost, _entries(case) / (1.4e6 if case["kind"] == "staged" else 3.5e5))
    return cost


def work(case):
    st = 2 if case["values"] == "f16" else 4
    si = 4 if case["index"] == "i32" else 8
    M, K, N = case["M"], case["K"], case["N"]
    nnz, nnzb = _entries(case), _blocks(case)
    dense = K * N * st + M * N * 4
    csr = nnz * (st + si) + (M + 1) * si
    bcsr = nnzb * (256 * st + si) + (-(-M // 16) + 1) * si
    if case["kind"] == "tier1":
        moved = bcsr
    elif case["kind"] == "staged":
        moved = csr + bcsr + M * si
    else:
        moved = csr
    return {"bytes": float(moved + dense), "flops": 2.0 * nnz * N}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _keys(case, g):
    """Sorted distinct row * K + column of the entries, on the GPU."""
    M, K, d = case["M"], case["K"], case["density"]
    pattern = case["pattern"]
    ar = torch.arange
    if pattern == "band":
        w = _bandwidth(case)
        i = ar(M, device=DEVICE)
        lo, hi = (i - w).clamp(min=0), (i + w).clamp(max=K - 1)
        n = hi - lo + 1
        first = torch.cumsum(n, 0) - n
        return ar(int(n.sum()), device=DEVICE) + torch.repeat_interleave(i * K + lo - first, n)
    if pattern == "graph":
        # out-degrees from a Pareto law of exponent 2.1 cut at 4096, scaled
        # to the mean
        u = torch.rand(M, generator=g, device=DEVICE, dtype=torch.float64)
        top = min(4096, K // 4)
        x = (1 - u * (1 - float(top) ** -1.1)) ** (-1 / 1.1)
        deg = (x * (d * K / x.mean())).clamp(1, top).round().long()
        rows = torch.repeat_interleave(ar(M, device=DEVICE), deg)
        cols = torch.randint(K, rows.shape, generator=g, device=DEVICE)
        return torch.unique(rows * K + cols)
    if pattern == "templates":
        # 16 rows share a template of t columns; a row keeps 70 % of them
        # and draws the others anywhere; rows are in random order unless grouped
        t = max(2, round(d * K))
        kinds = max(1, M // 16)
        keep = max(1, round(0.7 * t))
        columns = torch.randint(K, (kinds, t), generator=g, device=DEVICE)
        i = ar(M, device=DEVICE)
        rows = i if _grouped(case) else torch.randperm(M, generator=g, device=DEVICE)
        pick = torch.rand((M, t), generator=g, device=DEVICE).topk(keep, dim=1).indices
        kept = torch.gather(columns[(i // 16) % kinds], 1, pick)
        others = torch.randint(K, (M, t - keep), generator=g, device=DEVICE)
        return torch.unique((rows[:, None] * K + torch.cat([kept, others], 1)).reshape(-1))
    if pattern == "blocks":
        Mb, Kb = -(-M // 16), -(-K // 16)
        b = torch.nonzero(torch.rand(Mb * Kb, generator=g, device=DEVICE) < d).reshape(-1)
        bi, bj = b // Kb, b % Kb
        i = (bi * 16)[:, None, None] + ar(16, device=DEVICE)[None, :, None]
        j = (bj * 16)[:, None, None] + ar(16, device=DEVICE)[None, None, :]
        keys = (i * K + j)[(i < M) & (j < K)]
        return torch.sort(keys).values
    # uniform, pruned, triangular: each entry on its own
    on = torch.rand((M, K), generator=g, device=DEVICE) < d
    if pattern == "triangular":
        on = torch.triu(on)
        on.fill_diagonal_(True)
    return torch.nonzero(on.reshape(-1)).reshape(-1)


def _csr(case, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    M, K = case["M"], case["K"]
    keys = _keys(case, g)
    ends = torch.arange(M + 1, device=DEVICE) * K
    row_ptr = torch.searchsorted(keys, ends)
    columns = keys % K
    if case["pattern"] == "graph":  # mean aggregation
        deg = torch.diff(row_ptr)
        values = torch.repeat_interleave(1.0 / deg.clamp(min=1).float(), deg)
    else:
        values = torch.randn(keys.numel(), generator=g, device=DEVICE)
        if case["pattern"] == "pruned":
            values *= 0.02
    it, vt = _INDEX[case["index"]], _VALUES[case["values"]]
    A = X.CSRMatrix(M, K, row_ptr.to(it), columns.to(it), values.to(vt))
    B = torch.randn((K, case["N"]), generator=g, device=DEVICE).to(vt)
    return A, B


def prepare(case, seed):
    A, B = _csr(case, seed)
    state = {"kind": case["kind"], "cluster": case["cluster"], "B": B}
    if case["kind"] == "tier1":
        state["A"] = X.csr_to_bcsr(A)
        state["C"] = torch.empty((case["M"], case["N"]), dtype=torch.float32, device=DEVICE)
    elif case["kind"] == "prepared":
        state["A"] = X.SpMMPlan(A, optimize_pattern=case["cluster"])
        state["C"] = torch.empty((case["M"], case["N"]), dtype=torch.float32, device=DEVICE)
    else:
        state["A"] = A
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(state):
    A, B = state["A"], state["B"]
    if state["kind"] == "tier1":
        return X.spmm(A, B, state["C"])
    if state["kind"] == "prepared":
        return A.execute(B, state["C"])
    if state["kind"] == "pipeline":
        return X.spmm_pipeline(A, B, optimize_pattern=state["cluster"], timings=False)[0]
    perm = X.jaccard_clustering(A)
    blocks = X.csr_to_bcsr(X.apply_permutation(A, perm))
    C = X.unpermute_dense_matrix(X.spmm(blocks, B), perm)
    return perm, blocks.row_ptr, C


def tolerance(case):
    # fp32 sums of exact (fp16) or once-rounded (fp32) products: rounding
    # grows with the length of a sum, up to 16384 terms here (measured against
    # exact: 2e-8 to 8e-7).  Permutations and block counts stay exact.
    return {"rel": 4e-6}


def exact(case, seed):
    A, B = _csr(case, seed)
    M, K, N = case["M"], case["K"], case["N"]
    B64 = B.double()
    C = torch.empty((M, N), dtype=torch.float64, device=DEVICE)
    step = max(1, (1 << 27) // K)
    row_ptr = A.row_ptr.long()
    for r0 in range(0, M, step):
        r1 = min(M, r0 + step)
        e0, e1 = int(row_ptr[r0]), int(row_ptr[r1])
        rows = torch.repeat_interleave(torch.arange(r1 - r0, device=DEVICE),
                                       torch.diff(row_ptr[r0:r1 + 1]))
        dense = torch.zeros((r1 - r0, K), dtype=torch.float64, device=DEVICE)
        dense[rows, A.col_ind[e0:e1].long()] = A.values[e0:e1].double()
        C[r0:r1] = dense @ B64
    return [None, None, C] if case["kind"] == "staged" else C

