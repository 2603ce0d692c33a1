"""The GPU clustering kernel on either side of the sizes that decide where it
keeps its loop state (LDS up to about 12100 rows, memory above) and how it
tests and commits (words in registers up to 16 bitmap words, one wave up to 64,
the workgroup above): the same
permutation as the host engine, for both engines.
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


def rows_like_templates(M, K, seed):
    """Rows of 10 entries: 8 or 9 of a template's (eight rows to a template) and
    the rest anywhere, rows in random order, some empty, some single."""
    rng = np.random.default_rng(seed)
    tmpl = rng.integers(0, K, size=(max(1, M // 8), 10))
    rows = []
    for r in rng.permutation(M):
        u = rng.random()
        if u < 0.02:
            c = np.zeros(0, np.int64)
        elif u < 0.05:
            c = rng.integers(0, K, size=1)
        else:
            c = tmpl[r % len(tmpl)].copy()
            k = int(rng.integers(0, 3))
            c[:k] = rng.integers(0, K, size=k)
        rows.append(np.unique(c))
    rp = np.zeros(M + 1, np.int32)
    np.cumsum([len(c) for c in rows], out=rp[1:])
    return rp, np.concatenate(rows).astype(np.int32)


@pytest.mark.parametrize("itype", [np.int32, np.int64])
@pytest.mark.parametrize("engine", ["scan", "index"])
@pytest.mark.parametrize("M,K", [(1, 40), (2, 1), (1023, 700), (1025, 5000), (12050, 1000), (12200, 1000),
                                 (5000, 16384), (5000, 16385),
                                 (3000, 73600), (11000, 16384 * 16), (13000, 73600)])
def test_same_permutation_as_the_host(torch, M, K, engine, itype, monkeypatch):
    rp, ci = rows_like_templates(M, K, seed=M + K)
    rp, ci = rp.astype(itype), ci.astype(itype)
    print(M, K, engine, itype.__name__, flush=True)
    want = X.compute_1d_jaccard_clustering(M, K, rp, ci)
    monkeypatch.setenv("XSPMM_CLUSTER_ENGINE", engine)
    A = X.CSRMatrix.from_host(M, K, rp, ci, np.ones(len(ci), np.float32), device="cuda:0")
    for thr in (0.5, 0.2):
        if thr != 0.5:
            want = X.compute_1d_jaccard_clustering(M, K, rp, ci, dist_thresh=thr)
        perm, used = X.jaccard_clustering(A, thr, 16, return_engine=True)
        assert used == engine
        assert np.array_equal(perm.cpu().numpy(), want)
