"""Prunes against the oracle row by row: a node's row may differ only where a product of two of its neighbours ties with one of their norms,
so a bound that is wrong for a few pairs is seen. On the corpora of the bound kernel's test and on ones whose terms draw the Gram tiles' lines."""
import numpy as np
import pytest

import test_gpu_prune_bounds as bounds

pytestmark = pytest.mark.gpu
N = bounds.N


def make(kind, wide):
    if kind not in ("few shared", "few terms"):
        return bounds.make(kind, wide)
    rng = np.random.default_rng(5)
    a = list(bounds.make("pairs decide", False))
    if kind == "few shared":  # eight rows of a Gram tile fit the whole LDS, not half of it
        cnt = rng.integers(140, 180, N)
        off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.uint32)
        idx = np.concatenate([np.sort(rng.choice(30000, c, replace=False)) for c in cnt]).astype(np.uint32)
        a[1:4] = off, idx, rng.uniform(1.0, 8.0, len(idx)).astype(np.float32)
    elif kind == "few terms":  # as "few shared", in the wide format too: eight rows share their terms with each other, and few terms a bit of the table
        cnt = rng.integers(280, 320, N)
        off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.uint32)
        idx = np.concatenate([np.sort(rng.choice(2000, c, replace=False)) for c in cnt]).astype(np.uint32)
        a[1:4] = off, idx, rng.uniform(1.0, 4.0, len(idx)).astype(np.float32)
    if wide:
        a[5] = a[5] + np.uint32(70000)
    return tuple(a)


def equal_but_for_ties(arrays, scale, ids, dist, got, want):
    """All outputs of every node, but for nodes with a pair of neighbours whose product lies within the rounding of an fp32 sum of one
    of their norms (1e-5 of what the parts of either can reach, as the kernels' own room); few nodes at most."""
    import apoe
    from scipy.sparse import csr_matrix
    differ = np.flatnonzero(~np.logical_and.reduce([(g == w).reshape(len(ids), -1).all(axis=1) for g, w in zip(got, want)]))
    dense, *pairs = arrays
    for u in differ:
        near = ids[u][(dist[u] < apoe.INF_DIS) & (ids[u] != u)]
        d = dense[near].astype(np.float64) * scale
        prod, reach = d @ d.T, np.outer(*2 * [np.linalg.norm(d, axis=1)])
        with np.errstate(invalid="ignore"):
            sq = 0.0
            for off, idx, val in (pairs[:3], pairs[3:]):
                m = csr_matrix((val.astype(np.float64), idx.astype(np.int64), off.astype(np.int64)), (len(dense), int(idx.max()) + 1))[near]
                prod = prod + (m @ m.T).toarray()
                sq = sq + np.asarray(m.multiply(m).sum(axis=1)).ravel()
            reach = reach + np.sqrt(np.outer(sq, sq)) + 1.0
            tie = np.abs(prod - np.diag(prod)) <= 1e-5 * reach
        assert (tie & ~np.eye(len(near), dtype=bool)).any(), (u, [(g[u], w[u]) for g, w in zip(got, want)])
    assert len(differ) <= 0.005 * len(ids), differ


def check(gpu_ctx, kind, K, degree, wide, without=0):
    import apoe
    import oracle as O
    arrays = make(kind, wide)
    C = O.HybridSet(*arrays)
    ids, dist = O.bruteforce_knn_self(C, 7.0, K)
    counts = [c for c in (0, 1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 96, 113, 127) if c < K]
    for i, u in enumerate(np.random.default_rng(6).choice(N, 6 * len(counts), replace=False)):
        dist[u, counts[i % len(counts)]:] = apoe.INF_DIS
    gc = apoe.Corpus(gpu_ctx, *arrays, without=without)
    knn = apoe.Knn(gpu_ctx, gc, K, 7.0)
    knn.upload(ids, dist)
    knn.prune(degree)
    g_fwd, g_det, g_cnt, g_kw = knn.prune_download()
    knn.close()
    gc.close()
    c_fwd, c_det, c_cnt, c_kw = O.prune(C, 7.0, O.norms(C, 7.0), ids, dist, degree)
    equal_but_for_ties(arrays, 7.0, ids, dist, (g_fwd, g_det, g_cnt, g_kw), (c_fwd, c_det, c_cnt, c_kw))
    if kind == "near twins":
        assert np.any(c_cnt < min(degree, K - 1))  # the rule does reject here


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("K,degree", [(64, 32), (64, 64), (128, 48)])
@pytest.mark.parametrize("kind", ["bounds settle", "pairs decide", "near twins", "rich rows", "few shared", "few terms", "odd rows"])
def test_rows_differ_at_ties_only(gpu_ctx, kind, K, degree, wide):
    check(gpu_ctx, kind, K, degree, wide)
