"""The ways the prune answers its question about two neighbours of a node (does their product exceed either one's norm?): bounds alone, the
sparse products of the terms that two rows share, the rank table for rows that keep too many of those, dense products where the bounds stay
open. Rows, detour counts and keyword candidates are the oracle's whichever it is, on full, short and ragged lists."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N = 1200


def make(kind, wide):
    import apoe_synth as S
    rng = np.random.default_rng(5)
    a = list(S.to_numpy((S.corpus if kind == "pairs decide" else S.latent_corpus)(N, seed=21, device="cpu")))
    if kind == "near twins":  # copies of documents, a little longer or shorter: products within the sketch's error of a norm, and clear of it
        half = N // 2
        dense, s_off, s_idx, s_val, b_off, b_idx, b_val = a
        longer = rng.choice([0.9, 0.99, 1.01, 1.05], half).astype(np.float32)[:, None]
        twice = lambda off, x: (np.concatenate([off[:half + 1], off[half] + off[1:half + 1]]).astype(np.uint32), np.concatenate([x[:off[half]]] * 2))
        a = [np.concatenate([dense[:half], dense[:half] * longer])]
        for off, idx, val in ((s_off, s_idx, s_val), (b_off, b_idx, b_val)):
            a += [twice(off, idx)[0], twice(off, idx)[1], twice(off, val)[1]]
    elif kind == "rich rows":  # more pairs than a wave keeps in registers, most of them shared
        cnt = rng.integers(200, 420, N)
        off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.uint32)
        idx = np.concatenate([np.sort(rng.choice(600, c, replace=False)) for c in cnt]).astype(np.uint32)
        a[1:4] = off, idx, rng.uniform(0.1, 0.4, len(idx)).astype(np.float32)
    elif kind == "odd rows":  # no dense part, no terms, far magnitudes
        a[0] = a[0] * rng.choice([0.0, 1e-3, 1.0, 1.0, 30.0], N).astype(np.float32)[:, None]
        keep = rng.random(N) < 0.8
        for o in (1, 4):
            cnt = np.diff(a[o].astype(np.int64))
            sel = np.repeat(keep, cnt)
            a[o], a[o + 1], a[o + 2] = np.concatenate([[0], np.cumsum(cnt * keep)]).astype(np.uint32), a[o + 1][sel], a[o + 2][sel]
    if wide:
        a[5] = a[5] + np.uint32(70000)
    return tuple(a)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("K,degree", [(64, 32), (64, 64), (128, 48)])
@pytest.mark.parametrize("kind", ["bounds settle", "pairs decide", "near twins", "rich rows", "odd rows"])
def test_prune_matches_oracle(gpu_ctx, kind, K, degree, wide):
    import apoe
    import oracle as O
    arrays = make(kind, wide)
    C = O.HybridSet(*arrays)
    ids, dist = O.bruteforce_knn_self(C, 7.0, K)
    counts = [c for c in (0, 1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 96, 113, 127) if c < K]
    for i, u in enumerate(np.random.default_rng(6).choice(N, 6 * len(counts), replace=False)):
        dist[u, counts[i % len(counts)]:] = apoe.INF_DIS
    gc = apoe.Corpus(gpu_ctx, *arrays)
    knn = apoe.Knn(gpu_ctx, gc, K, 7.0)
    knn.upload(ids, dist)
    knn.prune(degree)
    g_fwd, g_det, g_cnt, g_kw = knn.prune_download()
    knn.close()
    gc.close()
    c_fwd, c_det, c_cnt, c_kw = O.prune(C, 7.0, O.norms(C, 7.0), ids, dist, degree)
    same = np.all(g_fwd == c_fwd, axis=1)
    assert same.mean() >= 0.995, np.flatnonzero(~same)[:10]  # a product that rounds to either side of a norm
    assert np.array_equal(g_det[same], c_det[same]) and np.array_equal(g_cnt[same], c_cnt[same])
    assert np.all(g_kw == c_kw, axis=1)[same].mean() >= 0.995
    if kind == "near twins":
        assert np.any(c_cnt < min(degree, K - 1))  # the rule does reject here
