"""The 8-bit sketch of the dense rows only ever rejects what its 4 KB row would reject: whole rows of results are bit for bit
those of a walk that reads every row (variant 0x100), on rows where a wrong bound would show: magnitudes from denormal to
beyond half precision, one-hot rows, zero rows, entries that are no numbers, and weights that make the dense part decide."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N, D, NQ = 3000, 32, 40


def world(kind, seed, wide):
    rng = np.random.default_rng(seed)
    centre = rng.standard_normal((8, 1024))
    dense = (centre[rng.integers(0, 8, N)] + rng.standard_normal((N, 1024))).astype(np.float32)
    q = (centre[rng.integers(0, 8, NQ)] + rng.standard_normal((NQ, 1024))).astype(np.float32)
    if kind == "magnitudes":
        dense *= (10.0 ** rng.choice([-40, -33, -20, -3, 0, 0, 0, 1, 3, 4], N)).astype(np.float32)[:, None]
        dense[::97] = 0
        q[::7] *= np.float32(1e-36)
        q[1] = 0
    elif kind == "spikes":  # one entry far above the rest: a coarse scale, a large error
        dense[np.arange(N), rng.integers(0, 1024, N)] *= rng.choice([1, 10, 1000], N).astype(np.float32)
        dense[::50] = np.eye(1024, dtype=np.float32)[rng.integers(0, 1024, len(dense[::50]))]
        q[np.arange(NQ), rng.integers(0, 1024, NQ)] *= 100
    elif kind == "not numbers":
        dense[5::200, 3] = np.inf
        dense[7::200, 900] = np.nan
        dense[9::200, 12] = 7e4
    idx = (rng.integers(0, 300, (N, 12)).cumsum(1) % 60000).astype(np.uint32) + np.uint32(70000 if wide else 0)
    off = np.arange(0, 12 * N + 1, 12, dtype=np.uint32)
    q_off = np.arange(0, 12 * NQ + 1, 12, dtype=np.uint32)
    corpus = (dense, off, idx.reshape(-1), rng.random(12 * N).astype(np.float32), off, idx[::-1].reshape(-1).copy(), rng.random(12 * N).astype(np.float32))
    queries = (q, q_off, idx[:NQ].reshape(-1).copy(), rng.random(12 * NQ).astype(np.float32), q_off, idx[-NQ:].reshape(-1).copy(), rng.random(12 * NQ).astype(np.float32))
    rows = np.zeros((N, D + 8), np.uint32)
    rows[:, :D] = rng.integers(0, N, (N, D))
    return corpus, queries, rows, rng.choice(N, D, replace=False).astype(np.uint32)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("kind", ["plain", "magnitudes", "spikes", "not numbers"])
def test_rows_are_those_of_reading_every_dense_row(gpu_ctx, kind, wide):
    import apoe
    corpus, queries, rows, entry = world(kind, 6, wide)
    gc, gq, gg = apoe.Corpus(gpu_ctx, *corpus), apoe.Queries(gpu_ctx, *queries), apoe.Graph(gpu_ctx, rows, entry)
    for w3, cands, shape in (((1, 0, 0), 24, 0), ((49, 1, 1), 64, 4), ((0.01, 1, 1), 33, 3), ((1, 1, 0), 200, 2)):
        a, ad, sa = apoe.search(gpu_ctx, gc, gq, gg, w3, cands, variant=shape)
        b, bd, sb = apoe.search(gpu_ctx, gc, gq, gg, w3, cands, variant=shape | 0x100)
        assert np.array_equal(a, b) and np.array_equal(ad, bd, equal_nan=True), (w3, cands)
        assert sa.evaluations == sb.evaluations and sa.dense_rows <= sb.dense_rows == sb.evaluations
        if kind == "plain" and w3 == (1, 0, 0):
            # the sketch is in use: without pairs nothing else settles an evaluation, and a row that it settles is not read
            assert sa.dense_rows < 0.6 * sb.dense_rows
            read = sb.algo_bytes - sa.algo_bytes - 4096 * (sb.dense_rows - sa.dense_rows)
            assert read <= 0 and read % (1024 + 8) == 0  # what it costs: a sketch with its scale and error each


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("kind", ["plain", "magnitudes", "spikes", "not numbers"])
def test_knowledge_graph_and_keyword_search(gpu_ctx, kind, wide):
    """The bound with the bonus of a linking entity in it, and the walk that keeps hits pushed out of the pool: whole rows bit for bit
    those of reading every dense row, under weights where the sketch settles evaluations."""
    import apoe
    import apoe_synth as S
    corpus, queries, rows, entry = world(kind, 7, wide)
    b_idx = queries[5].copy()
    b_idx[::12] |= np.uint32(0x80000000)  # the first BM25 term of every query is required
    gc, gq, gg = apoe.Corpus(gpu_ctx, *corpus), apoe.Queries(gpu_ctx, *queries), apoe.Graph(gpu_ctx, rows, entry)
    gk = apoe.Queries(gpu_ctx, *queries[:5], b_idx, queries[6])
    kg = apoe.KnowledgeGraph(gpu_ctx, *S.to_numpy(S.knowledge_graph(800, N, NQ, seed=23, device="cpu", mean_out=6.0)))
    for w3, cands, shape in (((1, 0, 0), 24, 0), ((49, 1, 1), 64, 4), ((49, 1, 1), 300, 2), ((0.01, 1, 1), 33, 3), ((1, 1, 0), 200, 1)):
        calls = [dict(queries=gq, kg=kg, kg_weight=weight) for weight in (0.5, 40.0, 400.0)] + [dict(queries=gk, keyword_filter=True)]
        for c in calls:
            q = c.pop("queries")
            a, ad, sa = apoe.search(gpu_ctx, gc, q, gg, w3, cands, variant=shape, **c)
            b, bd, sb = apoe.search(gpu_ctx, gc, q, gg, w3, cands, variant=shape | 0x100, **c)
            assert np.array_equal(a, b) and np.array_equal(ad, bd, equal_nan=True), (w3, cands, c)
            assert sa.evaluations == sb.evaluations and sa.dense_rows <= sb.dense_rows == sb.evaluations
            if kind == "plain" and w3 == (49, 1, 1) and cands == 64:
                assert sa.dense_rows < 0.6 * sb.dense_rows
                assert sa.algo_bytes + 4096 * (sb.dense_rows - sa.dense_rows) > sb.algo_bytes + 1032 * 0.3 * sb.evaluations # by sketches, not by the norm bound


@pytest.mark.parametrize("kind", ["plain", "magnitudes", "spikes"])
def test_half_precision_walk(gpu_ctx, kind):
    """The walk on half-precision rows under the sketch against the same walk without any bound."""
    import apoe
    corpus, queries, rows, entry = world(kind, 8, False)
    gc, gq, gg = apoe.Corpus(gpu_ctx, *corpus), apoe.Queries(gpu_ctx, *queries), apoe.Graph(gpu_ctx, rows, entry)
    gc.make_half_rows()
    for w3 in ((1, 0, 0), (49, 1, 1)):
        a, ad, _ = apoe.search(gpu_ctx, gc, gq, gg, w3, 48, variant=0x200)
        b, bd, _ = apoe.search(gpu_ctx, gc, gq, gg, w3, 48, variant=0x300)
        assert np.array_equal(a, b) and np.array_equal(ad, bd)


@pytest.mark.parametrize("K,mode", [(64, 1), (64, 2), (128, 1)])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("kind", ["plain", "spikes"])
def test_join_step_from_settled_lists(gpu_ctx, kind, wide, K, mode):
    """Uploaded lists count as settled: a join step asks the sketches which columns of a tile it can leave out. From the exact lists with
    three entries in ten replaced by random documents, a step's lists hold the oracle's distances, row for row."""
    import apoe
    import oracle as O
    corpus, _, _, _ = world(kind, 6, wide)
    dense = corpus[0] / np.linalg.norm(corpus[0], axis=1, keepdims=True) * np.random.default_rng(8).uniform(0.5, 2.0, (N, 1)).astype(np.float32)
    dense[::97] = 0
    idx = np.random.default_rng(9).integers(1, 300, (N, 12)).cumsum(1).astype(np.uint32) + np.uint32(70000 if wide else 0)  # no term twice in a row
    corpus = (dense.astype(np.float32), corpus[1], idx.reshape(-1), corpus[3], corpus[4], idx[::-1].reshape(-1).copy(), corpus[6])
    C = O.HybridSet(*corpus)
    rng = np.random.default_rng(K)
    ids, _ = O.bruteforce_knn_self(C, 7.0, K)
    some = rng.random(ids.shape) < 0.3
    ids[some] = rng.integers(0, N, int(some.sum()))
    dist = O.distance_pairs(C, 7.0, np.repeat(np.arange(N, dtype=np.uint32), K), ids.reshape(-1)).reshape(N, K)
    order = np.argsort(dist, 1, kind="stable")
    ids, dist = np.take_along_axis(ids, order, 1), np.take_along_axis(dist, order, 1)
    st = O.nnd_init(N, K, 1)  # its reverse lists are empty
    st.ids[:], st.dist[:] = ids, dist
    gc = apoe.Corpus(gpu_ctx, *corpus)
    knn = apoe.Knn(gpu_ctx, gc, K, 7.0)
    knn.upload(ids, dist)
    knn.set_join(mode)
    ins = knn.iterate(last=True)
    oins, _ = O.join_iterate(C, 7.0, st, slots=2 * K, symmetric=mode == 2)
    got, gd = knn.download()
    assert 0 < ins and abs(ins - oins) <= 0.002 * oins + 2
    # a list that lost an entry differs from there on by the gap between two entries, about a hundredth of its range of 50; a different
    # order of the float sums moves a distance by at most 1024 x 2^-24 = 6e-5 of it, and may swap neighbours
    scale = np.maximum(1.0, np.abs(st.dist))
    same = np.all(np.abs(gd - st.dist) <= 6e-5 * scale, axis=1)
    assert same.mean() >= 0.999, np.flatnonzero(~same)[:10]
    assert np.mean(got == (st.ids & 0x7FFFFFFF)) >= 0.99
    knn.close()
    gc.close()
