"""The byte codes of a record's values only ever reject what the pairs themselves would reject: whole rows of results are bit for bit
those of a walk without any bound (variant 0x100), on values where a wrong bound would show: magnitudes from denormal to 1e30, negative
ones, values that are no numbers, rows without pairs, of one path and longer than a wave's loads, in each mode that asks the codes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N, D, NQ, VOCAB = 3000, 32, 40, 400


def rows_of(rng, n, lengths, kind):
    off = np.zeros(n + 1, np.uint32)
    off[1:] = np.cumsum(rng.choice(lengths, n))
    idx = np.concatenate([rng.choice(VOCAB, off[i + 1] - off[i], replace=False) for i in range(n)]).astype(np.uint32) * 163
    val = rng.gamma(1.0, 1.0, len(idx)).astype(np.float32)
    if kind == "magnitudes":
        val *= (10.0 ** rng.choice([-44, -38, -30, -9, 0, 0, 0, 2, 8], len(val))).astype(np.float32)
    elif kind == "negative":
        val *= rng.choice([-1, 1, 1], len(val)).astype(np.float32)
    elif kind == "not numbers":
        val[::997] = np.inf
        val[5::997] = np.nan
    return off, idx, val


def world(kind, seed):
    rng = np.random.default_rng(seed)
    dense = rng.standard_normal((N, 1024)).astype(np.float32) * np.float32(0.1)
    q = rng.standard_normal((NQ, 1024)).astype(np.float32) * np.float32(0.1)
    corpus = (dense, *rows_of(rng, N, [0, 1, 63, 64, 65, 130, 250], kind), *rows_of(rng, N, [0, 1, 31, 64, 129], kind))
    queries = (q, *rows_of(rng, NQ, [1, 20, 60], "negative" if kind == "negative" else "plain"), *rows_of(rng, NQ, [1, 20, 60], "plain"))
    rows = np.zeros((N, D + 8), np.uint32)
    rows[:, :D] = rng.integers(0, N, (N, D))
    return corpus, queries, rows, rng.choice(N, D, replace=False).astype(np.uint32)


@pytest.mark.parametrize("kind", ["plain", "magnitudes", "negative", "not numbers"])
def test_rows_are_those_of_a_walk_without_bounds(gpu_ctx, kind):
    import apoe
    import apoe_synth as S
    corpus, queries, rows, entry = world(kind, 3)
    b_idx = queries[5].copy()
    b_idx[queries[4][:-1]] |= np.uint32(0x80000000)  # the first BM25 term of every query is required
    gc, gq, gg = apoe.Corpus(gpu_ctx, *corpus), apoe.Queries(gpu_ctx, *queries), apoe.Graph(gpu_ctx, rows, entry)
    gk = apoe.Queries(gpu_ctx, *queries[:5], b_idx, queries[6])
    kg = apoe.KnowledgeGraph(gpu_ctx, *S.to_numpy(S.knowledge_graph(800, N, NQ, seed=23, device="cpu", mean_out=6.0)))
    gc.make_half_rows()
    for w3, cands, shape in (((8, 1, 1), 24, 4), ((49, 1, 1), 64, 1), ((24, 3, 0), 33, 1), ((16, 0, 2), 100, 4), ((1, 1, 1), 24, 4)):
        for query, more in ((gq, {}), (gk, dict(keyword_filter=True)), (gq, dict(kg=kg, kg_weight=5.0))):
            a, ad, sa = apoe.search(gpu_ctx, gc, query, gg, w3, cands, variant=shape, **more)
            b, bd, sb = apoe.search(gpu_ctx, gc, query, gg, w3, cands, variant=shape | 0x100, **more)
            assert np.array_equal(a, b) and np.array_equal(ad, bd, equal_nan=True), (w3, cands, sorted(more))
            assert sa.evaluations == sb.evaluations and sa.dense_rows <= sb.dense_rows
            if kind == "plain" and w3 == (49, 1, 1):  # codes are in use: sketches and dense rows alone (1 032 and 4 096 bytes each) do not explain what was read
                assert (sb.algo_bytes - sa.algo_bytes - 4096 * (sb.dense_rows - sa.dense_rows)) % 1032 != 0
        a, ad, _ = apoe.search(gpu_ctx, gc, gq, gg, w3, cands, variant=shape | 0x200)
        b, bd, _ = apoe.search(gpu_ctx, gc, gq, gg, w3, cands, variant=shape | 0x300)
        assert np.array_equal(a, b) and np.array_equal(ad, bd, equal_nan=True), (w3, cands, "half")


def test_which_weights_ask_codes(gpu_ctx):
    """A corpus without codes reads other bytes where they are asked: the dense part reaches an eighth of the pairs' under all but equal weights."""
    import apoe
    import apoe_synth as S
    corpus, queries, rows, entry = world("plain", 3)
    b_idx = queries[5].copy()
    b_idx[queries[4][:-1]] |= np.uint32(0x80000000)
    full, less = apoe.Corpus(gpu_ctx, *corpus), apoe.Corpus(gpu_ctx, *corpus, without=apoe.WITHOUT_CODES)
    gq, gk, gg = apoe.Queries(gpu_ctx, *queries), apoe.Queries(gpu_ctx, *queries[:5], b_idx, queries[6]), apoe.Graph(gpu_ctx, rows, entry)
    kg = apoe.KnowledgeGraph(gpu_ctx, *S.to_numpy(S.knowledge_graph(800, N, NQ, seed=23, device="cpu", mean_out=6.0)))
    for w3, cands, shape in (((8, 1, 1), 24, 4), ((49, 1, 1), 64, 1), ((24, 3, 0), 33, 1), ((16, 0, 2), 100, 4), ((1, 1, 1), 24, 4)):
        for query, more in ((gq, {}), (gk, dict(keyword_filter=True)), (gq, dict(kg=kg, kg_weight=5.0))):
            read = [apoe.search(gpu_ctx, gc, query, gg, w3, cands, variant=shape, **more)[2].algo_bytes for gc in (full, less)]
            assert (read[0] != read[1]) == (w3[0] > 1), (w3, cands, sorted(more))


def test_bytes_of_evaluations_that_the_codes_leave_open(gpu_ctx):
    """Documents that no bound tells apart (all alike): whatever the codes are asked for stays open, and what was read is codes (a byte and a
    16-bit term a pair) and sketch beside what a walk without bounds reads."""
    import apoe
    rng = np.random.default_rng(8)
    pairs_s, pairs_b = 40, 20
    off = lambda n, m: np.arange(n + 1, dtype=np.uint32) * np.uint32(m)
    same = lambda x, n: np.ascontiguousarray(np.broadcast_to(x, (n, len(x)))).astype(x.dtype)
    dense, terms = rng.standard_normal(1024).astype(np.float32), np.arange(64, dtype=np.uint32)
    val = rng.gamma(1.0, 1.0, 64).astype(np.float32)
    corpus = (same(dense, N), off(N, pairs_s), same(terms[:pairs_s], N).ravel(), same(val[:pairs_s], N).ravel(),
              off(N, pairs_b), same(terms[:pairs_b], N).ravel(), same(val[:pairs_b], N).ravel())
    queries = (same(dense, NQ), off(NQ, 10), same(terms[:10], NQ).ravel(), same(val[:10], NQ).ravel(),
               off(NQ, 10), same(terms[:10], NQ).ravel(), same(val[:10], NQ).ravel())
    rows = np.zeros((N, D + 8), np.uint32)
    rows[:, :D] = rng.integers(0, N, (N, D))
    gc, gq, gg = apoe.Corpus(gpu_ctx, *corpus), apoe.Queries(gpu_ctx, *queries), apoe.Graph(gpu_ctx, rows, np.arange(D, dtype=np.uint32))
    for w3, pairs in (((49, 1, 1), pairs_s + pairs_b), ((49, 1, 0), pairs_s)):
        _, _, sa = apoe.search(gpu_ctx, gc, gq, gg, w3, 24, variant=4)
        _, _, sb = apoe.search(gpu_ctx, gc, gq, gg, w3, 24, variant=4 | 0x100)
        assert sa.evaluations == sa.dense_rows == sb.evaluations == sb.dense_rows
        coded, rest = divmod(sa.algo_bytes - sb.algo_bytes, 3 * pairs + 1032)
        assert rest == 0 and 0 < coded < sa.evaluations, (coded, rest)


def test_codes_are_asked_where_the_dense_part_decides(gpu_ctx):
    """Under one set of weights: asked on a corpus whose dense parts weigh as much as its pairs, not on one whose values are ten times as
    large, and not where the bonus of a linking entity exceeds the dense part. A corpus without codes reads other bytes if they are asked."""
    import apoe
    import apoe_synth as S
    corpus, queries, rows, entry = world("plain", 3)
    kg = apoe.KnowledgeGraph(gpu_ctx, *S.to_numpy(S.knowledge_graph(800, N, NQ, seed=23, device="cpu", mean_out=6.0)))
    gq, gg = apoe.Queries(gpu_ctx, *queries), apoe.Graph(gpu_ctx, rows, entry)
    for scale, more, asked in ((1, {}, True), (10, {}, False), (1, dict(kg=kg, kg_weight=100.0), True), (1, dict(kg=kg, kg_weight=2000.0), False)):
        arrays = list(corpus)
        arrays[3], arrays[6] = arrays[3] * np.float32(scale), arrays[6] * np.float32(scale)
        read = []
        for without in (0, apoe.WITHOUT_CODES):
            gc = apoe.Corpus(gpu_ctx, *arrays, without=without)
            read.append(apoe.search(gpu_ctx, gc, gq, gg, (49, 1, 1), 64, variant=4, **more)[2].algo_bytes)
            gc.close()
        assert (read[0] != read[1]) == asked, (scale, sorted(more))


@pytest.mark.parametrize("pairs", [190, 194, 318, 322])
def test_codes_are_asked_up_to_a_row_length(gpu_ctx, pairs):
    """Rows of one length: to 192 pairs, what a batch of loads holds, in every search; to 320 in plain ones. Rows are those without codes either way."""
    import apoe
    rng = np.random.default_rng(pairs)
    corpus, queries, rows, entry = world("plain", 3)
    corpus = (corpus[0], *rows_of(rng, N, [pairs // 2], "plain"), *rows_of(rng, N, [pairs // 2], "plain"))
    b_idx = queries[5].copy()
    b_idx[queries[4][:-1]] |= np.uint32(0x80000000)
    gq, gk, gg = apoe.Queries(gpu_ctx, *queries), apoe.Queries(gpu_ctx, *queries[:5], b_idx, queries[6]), apoe.Graph(gpu_ctx, rows, entry)
    full, less = apoe.Corpus(gpu_ctx, *corpus), apoe.Corpus(gpu_ctx, *corpus, without=apoe.WITHOUT_CODES)
    full.make_half_rows()
    less.make_half_rows()
    for query, variant, more, limit in ((gq, 4, {}, 320), (gq, 4 | 0x200, {}, 192), (gk, 4, dict(keyword_filter=True), 192)):
        a, ad, sa = apoe.search(gpu_ctx, full, query, gg, (49, 1, 1), 64, variant=variant, **more)
        b, bd, sb = apoe.search(gpu_ctx, less, query, gg, (49, 1, 1), 64, variant=variant, **more)
        assert np.array_equal(a, b) and np.array_equal(ad, bd)
        assert (sa.algo_bytes != sb.algo_bytes) == (pairs <= limit), (variant, sorted(more))
    for x in (less, full, gg, gk, gq):
        x.close()
