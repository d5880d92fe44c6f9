"""A corpus that goes without the byte codes of its values, without the sketches of its dense rows, or without either, as a large one does when
device memory is short: distances, searches, join steps and prunes are those of a corpus that has them."""
import numpy as np
import pytest

import test_gpu_join_tiles as tiles
import test_gpu_prune_ties as prune
import test_gpu_value_codes as values

pytestmark = pytest.mark.gpu
CODES, SKETCHES = 1, 2


@pytest.mark.parametrize("without", [CODES, SKETCHES, CODES | SKETCHES])
@pytest.mark.parametrize("kind", ["plain", "not numbers"])
def test_searches_and_distances(gpu_ctx, kind, without):
    import apoe
    import apoe_synth as S
    corpus, queries, rows, entry = values.world(kind, 9)
    b_idx = queries[5].copy()
    b_idx[queries[4][:-1]] |= np.uint32(0x80000000)  # the first BM25 term of every query is required
    full, less = apoe.Corpus(gpu_ctx, *corpus), apoe.Corpus(gpu_ctx, *corpus, without=without)
    assert full.bytes() == less.bytes() and full.pair_bytes() == less.pair_bytes() == 6
    gq, gk, gg = apoe.Queries(gpu_ctx, *queries), apoe.Queries(gpu_ctx, *queries[:5], b_idx, queries[6]), apoe.Graph(gpu_ctx, rows, entry)
    kg = apoe.KnowledgeGraph(gpu_ctx, *S.to_numpy(S.knowledge_graph(800, values.N, values.NQ, seed=23, device="cpu", mean_out=6.0)))
    full.make_half_rows()
    less.make_half_rows()
    ids = np.random.default_rng(1).integers(0, values.N, (values.NQ, 50)).astype(np.uint32)
    for w3, cands, shape in (((49, 1, 1), 64, 4), ((16, 0, 2), 100, 1), ((1, 1, 1), 24, 3), ((1, 0, 0), 33, 0)):
        assert np.array_equal(apoe.distance_batch(gpu_ctx, full, gq, w3, ids), apoe.distance_batch(gpu_ctx, less, gq, w3, ids), equal_nan=True)
        for query, variant, more in ((gq, shape, {}), (gq, shape | 0x200, {}), (gk, shape, dict(keyword_filter=True)), (gq, shape, dict(kg=kg, kg_weight=5.0))):
            a, ad, sa = apoe.search(gpu_ctx, full, query, gg, w3, cands, variant=variant, **more)
            b, bd, sb = apoe.search(gpu_ctx, less, query, gg, w3, cands, variant=variant, **more)
            assert np.array_equal(a, b) and np.array_equal(ad, bd, equal_nan=True), (w3, cands, variant, sorted(more))
            assert sa.evaluations == sb.evaluations
            if not without & SKETCHES:
                assert sa.dense_rows >= sb.dense_rows if w3[0] >= 8 else sa.dense_rows == sb.dense_rows  # codes leave a little more open than pairs do
            elif w3 == (1, 0, 0) and not more:
                assert sa.dense_rows < sb.dense_rows == sb.evaluations
    assert np.array_equal(apoe.norms(gpu_ctx, full, 7.0), apoe.norms(gpu_ctx, less, 7.0), equal_nan=True)
    for x in (kg, gg, gk, gq, less, full):
        x.close()


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("K,degree", [(64, 32), (128, 48)])
@pytest.mark.parametrize("kind", ["bounds settle", "near twins", "rich rows", "odd rows"])
def test_prune_without_sketches_matches_oracle(gpu_ctx, kind, K, degree, wide):
    prune.check(gpu_ctx, kind, K, degree, wide, without=CODES | SKETCHES)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("K", [64, 128])
def test_join_step_without_sketches_matches_oracle(gpu_ctx, small_world, K, wide):
    import apoe
    import oracle as O
    arrays = list(small_world["corpus"])
    if wide:
        arrays[5] = arrays[5] + np.uint32(70000)
    n, rng = small_world["C"].n, np.random.default_rng(K)
    ids = np.stack([rng.choice(n, K, replace=False) for _ in range(n)]).astype(np.uint32)
    gc = apoe.Corpus(gpu_ctx, *arrays, without=CODES | SKETCHES)
    tiles.step_equals_oracle(gpu_ctx, gc, O.HybridSet(*arrays), ids, K)
    gc.close()


def test_a_build_and_its_counters(gpu_ctx):
    import apoe
    import apoe_synth as S
    arrays = S.to_numpy(S.latent_corpus(3000, seed=31, device="cpu"))
    read = []
    for without in (0, SKETCHES):
        gc = apoe.Corpus(gpu_ctx, *arrays, without=without)
        knn = apoe.Knn(gpu_ctx, gc, 64, 7.0)
        knn.set_join(1)
        knn.init(1)
        for it in range(10):
            knn.iterate(last=(it == 9))
        dense, pair_rows, sketches = knn.read_counters()
        read.append(dense)
        assert (dense == pair_rows and sketches == 0) if without else (dense < pair_rows and sketches > 0)
        knn.merge_reverse()
        knn.prune(32)
        knn.finalize().close()
        knn.close()
        gc.close()
    assert read[0] < 0.95 * read[1]  # the same build reads fewer dense rows with them


def test_unknown_flags_are_refused(gpu_ctx):
    import apoe
    corpus = values.world("plain", 9)[0]
    with pytest.raises(apoe.ApoeError, match="flags"):
        apoe.Corpus(gpu_ctx, *corpus, without=4)
