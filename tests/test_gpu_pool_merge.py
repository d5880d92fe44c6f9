"""The pool merge (groups of 4 x 64 entries read from the pool's end) at pool sizes around its group and round edges, and
keyword flags that travel in the keys of the query's term table, overflow entries included."""
import numpy as np
import pytest

from keyword_worlds import EMPTY_ID, KW
from parity import assert_dist_close, assert_topk_match

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [1, 4, 5])
@pytest.mark.parametrize("cands", [2, 63, 64, 65, 255, 256, 257, 320, 513])
def test_pool_sizes_around_the_merge_groups(gpu_world, cands, variant):
    """Whole pools, not only their heads: an entry that a merge loses or doubles shows up behind the top ten."""
    import apoe
    import oracle as O
    w = gpu_world
    nq = 24
    ids, dist, _ = apoe.search(w["ctx"], w["gc"], w["gq"], w["gg"], (1, 1, 1), cands, q_count=nq, variant=variant)
    oid, odist, _ = O.search(w["C"], w["Q"].head(nq), w["rows"], w["entry"], (1, 1, 1), cands)
    assert_topk_match(ids, dist, oid, odist, cands, f"cands {cands}")
    assert_dist_close(dist, odist, f"cands {cands}: pool distances") # an order that differs at a tie keeps the sorted distances
    for row in ids:
        real = row[row != EMPTY_ID]
        assert len(set(real.tolist())) == len(real)


@pytest.mark.parametrize("variant", [1, 4, 5])
@pytest.mark.parametrize("cands", [1, 7, 16, 65, 255, 256, 257, 320, 513])
def test_knowledge_graph_pools_around_the_merge_groups(gpu_world, cands, variant):
    """Linking entity and hop travel with an entry through the groups: one that goes astray sends the walk to other documents. The
    smallest pools hold fewer entries than the walk has seeds."""
    import apoe
    import apoe_synth as S
    import oracle as O
    w = gpu_world
    nq = 24
    kg = S.to_numpy(S.knowledge_graph(1500, w["C"].n, nq, seed=31, device="cpu", mean_out=6.0))
    gkg = apoe.KnowledgeGraph(w["ctx"], *kg)
    ids, dist, st = apoe.search(w["ctx"], w["gc"], w["gq"], w["gg"], (1, 1, 1), cands, kg=gkg, kg_weight=20.0, q_count=nq, variant=variant)
    oid, odist, cnt = O.search(w["C"], w["Q"].head(nq), w["rows"], w["entry"], (1, 1, 1), cands, kg=O.Kg(*kg), kg_weight=20.0)
    assert_topk_match(ids, dist, oid, odist, cands, f"kg, cands {cands}")
    assert_dist_close(dist, odist, f"kg, cands {cands}: pool distances")
    assert abs(int(st.evaluations) - int(cnt[:, 1].sum())) <= 0.01 * cnt[:, 1].sum()
    gkg.close()


@pytest.mark.parametrize("variant", [1, 4, 5])
@pytest.mark.parametrize("cands", [65, 66, 80, 129, 130, 257, 321])
def test_hits_pushed_out_around_the_last_round(gpu_world, cands, variant):
    """Pools whose last 64-entry round holds one, two or sixteen entries: a merge of up to 32 new candidates pushes out entries of that
    round and of the one before. Of each query the term that about three tenths of the documents hold is required, and BM25 has no
    weight: hits enter and leave the pool like any other document, and a row ends with those that were pushed out last."""
    import apoe
    import oracle as O
    w = gpu_world
    nq = 24
    qa = list(O.HybridSet(*w["queries"]).head(nq).arrays())
    off, idx = qa[4], qa[5].copy()
    df = np.bincount(w["corpus"][5], minlength=int(max(w["corpus"][5].max(), idx.max())) + 1)
    for q in range(nq):
        if off[q] < off[q + 1]:
            idx[off[q] + np.argmin(np.abs(df[idx[off[q]:off[q + 1]]] - 0.3 * w["C"].n))] |= np.uint32(KW)
    qa[5] = idx
    gq = apoe.Queries(w["ctx"], *qa)
    ids, dist, _ = apoe.search(w["ctx"], w["gc"], gq, w["gg"], (1, 1, 0), cands, keyword_filter=True, variant=variant)
    oid, odist, _ = O.search(w["C"], O.HybridSet(*qa), w["rows"], w["entry"], (1, 1, 0), cands, keyword_filter=True)
    assert_topk_match(ids, dist, oid, odist, cands, f"keyword, cands {cands}")
    assert_dist_close(dist, odist, f"keyword, cands {cands}: row distances")
    worst = O.search(w["C"], w["Q"].head(nq), w["rows"], w["entry"], (1, 1, 0), cands)[1][:, -1]
    behind = ((oid != EMPTY_ID) & (odist > worst[:, None])).sum(axis=1) # hits beyond the last entry of the pool
    assert np.median(behind) >= 20


def colliding_terms(count, buckets):
    """Term ids below 65 536 whose table bucket is the same: ((term * 0x9E3779) mod 2^32 >> 10) mod buckets."""
    t = np.arange(1, 65536, dtype=np.uint64)
    h = ((t * 0x9E3779) & 0xFFFFFFFF) >> 10
    return t[h % buckets == 5][:count].astype(np.uint32)


@pytest.mark.parametrize("n_flagged", [0, 1, 3, 6, 12])
@pytest.mark.parametrize("wide", [False, True])
def test_flags_of_overflow_entries(gpu_ctx, wide, n_flagged):
    """Twelve query terms in one bucket of two entries: ten go to the overflow list, required ones from its end. Every document
    holds one of the terms, so the hits are exactly the documents of the flagged ones (the walk reaches every document)."""
    import apoe
    import oracle as O
    n, d, nt = 48, 8, 12
    rng = np.random.default_rng(4)
    terms = colliding_terms(nt, 32) # 12 terms: next power of two above 24 buckets
    dense = rng.standard_normal((n + 1, 1024)).astype(np.float32)
    dense /= np.linalg.norm(dense, axis=1, keepdims=True)
    none = lambda k: (np.zeros(k + 1, np.uint32), np.zeros(0, np.uint32), np.zeros(0, np.float32))
    doc_terms = terms[np.arange(n) % nt]
    extra = np.full(n, 69999 if wide else 9, np.uint32) # one term past 65 535 takes the wide pair format
    b_idx = np.stack([doc_terms, extra], 1).reshape(-1)
    C = O.HybridSet(dense[:n], *none(n), np.arange(0, 2 * n + 1, 2, dtype=np.uint32), b_idx, rng.random(2 * n).astype(np.float32))
    flags = np.zeros(nt, np.uint32)
    flags[rng.permutation(nt)[:n_flagged]] = KW
    Q = O.HybridSet(dense[n:], *none(1), np.array([0, nt], np.uint32), terms | flags, rng.random(nt).astype(np.float32))
    rows = np.zeros((n, d + 8), np.uint32)
    rows[:, :d] = (np.arange(n)[:, None] + np.arange(1, d + 1)) % n
    entry = np.arange(d, dtype=np.uint32)
    gc, gq, gg = apoe.Corpus(gpu_ctx, *C.arrays()), apoe.Queries(gpu_ctx, *Q.arrays()), apoe.Graph(gpu_ctx, rows, entry)
    ids, dist, _ = apoe.search(gpu_ctx, gc, gq, gg, (1, 1, 1), 64, keyword_filter=True)
    oid, odist, _ = O.search(C, Q, rows, entry, (1, 1, 1), 64, keyword_filter=True)
    assert np.array_equal(ids, oid)
    assert_dist_close(dist, odist, "hits and the empty rest")
    assert set(ids[0][ids[0] != EMPTY_ID].tolist()) == {v for v in range(n) if flags[v % nt]}


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("keyword_filter", [False, True])
def test_query_terms_that_no_document_can_hold(gpu_ctx, wide, keyword_filter):
    """The BM25 id 0xFFFFFFFF (0x7FFFFFFF flagged as required) is no document's and reads as an empty table slot. Queries of 192 terms,
    64 of them that id, the terms that share its bucket handled by other waves: the rows are those of the queries without it."""
    import apoe
    n, d, nq, nt = 64, 16, 2000, 192
    rng = np.random.default_rng(11)
    k = np.uint64(0x7FFFFFFF)
    t = np.arange(70000, 200000, dtype=np.uint64) if wide else np.arange(1, 65536, dtype=np.uint64)
    low = (lambda x: (x ^ (x >> np.uint64(16))) & np.uint64(0xFFFFFF)) if wide else (lambda x: x & np.uint64(0xFFFFFF))
    bucket = lambda x: (((low(x) * np.uint64(0x9E3779)) & np.uint64(0xFFFFFFFF)) >> np.uint64(10)) % np.uint64(512) # next power of two above 2 * 192 terms
    same, other = t[bucket(t) == bucket(k)].astype(np.uint32), t[bucket(t) != bucket(k)].astype(np.uint32)
    terms = np.concatenate([np.full(64, 0xFFFFFFFF, np.uint32), same[:1], other[:63], same[1:2], other[63:126]])
    dense = rng.standard_normal((n, 1024)).astype(np.float32)
    none = lambda m: (np.zeros(m + 1, np.uint32), np.zeros(0, np.uint32), np.zeros(0, np.float32))
    corpus = (dense, *none(n), np.arange(0, 2 * n + 1, 2, dtype=np.uint32), np.tile(same[:2], n), rng.random(2 * n).astype(np.float32) + 1)
    rows = np.zeros((n, d + 8), np.uint32)
    rows[:, :d] = (np.arange(n)[:, None] + np.arange(1, d + 1)) % n
    gc, gg = apoe.Corpus(gpu_ctx, *corpus), apoe.Graph(gpu_ctx, rows, np.arange(d, dtype=np.uint32))
    assert gc.pair_bytes() == (8 if wide else 6)
    q = rng.standard_normal((nq, 1024)).astype(np.float32)
    val = rng.random((nq, nt)).astype(np.float32) + 1
    flag = np.uint32(KW if keyword_filter else 0)
    off = lambda m: np.arange(0, m * nq + 1, m, dtype=np.uint32)
    with_it = apoe.Queries(gpu_ctx, q, *none(nq), off(nt), np.tile(terms | flag, nq), val.reshape(-1))
    without = apoe.Queries(gpu_ctx, q, *none(nq), off(nt - 64), np.tile(terms[64:] | flag, nq), np.ascontiguousarray(val[:, 64:]).reshape(-1))
    for variant in (1, 4, 2, 5):
        a, ad, _ = apoe.search(gpu_ctx, gc, with_it, gg, (0, 0, 1), 40, keyword_filter=keyword_filter, variant=variant)
        b, bd, _ = apoe.search(gpu_ctx, gc, without, gg, (0, 0, 1), 40, keyword_filter=keyword_filter, variant=variant)
        assert np.array_equal(a, b) and np.array_equal(ad, bd), (variant, int((a != b).any(axis=1).sum()))
