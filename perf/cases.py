"""The calls whose time counts: searches over a stored index and index builds, through the ctypes binding (`apoe.py`)
of the C-ABI, on the synthetic corpora of `apoe_synth.py`.

A search case names the index it runs on (corpus kind, documents, degree, pair format): that is what a serving program
keeps, so it is made once per process and shared by every state; the queries come from the seed. Its graph is made here
with plain torch and not with the library's builder, whose result depends on the arrival order of reverse edges: two
runs of a case walk the same rows. A build case's input is its corpus: every seed gives another one. For the same reason
a whole build is followed by a search and gives that search's distances (they tell a good graph from a bad one, the
edge ids of two runs of one build differ; on the corpora whose rows have neighbours the distances agree to 1e-3); the stages whose ids do not depend on any order have a case of their own that
gives the rows.
"""
import collections
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.join(os.getcwd(), "allan-poe_amd"))
import apoe  # noqa: E402
import apoe_synth as S  # noqa: E402

DEV = "cuda:0"
WIDE_SHIFT = 70000          # added to BM25 term ids: past 65535 the records take the wide pair format
INDEXES_KEPT = 2            # the largest index is about 8 GB of records, graph and half-precision rows

_ctx = None
_indexes = collections.OrderedDict()


def search_case(name, corpus, docs, degree, queries, cands, weights=None, mode="plain", host=False, wide=False):
    """weights: dense, splade, bm25; by default what bench.py searches the corpus under."""
    w = weights or ((49.0, 1.0, 1.0) if corpus == "latent" else (1.0, 1.0, 1.0))
    c = dict(task="search", corpus=corpus, docs=docs, degree=degree, queries=queries, cands=cands, w_dense=w[0], w_splade=w[1], w_bm25=w[2],
             mode=mode, host=host, wide=wide)
    return dict(name=name, **c) if name else c


def build_case(name, corpus, docs, K, degree, iters=10, host=False, wide=False, queries=500, cands=64):
    c = dict(task="build", corpus=corpus, docs=docs, K=K, degree=degree, iters=iters, host=host, wide=wide, queries=queries, cands=cands, mode="plain")
    return dict(name=name, **c) if name else c


def refine_case(name, corpus, docs, K, degree, wide=False):
    c = dict(task="refine", corpus=corpus, docs=docs, K=K, degree=degree, wide=wide)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one user's query against a small index: the time to an answer
        search_case("search_1", "iid", 100_000, 32, 1, 128),
        # a request to a server: a few dozen new queries arrive in host memory, the rows go back there
        search_case("serve_64_host", "latent", 200_000, 48, 64, 100, host=True),
        # a keyword-filter search on a corpus whose term ids need the wide pair format
        search_case("keyword_777_wide", "iid", 99_991, 32, 777, 128, mode="keyword", wide=True),
        # a deep pool, weighted as in the weight sweep
        search_case("deep_pool_500", "iid", 100_000, 32, 500, 1000, weights=(1.0, 0.5, 2.0)),
        # the headline batch: 10 000 queries, a million documents, all paths, the largest configured pool
        search_case("batch_10k_iid_1m", "iid", 1_000_000, 48, 10_000, 256),
        # the same index with a knowledge graph of 200 000 entities
        search_case("kg_10k_1m", "iid", 1_000_000, 48, 10_000, 128, mode="kg"),
        # a million documents whose dense rows have neighbours, at the pool where recall@10 passes 0.95
        search_case("batch_10k_latent_1m", "latent", 1_000_000, 48, 10_000, 80),
        # the same index, a shorter batch, the walk on half-precision rows
        search_case("half_1000_latent_1m", "latent", 1_000_000, 48, 1000, 64, mode="half"),
        # builds: a small corpus that arrives in host memory, a larger one resident on the GPU, and the K = 128 lists
        build_case("build_4k_host", "latent", 4000, 64, 32, host=True),
        build_case("build_100k_latent", "latent", 100_000, 64, 48),
        build_case("build_30k_k128", "latent", 30_011, 128, 64),
        # saved neighbour lists taken up again: one more step, then a graph of another degree
        refine_case("refine_100k_lists", "iid", 100_000, 64, 32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.3:
        K = 128 if rng.random() < 0.3 else 64
        docs = _log_int(rng, 2000, 100_000 if K == 64 else 30_000)
        if rng.random() < 0.3:
            return refine_case(None, rng.choice(("iid", "latent")), docs, K, rng.choice((24, 32, 48, 64)), wide=rng.random() < 0.2)
        return build_case(None, "latent", docs, K, rng.choice((24, 32, 48, 64)), iters=rng.randint(6, 10),
                          host=rng.random() < 0.4, wide=rng.random() < 0.2)
    corpus = rng.choice(("iid", "latent"))
    mode = rng.choice(("plain", "plain", "plain", "kg", "keyword", "half"))
    weights = None if rng.random() < 0.6 else rng.choice(((1.0, 0.0, 0.0), (0.0, 1.0, 0.0), (0.0, 0.0, 1.0), (1.0, 0.5, 2.0)))
    docs = _log_int(rng, 4000, 500_000)
    cands = _log_int(rng, 16, 1024)
    queries = min(_log_int(rng, 1, 10_000), max(1, 10_000 * 256 // cands))
    return search_case(None, corpus, docs, rng.choice((24, 32, 48, 64)), queries, cands, weights=weights, mode=mode,
                       host=rng.random() < 0.3, wide=rng.random() < 0.2)


# ---- what a program has in hand ----

def _context():
    global _ctx
    if _ctx is None:
        _ctx = apoe.Context(0)
    return _ctx


def _widen(arrays):
    return tuple(arrays[:5]) + (arrays[5] + WIDE_SHIFT,) + tuple(arrays[6:])


def _corpus_arrays(case, seed):
    a = (S.latent_corpus if case["corpus"] == "latent" else S.corpus)(case["docs"], seed=seed, device=DEV)
    return _widen(a) if case["wide"] else a


def _query_arrays(case, seed):
    a = (S.latent_queries if case["corpus"] == "latent" else S.queries)(case["queries"], seed=seed, device=DEV)
    a = _widen(a) if case["wide"] else a
    if case["mode"] == "keyword":  # one BM25 term of every query, somewhere in its row, is a required keyword
        off, idx = a[4].long(), a[5].clone()
        cnt = off[1:] - off[:-1]
        g = torch.Generator(device=DEV).manual_seed(seed)
        at = off[:-1] + (torch.rand(cnt.numel(), generator=g, device=DEV) * cnt).long().clamp_max(torch.clamp(cnt - 1, min=0))
        at = at[cnt > 0]
        idx[at] = torch.bitwise_or(idx[at], -2 ** 31)
        a = a[:5] + (idx,) + a[6:]
    return a


def _features(arrays, wide, terms=128):
    """Rows whose inner products come near the build metric: the dense row times 7 and the values of the most frequent
    terms of either path (the generator's term ids are frequency ranks)."""
    dense, s_off, s_idx, s_val, b_off, b_idx, b_val = arrays
    n = dense.shape[0]
    f = torch.zeros(n, dense.shape[1] + 2 * terms, device=DEV)
    f[:, :dense.shape[1]] = dense * 7.0
    for k, (off, idx, val) in enumerate(((s_off, s_idx, s_val), (b_off, b_idx - (WIDE_SHIFT if wide else 0), b_val))):
        row = torch.repeat_interleave(torch.arange(n, device=DEV), (off[1:] - off[:-1]).long())
        m = idx < terms
        f[row[m], dense.shape[1] + k * terms + idx[m].long()] = val[m]
    return f


def _near_in_blocks(f, k, g, block=256):
    """The k rows of largest inner product with every row among about 256 rows that lie near it, and the products: rows
    sorted by the random pivot row they are closest to in direction, cut into blocks."""
    n = f.shape[0]
    block = min(block, n)
    pivots = f[torch.randperm(n, generator=g, device=DEV)[:max(8, min(2048, n // 128))]]
    pivots = pivots / pivots.norm(dim=1, keepdim=True)
    cell = torch.cat([(f[i:i + 65536] @ pivots.T).argmax(1) for i in range(0, n, 65536)])
    order = torch.sort(cell, stable=True)[1]
    near, value = torch.empty(n, k, dtype=torch.int64, device=DEV), torch.empty(n, k, device=DEV)
    whole = n // block
    parts = [order[b * block:min(b + 128, whole) * block] for b in range(0, whole, 128)] + [order[n - block:]]  # a partial block: the last rows again
    for part in parts:
        at = part.reshape(-1, block)
        x = f[at]
        ip = torch.bmm(x, x.transpose(1, 2).contiguous())
        ip.diagonal(dim1=1, dim2=2).fill_(float("-inf"))
        val, top = ip.topk(k, dim=2)
        near[at.reshape(-1)] = torch.gather(at, 1, top.reshape(at.shape[0], -1)).reshape(-1, k)
        value[at.reshape(-1)] = val.reshape(-1, k)
    return near, value


def _graph_rows(arrays, degree, wide, seed):
    """Rows [n, degree + 8] and entry points: near rows under two partitions, two random rows, up to seven keyword edges;
    an edge that repeats one of its row is replaced by a random one."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    f = _features(arrays, wide)
    n, half = f.shape[0], degree // 2
    adj = torch.cat([_near_in_blocks(f, half, g)[0], _near_in_blocks(f, degree - half - 2, g)[0], torch.randint(n, (n, 2), generator=g, device=DEV)], 1)
    srt, pos = torch.sort(adj, dim=1, stable=True)
    again = torch.zeros_like(adj, dtype=torch.bool)
    again[:, 1:] = srt[:, 1:] == srt[:, :-1]
    again = torch.zeros_like(again).scatter(1, pos, again)
    adj = torch.where(again, torch.randint(n, adj.shape, generator=g, device=DEV), adj)
    rows = torch.zeros(n, degree + 8, dtype=torch.int32, device=DEV)
    rows[:, :degree] = adj.to(torch.int32)
    rows[:, degree] = torch.randint(8, (n,), generator=g, device=DEV).to(torch.int32)
    rows[:, degree + 1:] = torch.randint(n, (n, 7), generator=g, device=DEV).to(torch.int32)
    entry = torch.sort(f.norm(dim=1), stable=True)[1][:degree].to(torch.int32)
    return rows, entry


def _index(case):
    key = (case["corpus"], case["docs"], case["degree"], case["wide"])
    if key in _indexes:
        _indexes.move_to_end(key)
        return _indexes[key]
    while len(_indexes) >= INDEXES_KEPT:
        _, (gc, gg) = _indexes.popitem(last=False)
        gg.close()
        gc.close()
    arrays = _corpus_arrays(case, 20251125)
    rows, entry = _graph_rows(arrays, case["degree"], case["wide"], 7)
    torch.cuda.synchronize()
    gc = apoe.Corpus(_context(), *arrays)
    gg = apoe.Graph(_context(), rows, entry)
    _indexes[key] = (gc, gg)
    return gc, gg


def prepare(case, seed):
    ctx = _context()
    st = dict(case=case, ctx=ctx)
    if case["task"] == "build":
        arrays = _corpus_arrays(case, seed)
        queries = _query_arrays(case, seed)
        torch.cuda.synchronize()
        if case["host"]:
            st["arrays"] = S.to_numpy(arrays)
        else:
            st["corpus"] = apoe.Corpus(ctx, *arrays)
        st["queries"] = apoe.Queries(ctx, *queries)
        return st
    if case["task"] == "refine":
        arrays = _corpus_arrays(case, seed)
        near, ip = _near_in_blocks(_features(arrays, case["wide"]), case["K"], torch.Generator(device=DEV).manual_seed(seed))
        st["ids"], st["dist"] = near.to(torch.int32), 1.0 - ip
        torch.cuda.synchronize()
        st["corpus"] = apoe.Corpus(ctx, *arrays)
        return st
    st["corpus"], st["graph"] = _index(case)
    arrays = _query_arrays(case, seed)
    torch.cuda.synchronize()
    if case["host"]:
        st["arrays"] = S.to_numpy(arrays)
    else:
        st["queries"] = apoe.Queries(ctx, *arrays)
        st["out_ids"] = torch.empty((case["queries"], case["cands"]), dtype=torch.int32, device=DEV)
        st["out_dist"] = torch.empty((case["queries"], case["cands"]), dtype=torch.float32, device=DEV)
    if case["mode"] == "kg":
        kg = S.knowledge_graph(max(100, case["docs"] // 5), case["docs"], case["queries"], seed=seed, device=DEV)
        torch.cuda.synchronize()
        st["kg"] = apoe.KnowledgeGraph(ctx, *kg)
    if case["mode"] == "half":
        st["corpus"].make_half_rows()
    torch.cuda.synchronize()
    return st


# ---- one pass ----

def run(st):
    case, ctx = st["case"], st["ctx"]
    if case["task"] == "build":
        corpus = apoe.Corpus(ctx, *st["arrays"]) if case["host"] else st["corpus"]
        graph, _ = apoe.build_graph(ctx, corpus, K=case["K"], iters=case["iters"], degree=case["degree"], seed=1, join=1)
        _, dist, _ = apoe.search(ctx, corpus, st["queries"], graph, (49.0, 1.0, 1.0), case["cands"])
        graph.close()
        if case["host"]:
            corpus.close()
        return {"dist": dist}
    if case["task"] == "refine":
        knn = apoe.Knn(ctx, st["corpus"], case["K"], 7.0)
        knn.upload(st["ids"], st["dist"])
        knn.set_join(1)
        knn.iterate(last=True)
        knn.prune(case["degree"])
        graph = knn.finalize()
        knn.close()
        rows, entry = graph.download()
        graph.close()
        return {"rows": rows, "entry": entry}
    queries = apoe.Queries(ctx, *st["arrays"]) if case["host"] else st["queries"]
    ids, dist, _ = apoe.search(ctx, st["corpus"], queries, st["graph"], (case["w_dense"], case["w_splade"], case["w_bm25"]), case["cands"],
                               kg=st.get("kg"), kg_weight=40.0 if case["mode"] == "kg" else 0.0, variant=0x200 if case["mode"] == "half" else 0,
                               keyword_filter=case["mode"] == "keyword", out_ids=st.get("out_ids"), out_dist=st.get("out_dist"))
    if case["host"]:
        queries.close()
    return {"ids": ids, "dist": dist}


# ---- what a pass cannot do without ----

ROW_BYTES = 4 * S.DIM + 6 * 180   # a dense row and about 180 (term, value) pairs
PAIR_FLOPS = 2 * (S.DIM + 60)     # a dense product and the terms that two rows share


def work(case):
    n = case["docs"]
    if case["task"] != "search":
        # corpus read and rows written once (saved lists read once too); per step about 456 pairs per document and 64 list
        # entries, then the upper triangle of every list's products
        steps, lists = (case["iters"], 0) if case["task"] == "build" else (1, 8.0 * case["K"])
        pairs = n * (steps * 456.0 * (case["K"] / 64) ** 2 + case["K"] ** 2 / 2)
        return {"bytes": n * (ROW_BYTES + lists + 4.0 * (case["degree"] + 8)), "flops": pairs * PAIR_FLOPS}
    q = case["queries"]
    evaluated = min(n, 0.8 * case["cands"] * case["degree"])
    expanded = min(n, 1.03 * case["cands"])
    flops = 2 * 60 + (2 * S.DIM if case["w_dense"] > 0 else 0)
    row = (4 * S.DIM if case["w_dense"] > 0 else 0) + 6 * 180
    return {"bytes": min(n, q * evaluated) * row + min(n, q * expanded) * 4.0 * (case["degree"] + 8) + q * (4 * S.DIM + 8 * 38 + 8.0 * case["cands"]),
            "flops": q * evaluated * flops}


def tolerance(case):
    """About four times what a case gives when the 1024 dimensions are summed in another order. Searches: 6e-8 on distances, 4e-5
    of the ids (near-ties), and now and then a near-tie that sends the walk another way; the half-precision walk meets more of
    those (2e-4 and 1e-3). Builds: 9e-4, as two runs of one build do. Refined lists: no id differs."""
    if case["task"] == "build":
        return {"rel": 4e-3, "max": 0.1}
    if case["task"] == "refine":
        return {"differ": 1e-4}
    if case["mode"] == "half":
        return {"rel": 8e-4, "max": 5e-2, "differ": 4e-3}
    return {"rel": 1e-5, "max": 1e-2, "differ": 2e-4}
