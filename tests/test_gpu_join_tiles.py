"""Tile shapes of the local join: columns that fill one, two, four or eight blocks of sixteen (the waves of a workgroup then split the
dimensions sixteen, eight, four or two ways), and one more than a block; lists of 128 entries for the columns that 64 cannot hold."""
import numpy as np
import pytest

from parity import assert_dist_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("columns", [1, 15, 16, 17, 32, 33, 64, 65, 96, 112, 113, 127, 128])
def test_first_step_on_lists_of_few_documents(gpu_world, columns):
    """Every list names `columns` documents (repeated to K entries), so a tile has that many columns (reverse lists are empty);
    picked nodes have about 4 x K / columns pickers, whole and partial blocks of rows. The step's lists are the oracle's, row for row."""
    import apoe
    import oracle as O
    w = gpu_world
    n, K = w["C"].n, 64 if columns <= 64 else 128
    rng = np.random.default_rng(columns)
    few = rng.integers(0, n, (n, columns)).astype(np.uint32)
    ids = few[:, np.arange(K) % columns]
    dist = np.sort(rng.random((n, K)).astype(np.float32) + 900, axis=1)
    st = O.nnd_init(n, K, 1) # its reverse lists are empty
    st.ids[:] = ids
    st.dist[:] = dist
    knn = apoe.Knn(w["ctx"], w["gc"], K, 7.0)
    knn.upload(ids, dist)
    knn.set_join(1)
    ins = knn.iterate(last=True)
    oins, _ = O.join_iterate(w["C"], 7.0, st, slots=2 * K)
    got, gd = knn.download()
    oids = st.ids & 0x7FFFFFFF
    assert abs(ins - oins) <= 0.001 * oins + 1
    same = np.all(got == oids, axis=1)
    assert same.mean() >= 0.99
    assert_dist_close(gd[same], st.dist[same], "stored distances")
    knn.close()


def step_equals_oracle(ctx, corpus, oracle_corpus, ids, K):
    """One join step from the lists `ids` (reverse lists empty), row for row the oracle's."""
    import apoe
    import oracle as O
    n = len(ids)
    dist = np.sort(np.random.default_rng(1).random((n, K)).astype(np.float32) + 900, axis=1)
    st = O.nnd_init(n, K, 1)
    st.ids[:] = ids
    st.dist[:] = dist
    knn = apoe.Knn(ctx, corpus, K, 7.0)
    knn.upload(ids, dist)
    knn.set_join(1)
    ins = knn.iterate(last=True)
    oins, _ = O.join_iterate(oracle_corpus, 7.0, st, slots=2 * K)
    got, gd = knn.download()
    assert abs(ins - oins) <= 0.001 * oins + 1
    same = np.all(got == (st.ids & 0x7FFFFFFF), axis=1)
    assert same.mean() >= 0.99
    assert_dist_close(gd[same], st.dist[same], "stored distances")
    knn.close()


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("pickers", [1, 8, 9, 11, 12, 13, 16, 17, 22, 25, 26, 31, 32, 33])
def test_tiles_of_a_given_number_of_pickers(gpu_world, pickers, K):
    """Blocks of `pickers` documents pick the same four nodes: tiles of that many rows (staged whole, in halves or in quarters;
    one or two accumulators; groups of eight pivots whole and partial) with the 64 or 128 columns of a full list."""
    w = gpu_world
    n = w["C"].n
    rng = np.random.default_rng(pickers)
    ids = np.stack([rng.choice(n, K, replace=False) for _ in range(n)]).astype(np.uint32)
    ids[:, :4] = 4 * (np.arange(n) // pickers)[:, None] % (n - 4) + np.arange(4)
    step_equals_oracle(w["ctx"], w["gc"], w["C"], ids, K)


@pytest.mark.parametrize("shift,terms", [(0, 1200), (0, 1345), (0, 1700), (70000, 900), (70000, 1100)])
def test_a_row_that_takes_the_whole_table(gpu_ctx, shift, terms):
    """One document's row fills the table that two workgroups per CU leave room for, or exceeds it: then one workgroup per CU runs
    the tiles (`shift`: term ids past 65535 take the wide pair format, whose table hashes)."""
    import apoe
    import apoe_synth as S
    import oracle as O
    n, K, row = 600, 64, 17
    dense, s_off, s_idx, s_val, b_off, b_idx, b_val = S.to_numpy(S.corpus(n, seed=5, device="cpu"))
    rng = np.random.default_rng(terms)
    cnt = np.diff(s_off.astype(np.int64))
    cnt[row] = terms
    off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.uint32)
    keep = lambda a, new: np.concatenate([a[:s_off[row]], new, a[s_off[row + 1]:]]).astype(a.dtype)
    idx = keep(s_idx, np.sort(rng.choice(30000, terms, replace=False)))
    val = keep(s_val, rng.uniform(0.5, 2.0, terms))
    arrays = (dense, off, idx, val, b_off, (b_idx + np.uint32(shift)).astype(np.uint32), b_val)
    gc = apoe.Corpus(gpu_ctx, *arrays)
    assert gc.pair_bytes() == (8 if shift else 6)
    ids = np.stack([rng.choice(n, K, replace=False) for _ in range(n)]).astype(np.uint32)
    ids[:, 0] = row  # every document picks the long row, and it is a column wherever it is not
    step_equals_oracle(gpu_ctx, gc, O.HybridSet(*arrays), ids, K)
    gc.close()


@pytest.mark.parametrize("vocab,terms", [(30000, 300), (30000, 340), (30000, 700), (60000, 190), (60000, 215)])
def test_rows_of_many_terms(gpu_ctx, vocab, terms):
    """Rows on both sides of the line between two workgroups per CU, whose table holds four of them and more, and one."""
    import apoe
    import apoe_synth as S
    import oracle as O
    n, K = 600, 64
    rng = np.random.default_rng(terms)
    dense, _, _, _, b_off, b_idx, b_val = S.to_numpy(S.corpus(n, seed=5, device="cpu"))
    cnt = np.maximum(1, terms - np.diff(b_off.astype(np.int64)) + rng.integers(-20, 21, n))
    off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.uint32)
    idx = np.concatenate([np.sort(rng.choice(vocab, c, replace=False)) for c in cnt]).astype(np.uint32)
    idx[0] = 0
    idx[off[1] - 1] = vocab - 1
    arrays = (dense, off, idx, rng.uniform(0.1, 1.0, len(idx)).astype(np.float32), b_off, b_idx, b_val)
    gc = apoe.Corpus(gpu_ctx, *arrays)
    assert gc.pair_bytes() == 6
    ids = np.stack([rng.choice(n, K, replace=False) for _ in range(n)]).astype(np.uint32)
    step_equals_oracle(gpu_ctx, gc, O.HybridSet(*arrays), ids, K)
    gc.close()
