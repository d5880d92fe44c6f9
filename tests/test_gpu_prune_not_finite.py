"""Values that are infinite, no numbers, or so large that a norm overflows, in terms that rows of one list share: the selection takes
the products that do not involve them as they are, in each form of the prune."""
import numpy as np
import pytest

from test_gpu_prune_ties import equal_but_for_ties

pytestmark = pytest.mark.gpu
N = 1200


def world(wide):
    import apoe_synth as S
    import oracle as O
    a = list(S.to_numpy(S.corpus(N, seed=23, device="cpu")))
    if wide:
        a[5] = a[5] + np.uint32(70000)
    return a, O.HybridSet(*a)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("place", [0.0, 0.1, 0.3])
@pytest.mark.parametrize("K,degree", [(64, 32), (128, 48)])
def test_prune_matches_oracle(gpu_ctx, K, degree, place, wide):
    import apoe
    import oracle as O
    a, clean = world(wide)
    ids, dist = O.bruteforce_knn_self(clean, 7.0, K)
    # the documents that most lists name; in each one SPLADE and one BM25 value changes, of a term that many rows hold, several, or few
    # (term ids are frequency ranks)
    named = np.argsort(-np.bincount(ids.ravel(), minlength=N), kind="stable")[:24]
    for kind, doc in zip(np.tile([np.inf, -np.inf, np.nan, 3e25], 6), named):
        for off, idx, val in ((a[1], a[2], a[3]), (a[4], a[5], a[6])):
            lo, hi = int(off[doc]), int(off[doc + 1])
            if hi > lo:
                val[lo + np.argsort(idx[lo:hi])[int(place * (hi - lo))]] = kind
    C = O.HybridSet(*a)
    norms = O.norms(C, 7.0)
    assert np.sum(~np.isfinite(norms)) >= 20
    c_fwd, c_det, c_cnt, c_kw = O.prune(C, 7.0, norms, ids, dist, degree)
    gc = apoe.Corpus(gpu_ctx, *a)
    knn = apoe.Knn(gpu_ctx, gc, K, 7.0)
    knn.upload(ids, dist)
    for form in (0, 1):
        knn.set_prune_form(form)
        knn.prune(degree)
        equal_but_for_ties(a, 7.0, ids, dist, knn.prune_download(), (c_fwd, c_det, c_cnt, c_kw))
    knn.close()
    gc.close()
