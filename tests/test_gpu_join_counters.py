"""What the join steps of a build say they read: every row and column of a tile in full while the lists change, and once they have settled
(less than a twelfth of a step's pairs entered a list) a sketch for each and the dense rows of the columns that stay open only."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [64, 128])
def test_settled_steps_read_fewer_dense_rows(gpu_ctx, K):
    import apoe
    import apoe_synth as S
    gc = apoe.Corpus(gpu_ctx, *S.to_numpy(S.latent_corpus(3000, seed=31, device="cpu")))
    knn = apoe.Knn(gpu_ctx, gc, K, 7.0)
    knn.set_join(1)
    knn.init(1)
    settled, seen, before = False, set(), (0, 0, 0, 0)
    for it in range(10):
        inserted = knn.iterate(last=(it == 9))
        now = (knn.counters()[0], *knn.read_counters())
        assert knn.counters()[1] == now[1]
        evals, dense, pair_rows, sketches = (a - b for a, b in zip(now, before))
        assert evals > 0 and pair_rows > 0
        if settled:
            assert sketches == pair_rows and 0 < dense < pair_rows
        else:
            assert sketches == 0 and dense == pair_rows
        seen.add(settled)
        settled, before = inserted * 12 < evals, now
    assert seen == {False, True}
    assert dense < 0.8 * pair_rows  # the last step: few columns stay open
    knn.set_join(0)  # an expansion step reads the pairs of every evaluation
    knn.iterate(last=True)
    now = (knn.counters()[0], *knn.read_counters())
    evals, dense, pair_rows, sketches = (a - b for a, b in zip(now, before))
    assert sketches == 0 and pair_rows == evals >= dense > 0
    knn.close()
    gc.close()
