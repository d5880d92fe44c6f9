"""A join step twice from the same lists, with picked nodes of many more pickers than a tile has rows: which pickers share a tile is up to the
order in which they arrive, and neither an id nor a bit of a distance may depend on it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pickers", [33, 45, 250, 4000])
@pytest.mark.parametrize("K", [64, 128])
def test_same_lists_same_bits(gpu_ctx, small_world, pickers, K):
    import apoe
    n = small_world["C"].n
    rng = np.random.default_rng(pickers)
    gc = apoe.Corpus(gpu_ctx, *small_world["corpus"])
    ids = np.stack([rng.choice(n, K, replace=False) for _ in range(n)]).astype(np.uint32)
    ids[:, :4] = 4 * (np.arange(n) // pickers)[:, None] % (n - 4) + np.arange(4)
    # a last entry that between none and half of a row's columns beat
    at = rng.integers(0, n, (n, 64)).astype(np.uint32)
    d = apoe.distance_pairs(gpu_ctx, gc, 7.0, np.repeat(np.arange(n, dtype=np.uint32), 64), at.ravel()).reshape(n, 64)
    worst = np.sort(d, axis=1)[np.arange(n), rng.integers(1, 32, n)]
    dist = (worst[:, None] + np.linspace(-2, 0, K)).astype(np.float32)
    runs = []
    for _ in range(4):
        knn = apoe.Knn(gpu_ctx, gc, K, 7.0)
        knn.upload(ids, dist)  # saved lists: the step asks the sketches
        knn.set_join(1)
        assert knn.iterate(last=True) > 0
        runs.append(knn.download())
        knn.close()
    gc.close()
    for got, gd in runs[1:]:
        assert np.array_equal(got, runs[0][0])
        assert np.array_equal(gd.view(np.uint32), runs[0][1].view(np.uint32))
