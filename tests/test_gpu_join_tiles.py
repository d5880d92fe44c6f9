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
