"""One long row in a K = 64 corpus: as long as the rank table beside the Gram matrix holds it, the prune gathers every row once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("longest", [1100, 1160, 1216])
def test_gathered_form_runs(gpu_ctx, longest):
    import apoe
    import apoe_synth as S
    n, row = 3000, 17
    dense, s_off, s_idx, s_val, b_off, b_idx, b_val = S.to_numpy(S.corpus(n, seed=5, device="cpu"))
    assert 96 < np.diff(b_off.astype(np.int64)).max() <= 128 and 16384 <= max(s_idx.max(), b_idx.max()) < 32768  # what the table shares its LDS with
    rng = np.random.default_rng(longest)
    cnt = np.diff(s_off.astype(np.int64))
    cnt[row] = longest - np.diff(b_off.astype(np.int64)).max()
    off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.uint32)
    keep = lambda a, new: np.concatenate([a[:s_off[row]], new, a[s_off[row + 1]:]]).astype(a.dtype)
    gc = apoe.Corpus(gpu_ctx, dense, off, keep(s_idx, np.sort(rng.choice(30000, cnt[row], replace=False))), keep(s_val, rng.uniform(0.1, 0.4, cnt[row])),
                     b_off, b_idx, b_val)
    knn = apoe.Knn(gpu_ctx, gc, 64, 7.0)
    knn.set_join(1)
    knn.init(1)
    for it in range(5):
        knn.iterate(last=(it == 4))
    knn.merge_reverse()
    ms, rows = [], []
    for form in (0, 1, 0):
        knn.set_prune_form(form)
        t0 = knn.elapsed_ms()
        knn.prune(32)
        ms.append(knn.elapsed_ms() - t0)
        rows.append(knn.prune_download()[0])
    knn.close()
    gc.close()
    assert np.all(rows[0] == rows[1], axis=1).mean() >= 0.99 and np.array_equal(rows[0], rows[2])
    assert ms[2] < 0.5 * ms[1], ms  # reading every row again at every step of the selection is several times slower
