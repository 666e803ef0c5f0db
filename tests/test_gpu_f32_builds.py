"""f32-gradient trees in the record layouts around the sizes at which a child's histogram is
built elsewhere: by the scan itself (small children; all of them up to
HIST_FP_ALL_DIRECT = 8192 rows), in partial slots, and through the job's accumulator (more
than HIST_FP_SLOTS = 8 chunks of 1024 rows), with one and with several feature groups.
Bar: the oracle's splits and counts, leaf values within 1e-9 (one rounding of a fixed-point
sum a cell against the f64 fold)."""
import numpy as np
import pytest

from lightgbm_rs_amd import GainConfig, HipBackend, feature_meta
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,F,max_bin,leaves", [
    (40, 3, 15, 4), (3000, 7, 255, 31), (8192, 5, 63, 31), (8193, 5, 63, 31),
    (9001, 31, 255, 63), (60_000, 29, 255, 31), (300_000, 12, 255, 15),
    (250_000, 39, 63, 15), (30_000, 100, 80, 31)])
def test_trees_match_the_oracle(n, F, max_bin, leaves):
    print(f"f32 builds n={n} F={F} max_bin={max_bin}", flush=True)
    rng = np.random.default_rng(n + F)
    nb = rng.integers(2, max_bin + 1, F)
    nb[0] = max_bin
    bins = np.stack([rng.integers(0, k, n) for k in nb]).astype(np.uint8)
    mfb = [int(np.bincount(b).argmax()) if i % 3 else 0 for i, b in enumerate(bins)]
    meta = [feature_meta(int(k), m, 0, m, f) for f, (k, m) in enumerate(zip(nb, mfb))]
    upper = np.concatenate([np.append(np.arange(k - 1) + 0.5, np.inf) for k in nb])
    z = (bins[:3] / nb[:3, None]).sum(0) + rng.normal(0, 0.3, n)
    grad = (z - z.mean()).astype(np.float32)
    hess = rng.uniform(0.1, 1.0, n).astype(np.float32)
    cfg = GainConfig.make(min_data_in_leaf=5)
    be = HipBackend(0)
    be.upload_resident_bins(bins, meta, upper)
    ref, ref_layout = oracle.train_tree(bins, meta, upper, grad, hess, cfg, leaves, -1)
    be.upload_resident_grad_hess(grad, hess)
    for _ in range(2):  # the second tree finds what the first one left in the accumulators
        t, layout = be.grow_tree_on_device_with_cfg(cfg, leaves)
        assert t["num_leaves"] == ref["num_leaves"]
        for k in ("split_feature", "threshold_in_bin", "left_child", "right_child", "leaf_count"):
            assert np.array_equal(t[k], ref[k]), k
        np.testing.assert_allclose(t["leaf_value"], ref["leaf_value"], rtol=1e-9, atol=1e-12)
        assert np.array_equal(layout["indices"], ref_layout["indices"])
    be.close()
