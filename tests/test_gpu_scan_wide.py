"""Child scans of the wide layout (k_pair_scan_wide): features of 1 to 256 bins side by side,
an odd number of them, most frequent bins at either end and between, children too small to
split, against the oracle.  Bar: quantized trees bit-exact; f32 ones equal in structure,
leaf values within 1e-9 (one rounding of a fixed-point sum a cell against the f64 fold)."""
import numpy as np
import pytest

from lightgbm_rs_amd import GainConfig, HipBackend, feature_meta
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant", [True, False])
@pytest.mark.parametrize("n,F,leaves,min_data", [(300, 125, 15, 5), (5000, 131, 63, 1),
                                                 (20_000, 200, 40, 50)])
def test_trees_match_the_oracle(n, F, leaves, min_data, quant):
    print(f"wide scans n={n} F={F} quant={quant}", flush=True)
    rng = np.random.default_rng(n + F)
    nb = rng.integers(1, 257, F)
    nb[:8] = [1, 2, 3, 64, 65, 66, 255, 256]
    bins = np.stack([np.minimum(rng.geometric(min(1.0, 4 / k), n) - 1, k - 1) if f % 2
                     else rng.integers(0, k, n) for f, k in enumerate(nb)]).astype(np.uint8)
    mfb = [0 if f % 4 == 0 else int(k) - 1 if f % 4 == 2 else int(np.bincount(b).argmax())
           for f, (k, b) in enumerate(zip(nb, bins))]
    meta = [feature_meta(int(k), m, 0, m, f) for f, (k, m) in enumerate(zip(nb, mfb))]
    upper = np.concatenate([np.append(np.arange(k - 1) + 0.5, np.inf) for k in nb])
    z = (bins[3:9] / nb[3:9, None]).sum(0) + rng.normal(0, 0.5, n)
    grad = (z - z.mean()).astype(np.float32)
    hess = rng.uniform(0.1, 1.0, n).astype(np.float32)
    cfg = GainConfig.make(min_data_in_leaf=min_data)
    be = HipBackend(0)
    be.upload_resident_bins(bins, meta, upper)
    be.upload_resident_grad_hess(grad, hess)
    if quant:
        _, grad, hess = be.discretize_dequantize_in_place(4, True, 3, want_values=True)
    t, layout = be.grow_tree_on_device_with_cfg(cfg, leaves)
    be.close()
    ref, ref_layout = oracle.train_tree(bins, meta, upper, grad, hess, cfg, leaves, -1)
    assert t["num_leaves"] == ref["num_leaves"] > 2
    for k in ("split_feature", "threshold_in_bin", "left_child", "right_child", "leaf_count"):
        assert np.array_equal(t[k], ref[k]), k
    assert np.array_equal(layout["indices"], ref_layout["indices"])
    if quant:
        for k in ("leaf_value", "leaf_weight", "internal_value"):
            assert np.array_equal(t[k].view(np.uint64), ref[k].view(np.uint64)), k
    else:
        np.testing.assert_allclose(t["leaf_value"], ref["leaf_value"], rtol=1e-9, atol=1e-12)
