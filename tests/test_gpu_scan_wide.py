"""Child scans of the wide layout (k_pair_scan_wide): features of 1 to 256 bins side by side,
an odd number of them, most frequent bins at either end and between, children too small to
split, more than 64 feature groups of histograms, against the oracle.  Bar: quantized trees bit-exact; f32 ones equal in structure,
leaf values within 1e-9 (one rounding of a fixed-point sum a cell against the f64 fold)."""
import numpy as np
import pytest

from lightgbm_rs_amd import GainConfig, HipBackend, feature_meta
from oracle import oracle

pytestmark = pytest.mark.gpu


def _table(n, F):
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
    return bins, meta, upper, grad, hess


def _check(n, F, leaves, quant, cfg, max_depth=-1, contri=None):
    bins, meta, upper, grad, hess = _table(n, F)
    be = HipBackend(0)
    be.upload_resident_bins(bins, meta, upper)
    if contri is not None:
        be.set_feature_contri(contri)
    be.upload_resident_grad_hess(grad, hess)
    if quant:
        _, grad, hess = be.discretize_dequantize_in_place(4, True, 3, want_values=True)
    t, layout = be.grow_tree_on_device_with_cfg(cfg, leaves, max_depth)
    be.close()
    ref, ref_layout = oracle.train_tree(bins, meta, upper, grad, hess, cfg, leaves, max_depth,
                                        feature_contri=contri)
    assert t["num_leaves"] == ref["num_leaves"] > 2
    for k in ("split_feature", "threshold_in_bin", "left_child", "right_child", "leaf_count"):
        assert np.array_equal(t[k], ref[k]), k
    assert np.array_equal(layout["indices"], ref_layout["indices"])
    if quant:
        for k in ("leaf_value", "leaf_weight", "internal_value"):
            assert np.array_equal(t[k].view(np.uint64), ref[k].view(np.uint64)), k
    else:
        np.testing.assert_allclose(t["leaf_value"], ref["leaf_value"], rtol=1e-9, atol=1e-12)


@pytest.mark.parametrize("quant", [True, False])
@pytest.mark.parametrize("n,F,leaves,min_data", [(300, 125, 15, 5), (5000, 131, 63, 1),
                                                 (20_000, 200, 40, 50), (3000, 2100, 15, 5)])
def test_trees_match_the_oracle(n, F, leaves, min_data, quant):
    print(f"wide scans n={n} F={F} quant={quant}", flush=True)
    _check(n, F, leaves, quant, GainConfig.make(min_data_in_leaf=min_data))


# the terms of a candidate's gain beyond the plain quotient, one by one and together
@pytest.mark.parametrize("quant", [True, False])
@pytest.mark.parametrize("max_depth,contri,terms", [
    (-1, False, dict(lambda_l1=3.0)), (-1, False, dict(lambda_l2=20.0)),
    (-1, False, dict(max_delta_step=0.1)), (-1, False, dict(path_smooth=30.0)),
    (-1, False, dict(min_gain_to_split=25.0)), (-1, False, dict(min_sum_hessian_in_leaf=60.0)),
    (3, False, dict()), (-1, True, dict()),
    (6, True, dict(lambda_l1=0.5, lambda_l2=2.0, max_delta_step=0.3, path_smooth=5.0,
                   min_gain_to_split=0.1))])
def test_gain_terms(max_depth, contri, terms, quant):
    print(f"wide scans {terms} max_depth={max_depth} contri={contri} quant={quant}", flush=True)
    c = np.random.default_rng(1).uniform(0.2, 1.0, 131) if contri else None
    _check(5000, 131, 31, quant, GainConfig.make(min_data_in_leaf=20, **terms), max_depth, c)
