"""f32 children of the wide layout whose histogram is one row chunk or several, at the edge
of a chunk, in both child scans.  The first split parts off `small` rows and the next ones
split either side, so the children's cells are read again as a parent's.  Bar: structure
equal to the oracle's, leaf values within 1e-9 (one rounding of a fixed-point sum a cell
against the f64 fold)."""
import numpy as np
import pytest

from lightgbm_rs_amd import GainConfig, HipBackend, feature_meta
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("categorical", [False, True])  # True: the scans take k_pair_scan
@pytest.mark.parametrize("small", [1, 4095, 4096, 4097, 8193])
def test_small_child_at_a_chunks_edge(small, categorical):
    n, F = 20_000, 130
    print(f"wide chunks small={small} categorical={categorical}", flush=True)
    rng = np.random.default_rng(small)
    bins = rng.integers(0, 256, (F, n)).astype(np.uint8)
    part = np.zeros(n, np.uint8)
    part[rng.permutation(n)[:small]] = 1
    bins[0] = part
    nb = np.full(F, 256)
    nb[0] = 2
    if categorical:
        nb[F - 1] = 33
        bins[F - 1] = rng.integers(1, 33, n)
    types = [1 if categorical and f == F - 1 else 0 for f in range(F)]
    meta = [feature_meta(int(nb[f]), types[f], 0, types[f], f, bin_type=types[f]) for f in range(F)]
    upper = np.concatenate([np.arange(-1, k - 1) if t else np.append(np.arange(k - 1) + 0.5, np.inf)
                            for k, t in zip(nb, types)]).astype(np.float64)
    z = 40.0 * part + (bins[1:4] / 256).sum(0) + rng.normal(0, 0.3, n)
    grad = (z - z.mean()).astype(np.float32)
    hess = rng.uniform(0.5, 1.0, n).astype(np.float32)
    cfg = GainConfig.make(min_data_in_leaf=1)
    be = HipBackend(0)
    be.upload_resident_bins(bins, meta, upper)
    be.upload_resident_grad_hess(grad, hess)
    t, layout = be.grow_tree_on_device_with_cfg(cfg, 16)
    be.close()
    ref, ref_layout = oracle.train_tree(bins, meta, upper, grad, hess, cfg, 16, -1)
    assert t["split_feature"][0] == 0 and t["num_leaves"] == ref["num_leaves"] == 16
    for k in ("split_feature", "threshold_in_bin", "left_child", "right_child", "leaf_count"):
        assert np.array_equal(t[k], ref[k]), k
    assert np.array_equal(layout["indices"], ref_layout["indices"])
    np.testing.assert_allclose(t["leaf_value"], ref["leaf_value"], rtol=1e-9, atol=1e-12)
