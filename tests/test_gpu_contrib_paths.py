"""Feature contributions by leaf paths (k_shap_items / k_shap_rows) and the choice between
them and the one-thread-per-row kernel.  Bar: f64 bits equal to the oracle's recursion.

Trees are random with repeated features on their paths, from balanced ones to a chain of
SHAP_MAX_DEPTH = 31 levels (the deepest the leaf paths take) and one level more; rows from
fewer than any leaf's outcomes (items are rows) to more (items are outcomes)."""
import numpy as np
import pytest

from lightgbm_rs_amd import HipBackend, Model
from oracle import predict as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    b = HipBackend(0)
    yield b
    b.close()


def _tree(rng, leaves, cols, chain):
    left, right, at, depth = [], [], [None], [0]
    for node in range(leaves - 1):
        leaf = len(at) - 1 if chain else int(rng.integers(len(at)))
        if at[leaf] is not None:
            side, parent = at[leaf]
            side[parent] = node
        left.append(~leaf)
        right.append(~len(at))
        at.append((right, node))
        at[leaf] = (left, node)
    n = leaves - 1
    count = rng.integers(1, 50, leaves).astype(np.int32)
    cover = np.zeros(n, np.int32)
    for i in range(n - 1, -1, -1):
        cover[i] = sum(cover[k] if k >= 0 else count[~k] for k in (left[i], right[i]))
    return dict(num_leaves=leaves, split_feature=rng.integers(0, cols, n).astype(np.int32),
                threshold=rng.normal(size=n), left_child=np.array(left, np.int32),
                decision_type=rng.choice([0, 2, 4, 6, 8, 10], n).astype(np.int8),
                right_child=np.array(right, np.int32), internal_count=cover,
                leaf_value=rng.normal(size=leaves), leaf_count=count)


# (leaves, columns, classes, chain): short and long unique paths, one leaf, several
# classes, rows of many columns (fewer rows a block), depths 31 and 32
@pytest.mark.parametrize("leaves,cols,classes,chain", [
    (1, 3, 1, False), (2, 1, 1, False), (9, 2, 3, False), (40, 6, 1, False),
    (40, 40, 2, False), (20, 700, 1, False), (32, 12, 1, True), (32, 60, 1, True),
    (33, 12, 1, True)])
def test_bits_equal_the_recursion(be, leaves, cols, classes, chain):
    rng = np.random.default_rng(leaves * 1000 + cols)
    m = Model.create(num_class=classes, max_feature_idx=cols - 1)
    for i in range(3 * classes):
        m.add_tree(_tree(rng, leaves if i != classes else 1, cols, chain))
    pm = P.parse_model(m.to_text())
    for rows in (1, 7, 70):
        print(f"contrib leaves={leaves} cols={cols} classes={classes} rows={rows}", flush=True)
        X = rng.normal(size=(rows, cols)).astype(np.float32)
        X[rng.random(X.shape) < 0.1] = np.nan
        X[rng.random(X.shape) < 0.1] = 0.0
        got, ref = be.predict(m, X, "contrib"), P.predict_contrib(pm, X)
        assert np.array_equal(got.view(np.uint64), np.ascontiguousarray(ref).view(np.uint64))


# Each leaf of a chain whose nodes take the features in turn has the features of the leaf
# before it one position (and so one lane of k_shap_rows) further on: every add follows
# another lane's to the same sum.
@pytest.mark.parametrize("cols", [2, 3, 8, 9, 16])
def test_consecutive_leaves_meet_the_same_features(be, cols):
    rng = np.random.default_rng(cols)
    m = Model.create(num_class=1, max_feature_idx=cols - 1)
    for _ in range(3):
        t = _tree(rng, 30, cols, True)
        t["split_feature"] = (np.arange(29) % cols).astype(np.int32)
        m.add_tree(t)
    print(f"contrib rotating features cols={cols}", flush=True)
    X = rng.normal(size=(70, cols)).astype(np.float32)
    got, ref = be.predict(m, X, "contrib"), P.predict_contrib(P.parse_model(m.to_text()), X)
    assert np.array_equal(got.view(np.uint64), np.ascontiguousarray(ref).view(np.uint64))
