"""Feature contributions by leaf paths (k_shap_items / k_shap_rows) and the choice between
them and the one-thread-per-row kernel.  Bar: f64 bits equal to the oracle's recursion.

Trees are random with repeated features on their paths, from balanced ones to a chain of
SHAP_MAX_DEPTH = 31 levels (the deepest the leaf paths take) and one level more, and of up
to SHAP_MAX_LEAVES = 908 leaves and one more; rows from fewer than any leaf's outcomes
(items are rows) to more (items are outcomes), and so many that the values are cut into
runs of trees, chunks of rows, or k_contrib's chunks."""
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


# the widest trees of one feature and of 28 whose rows fit k_shap_rows's LDS, and one leaf more
@pytest.mark.parametrize("leaves,cols", [(908, 1), (909, 1), (884, 28), (885, 28)])
def test_either_side_of_the_leaf_limit(be, leaves, cols):
    rng = np.random.default_rng(leaves)
    m = Model.create(num_class=1, max_feature_idx=cols - 1)
    m.add_tree(_tree(rng, leaves, cols, False))
    print(f"contrib leaves={leaves} cols={cols}", flush=True)
    X = rng.normal(size=(3, cols)).astype(np.float32)
    got, ref = be.predict(m, X, "contrib"), P.predict_contrib(P.parse_model(m.to_text()), X)
    assert np.array_equal(got.view(np.uint64), np.ascontiguousarray(ref).view(np.uint64))


VALUES = 1 << 25  # of a launch of k_shap_items


def _comb(rng, leaves, cols, spine):
    """A chain of `spine` levels above a random subtree of the other leaves."""
    t, sub = _tree(rng, leaves, cols, True), _tree(rng, leaves - spine, cols, False)
    for side in ("left_child", "right_child"):
        t[side] = np.concatenate([t[side][:spine],
                                  [k + spine if k >= 0 else ~(~k + spine) for k in sub[side]]])
    return t


def _paths(t):
    """(depth, length of the unique path) of every leaf."""
    out, todo = [], [(0, ())]
    while todo:
        node, feats = todo.pop()
        if node < 0:
            out.append((len(feats), len(set(feats))))
            continue
        feats += (int(t["split_feature"][node]),)
        todo += [(int(t["left_child"][node]), feats), (int(t["right_child"][node]), feats)]
    return out


def _values(t, rows):
    return sum(min(rows, 2 ** d) * m for d, m in _paths(t))


def _check_slices(be, m, X, starts):
    got = be.predict(m, X, "contrib")
    pm = P.parse_model(m.to_text())
    for r0 in starts:
        sl = slice(r0, r0 + 6)
        ref = np.ascontiguousarray(P.predict_contrib(pm, X[sl]))
        assert np.array_equal(got[sl].view(np.uint64), ref.view(np.uint64)), r0


def test_trees_in_two_runs(be):
    """The second run goes on from the first one's sums, within an iteration of three classes."""
    rng, rows, cols = np.random.default_rng(1), 20_000, 12
    m = Model.create(num_class=3, max_feature_idx=cols - 1)
    trees = [_tree(rng, 32, cols, True) for _ in range(9)]
    for t in trees:
        m.add_tree(t)
    sizes = [_values(t, rows) for t in trees]
    first = next(i for i in range(9) if sum(sizes[:i + 1]) > VALUES)
    assert max(sizes) <= VALUES and 0 < first < 9 and first % 3
    print(f"contrib runs of {first} and {9 - first} trees", flush=True)
    X = rng.normal(size=(rows, cols)).astype(np.float32)
    _check_slices(be, m, X, (0, 9_000, rows - 6))


def test_rows_in_chunks(be):
    """A tree whose values of all rows are too many: chunks of rows, the last one shorter
    than the items that the plan has for a chunk."""
    rng, rows, cols = np.random.default_rng(2), 40_001, 24
    m = Model.create(num_class=1, max_feature_idx=cols - 1)
    trees = [_comb(rng, 200, cols, 13), _tree(rng, 20, cols, False)]
    for t in trees:
        m.add_tree(t)
    assert max(d for d, _ in _paths(trees[0])) <= 31
    chunk = rows
    while max(_values(t, chunk) for t in trees) > VALUES:
        chunk = (chunk + 1) // 2
    assert 0 < rows % chunk and rows > 2 * chunk and any(2 ** d > chunk for d, _ in _paths(trees[0]))
    print(f"contrib chunks of {chunk} of {rows} rows", flush=True)
    X = rng.normal(size=(rows, cols)).astype(np.float32)
    _check_slices(be, m, X, (0, chunk - 3, 2 * chunk - 3, rows - 6))


def test_k_contrib_in_two_chunks(be):
    """A tree deeper than the leaf paths take, over more rows than its path workspace holds."""
    rng, cols, depth = np.random.default_rng(3), 12, 32
    per_row = (depth + 1) * (depth + 2) // 2 * 28 + (depth + 1) * 24
    chunk = (256 << 20) // per_row // 256 * 256
    m = Model.create(num_class=1, max_feature_idx=cols - 1)
    for leaves in (depth + 1, 9):
        m.add_tree(_tree(rng, leaves, cols, True))
    print(f"contrib deep chunks of {chunk} rows", flush=True)
    X = rng.normal(size=(chunk + 500, cols)).astype(np.float32)
    _check_slices(be, m, X, (0, chunk - 3, chunk + 494))


def test_ranges_of_one_model(be):
    """Calls of ranges within, across and beyond the trees whose paths are there already."""
    rng, cols, classes = np.random.default_rng(5), 6, 2
    m = Model.create(num_class=classes, max_feature_idx=cols - 1)
    for i in range(6 * classes):
        m.add_tree(_tree(rng, int(rng.integers(1, 25)), cols, i == 7))
    pm = P.parse_model(m.to_text())
    X = rng.normal(size=(9, cols)).astype(np.float32)
    for start, num in ((3, 1), (3, 1), (2, 3), (3, 2), (0, 1), (4, 2), (0, -1), (1, 4), (5, 1)):
        print(f"contrib iterations from {start}, {num}", flush=True)
        got = be.predict(m, X, "contrib", start_iteration=start, num_iteration=num)
        ref = np.ascontiguousarray(P.predict_contrib(pm, X, start_iteration=start, num_iteration=num))
        assert np.array_equal(got.view(np.uint64), ref.view(np.uint64))
