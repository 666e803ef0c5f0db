"""Prediction from trees and rows in LDS (k_predict_lds): its block shapes (1024 rows a
block down to 8, several trees side by side), packed thresholds, default directions and
categorical nodes, from dense and CSR rows.  Bar: f64 bits and leaves equal to the oracle's
walk of the same model text."""
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


def _text(rng, leaves, cols, classes, iters, cat, infinite=False):
    out = ["tree", "version=v4", f"num_class={classes}", f"num_tree_per_iteration={classes}",
           "label_index=0", f"max_feature_idx={cols - 1}",
           "objective=" + (f"multiclass num_class:{classes}" if classes > 1 else "binary sigmoid:1"),
           "feature_names=" + " ".join(f"c{i}" for i in range(cols)),
           "feature_infos=" + " ".join(["none"] * cols), ""]

    def line(k, v):
        out.append(f"{k}=" + " ".join(map(repr, np.asarray(v).tolist())))

    for t in range(classes * iters):
        nl = leaves if t != 1 else 1
        left, right, at = [], [], [None]
        for node in range(nl - 1):
            leaf = int(rng.integers(len(at)))
            if at[leaf] is not None:
                at[leaf][0][at[leaf][1]] = node
            left.append(~leaf)
            right.append(~len(at))
            at.append((right, node))
            at[leaf] = (left, node)
        thr = rng.normal(size=nl - 1)
        thr[::5] = 0.0
        thr[1::7] = np.float32(0.5)
        if infinite:
            thr[2::9] = np.inf
        dt = rng.choice([0, 2, 4, 6, 8, 10], nl - 1)
        is_cat = (rng.random(nl - 1) < 0.3) if cat else np.zeros(nl - 1, bool)
        dt[is_cat] = 1
        thr[is_cat] = np.arange(is_cat.sum())
        out += [f"Tree={t}", f"num_leaves={nl}", f"num_cat={int(is_cat.sum())}"]
        if nl > 1:
            line("split_feature", rng.integers(0, cols, nl - 1))
            line("threshold", thr)
            line("decision_type", dt)
            line("left_child", left)
            line("right_child", right)
        line("leaf_value", rng.normal(size=nl))
        if is_cat.any():
            line("cat_boundaries", np.arange(is_cat.sum() + 1) * 2)
            line("cat_threshold", rng.integers(0, 1 << 32, 2 * int(is_cat.sum())))
        out += ["is_linear=0", "shrinkage=1", "", ""]
    return "\n".join(out + ["end of trees", ""])


def _rows(rng, rows, cols):
    """Values at, just above and just below the f32 thresholds, zeros, tiny and special ones."""
    X = rng.normal(size=(rows, cols)).astype(np.float32)
    at = rng.random(X.shape)
    for k, v in enumerate((np.nan, 0.0, -0.0, 0.5, np.nextafter(np.float32(0.5), np.float32(1)),
                           1e-35, -1e-35, 2e-35, np.inf, -np.inf, 3.0, 40.0, -2.0)):
        X[(at >= 0.03 * k) & (at < 0.03 * (k + 1))] = v
    return X


# (rows, repeats of them, columns, leaves, classes, iterations, categorical): repeats bring
# the rows to the sizes at which a block takes 1024, 512, .. rows, columns to those at
# which LDS holds fewer
@pytest.mark.parametrize("rows,repeat,cols,leaves,classes,iters,cat", [
    (1, 1, 4, 31, 1, 3, False), (9, 1, 1, 2, 3, 5, False), (50, 1, 28, 31, 1, 40, True),
    (101, 2600, 28, 255, 1, 3, False), (101, 1300, 9, 15, 2, 4, True),
    (101, 700, 66, 31, 1, 9, False), (64, 300, 501, 63, 10, 2, True),
    (33, 5, 1100, 40, 1, 6, False), (17, 1, 3900, 31, 1, 5, True),
    (40, 1, 5, 1300, 1, 3, False)])
def test_bits_equal_the_oracle(be, rows, repeat, cols, leaves, classes, iters, cat):
    rng = np.random.default_rng(rows * 7 + cols)
    text = _text(rng, leaves, cols, classes, iters, cat)
    m, pm = Model(text), P.parse_model(text)
    X = _rows(rng, rows, cols)
    big = np.tile(X, (repeat, 1))
    sparse = X.copy()
    sparse[rng.random(X.shape) < 0.5] = 0.0
    r, c = np.nonzero((sparse != 0) | np.isnan(sparse))
    ends = np.cumsum(np.bincount(r, minlength=rows))
    for kind in ("raw", "transformed", "leaf"):
        print(f"predict rows={len(big)} cols={cols} leaves={leaves} kind={kind}", flush=True)
        ref = np.asarray(P.predict(pm, X, kind=kind))
        got = be.predict(m, big, kind)
        if kind == "transformed":  # exp on the host and on the device
            np.testing.assert_allclose(got, np.tile(ref, (repeat, 1)), rtol=1e-14, atol=0)
        else:
            assert np.array_equal(got, np.tile(ref.reshape(rows, -1), (repeat, 1)))
        got = be.predict_csr(m, np.concatenate([[0], ends]), c, sparse[r, c], cols, kind)
        assert np.array_equal(got, be.predict(m, sparse, kind))
        part = be.predict(m, X, kind, start_iteration=1, num_iteration=1)
        ref = np.asarray(P.predict(pm, X, 1, 1, kind))
        np.testing.assert_allclose(part, ref.reshape(rows, -1), rtol=1e-14, atol=0)


# Calls just past what the packed trees or the block's LDS take (leaves, columns, an infinite
# threshold, wide rows beside a large tree) and one of few trees over wide rows: k_predict's.
@pytest.mark.parametrize("rows,cols,leaves,iters,infinite", [
    (40, 5, 1365, 2, False), (40, 5, 1366, 2, False), (30, 4096, 31, 4, False),
    (30, 4097, 31, 4, False), (20, 5001, 15, 3, False), (90, 12, 31, 5, True),
    (20, 4000, 900, 2, False), (300, 1000, 31, 1, False)])
def test_either_side_of_a_limit(be, rows, cols, leaves, iters, infinite):
    rng = np.random.default_rng(rows + cols)
    text = _text(rng, leaves, cols, 1, iters, False, infinite)
    m, pm = Model(text), P.parse_model(text)
    X = _rows(rng, rows, cols)
    sparse = X.copy()
    sparse[rng.random(X.shape) < 0.5] = 0.0
    r, c = np.nonzero((sparse != 0) | np.isnan(sparse))
    ends = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=rows))])
    for kind in ("raw", "leaf"):
        print(f"predict limit cols={cols} leaves={leaves} kind={kind}", flush=True)
        ref = np.asarray(P.predict(pm, X, kind=kind)).reshape(rows, -1)
        assert np.array_equal(be.predict(m, X, kind), ref)
        ref = np.asarray(P.predict(pm, sparse, kind=kind)).reshape(rows, -1)
        assert np.array_equal(be.predict_csr(m, ends, c, sparse[r, c], cols, kind), ref)


@pytest.mark.parametrize("rows,extra", [(1, 1), (70, 3), (70, 972), (3000, 972), (270_000, 9)])
def test_rows_wider_than_the_model(be, rows, extra):
    """Columns past max_feature_idx, which no tree reads."""
    rng = np.random.default_rng(rows + extra)
    text = _text(rng, 31, 28, 2, 20, True)
    m, pm = Model(text), P.parse_model(text)
    X = _rows(rng, min(rows, 70), 28)
    ref = np.asarray(P.predict(pm, X, kind="raw"))
    big = np.full((rows, 28 + extra), np.nan, np.float32)
    big[:, :28] = np.resize(X, (rows, 28))
    print(f"predict rows={rows} extra={extra}", flush=True)
    assert np.array_equal(be.predict(m, big, "raw"), np.resize(ref.reshape(len(X), -1), (rows, 2)))
