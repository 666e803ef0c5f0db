"""The work that a user of this package has it do, as cases to be timed and checked.

A case is a dict of plain values.  `listed()` names the fixed ones and `draw()` gives more
of the same ranges; `prepare()` makes what a program holds before the call, `run()` is one
pass through the public entry points, `exact()` the same outputs in 64 bits without this
package, `work()` the bytes and operations the pass cannot do without, `tolerance()` how
far two correct implementations may be apart.

Kinds of case:
  train    boosting on resident bins that the program made: labels in, `iters`
           iterations, every tree and the training scores out (a pass starts from the
           labels, so it can be repeated)
  fit      the same from a raw float32 table on the device: binning, then boosting
  seam     one tree for a host boosting loop: host gradients in, the quantized tree and
           the row layout out (the reference's whole-tree `Backend` call)
  predict  a forest over host rows, device rows or a host CSR matrix: raw scores, the
           objective's outputs, leaf indices or TreeSHAP contributions

Tables are synthetic: N(0, 1) columns, or LogNormal(0, 1) where a column is mostly zeros,
with a share of NaN where a case says so and categorical columns of equally likely levels
at the end.
"""
import math

import numpy as np
import torch

from lightgbm_rs_amd import (BinMapper, GainConfig, HipBackend, Model, boost_from_score,
                             feature_meta, sample_indices)

DEVICE = "cuda:0"
LEARNING_RATE = 0.1
MIN_DATA = 20
MIN_HESSIAN = 1e-3
BIN_SAMPLE = 20000  # bin_construct_sample_cnt: rows a mapper is made from
COL_SEED = 2        # feature_fraction_seed
EPS = float(np.float32(1e-15))

TREE_FIELDS = ("split_feature", "threshold_in_bin", "threshold", "split_gain", "decision_type",
               "left_child", "right_child", "internal_value", "internal_count",
               "internal_weight", "leaf_value", "leaf_weight", "leaf_count", "leaf_depth",
               "leaf_parent", "cat_boundaries", "cat_threshold")

# every value a training case reads, with the usual choice
TRAIN = dict(kind="train", objective="binary", rows=1000, features=10, cats=0, levels=32,
             zeros=0.0, nans=0.0, max_bin=255, leaves=31, quant=0, iters=1, classes=1,
             fraction=1.0, query=120)
PREDICT = dict(kind="predict", rows=1000, cols=28, cats=0, levels=32, density=1.0, nans=0.1,
               trees=100, leaves=31, classes=1, what="raw", source="host")


def listed():
    return [
        # a small table with the defaults (f32 gradients, 255 bins, 31 leaves): each
        # tree is a chain of short launches
        dict(TRAIN, name="train_small", rows=5003, features=13, iters=20),
        # the everyday training: a million rows, f32 gradients, 255 bins
        dict(TRAIN, name="train_f32", rows=1000000, features=28, leaves=63, iters=20),
        # the headline workload: 10.5M x 28, 63 bins, 4-bin quantized gradients, 255 leaves
        dict(TRAIN, name="train_quantized", rows=10500000, features=28, max_bin=63, leaves=255,
             quant=4, iters=30),
        # many sparse columns, L2, column sampling
        dict(TRAIN, name="train_sparse_wide", objective="regression", rows=1000000,
             features=2000, zeros=0.9, leaves=127, fraction=0.8, iters=10),
        # ranking over query groups, quantized gradients
        dict(TRAIN, name="train_rank", objective="lambdarank", rows=2000000, features=700,
             zeros=0.3, leaves=255, quant=4, iters=10),
        # softmax over ten classes with categorical columns: ten trees an iteration
        dict(TRAIN, name="train_multiclass", objective="multiclass", rows=2000000, features=100,
             cats=20, leaves=127, classes=10, iters=1),
        # ingest and a short training, as a parameter search does for each table
        dict(TRAIN, name="fit_table", kind="fit", objective="regression", rows=1500007,
             features=39, nans=0.05, max_bin=63, leaves=31, quant=4, iters=10),
        # a host boosting loop's tree: custom objective, gradients from the host
        dict(TRAIN, name="seam_tree", kind="seam", rows=1000003, features=28, nans=0.05,
             max_bin=63, leaves=127, quant=4),
        # an online request: a few rows, class probabilities
        dict(PREDICT, name="predict_request", rows=64, trees=100, what="transformed"),
        # batch scoring of device rows with a large model
        dict(PREDICT, name="predict_batch", rows=2000000, trees=100, leaves=255,
             source="device"),
        # batch scoring of a sparse host matrix, softmax model with categorical splits
        dict(PREDICT, name="predict_sparse", rows=200003, cols=500, cats=20, density=0.05,
             nans=0.0, trees=20, leaves=63, classes=10, what="transformed", source="csr"),
        # explanations of a batch
        dict(PREDICT, name="predict_contrib", rows=50000, trees=100, what="contrib"),
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("narrow", "narrow", "wide", "multiclass", "fit", "seam", "dense",
                       "sparse", "contrib"))
    if kind in ("narrow", "fit", "seam"):
        max_bin = rng.choice((15, 63, 63, 255))
        c = dict(TRAIN, rows=_between(rng, 1000, 3000000), max_bin=max_bin,
                 features=_between(rng, 4, 39 if max_bin < 64 else 30),
                 leaves=rng.choice((15, 31, 63, 127, 255)), quant=rng.choice((0, 4)), iters=5,
                 objective=rng.choice(("binary", "regression")))
        if kind != "narrow":
            c.update(kind=kind, nans=rng.choice((0.0, 0.05)))
        if kind == "seam":
            c.update(quant=4, iters=1, objective="binary")
        return c
    if kind == "wide":
        objective = rng.choice(("regression", "binary", "lambdarank"))
        return dict(TRAIN, rows=_between(rng, 20000, 400000), features=_between(rng, 130, 1000),
                    zeros=rng.choice((0.0, 0.3, 0.9)), objective=objective,
                    leaves=rng.choice((31, 63, 127, 255)), quant=rng.choice((0, 4)), iters=3,
                    fraction=rng.choice((0.8, 1.0)))
    if kind == "multiclass":
        features = rng.randint(20, 100)
        return dict(TRAIN, objective="multiclass", rows=_between(rng, 5000, 500000),
                    features=features, cats=rng.randint(0, features // 4),
                    leaves=rng.choice((31, 63, 127)), classes=rng.randint(3, 10),
                    max_bin=rng.choice((63, 255)), iters=1)
    if kind == "dense":
        source = rng.choice(("host", "device"))
        return dict(PREDICT, source=source, rows=_between(rng, 1, 1000000),
                    cols=rng.randint(5, 120), trees=_between(rng, 10, 100),
                    leaves=rng.choice((15, 31, 127, 255)),
                    what=rng.choice(("raw", "transformed", "leaf")))
    if kind == "sparse":
        classes = rng.choice((1, 3, 10))
        return dict(PREDICT, source="csr", rows=_between(rng, 10, 100000),
                    cols=_between(rng, 60, 1000), cats=rng.randint(0, 20), nans=0.0,
                    density=rng.choice((0.02, 0.1)), trees=_between(rng, 5, 100 // classes),
                    leaves=rng.choice((15, 31, 63)), classes=classes,
                    what=rng.choice(("raw", "transformed", "leaf")))
    return dict(PREDICT, rows=_between(rng, 10, 20000), cols=rng.randint(5, 60),
                trees=_between(rng, 5, 100), leaves=rng.choice((7, 15, 31, 63)), what="contrib")


# ---- inputs ---------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _table(case, seed):
    """The raw table on the device, float32 [features, rows]."""
    gen = _generator(seed)
    n, F, cats = case["rows"], case["features"], case["cats"]
    X = torch.empty((F, n), device=DEVICE, dtype=torch.float32)
    for f0 in range(0, F - cats, 64):
        b = X[f0:min(f0 + 64, F - cats)]
        b.normal_(generator=gen)
        if case["zeros"] > 0:
            u = torch.rand(b.shape, generator=gen, device=DEVICE)
            if case["zeros"] > 0.5:
                b.exp_()
            b[u < case["zeros"]] = 0.0
        if case["nans"] > 0:
            u = torch.rand(b.shape, generator=gen, device=DEVICE)
            b[(u < case["nans"]) & (torch.arange(f0, f0 + len(b), device=DEVICE) % 4 == 1)[:, None]] = math.nan
    if cats:
        X[F - cats:] = torch.randint(0, case["levels"], (cats, n), generator=gen, device=DEVICE).float()
    return X


def _target(case, X, seed):
    """Labels for the table as host float32, and the query boundaries of a ranking."""
    gen = _generator(seed + 1000003)
    n, F, cats, K = case["rows"], case["features"], case["cats"], case["classes"]
    use = min(F - cats, 50)

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=DEVICE)

    Z = torch.nan_to_num(X[:use])
    if case["objective"] == "multiclass":
        s = normal(K, use) @ Z / math.sqrt(use)
        for j in range(F - cats, F):
            s += 0.5 * normal(K, case["levels"])[:, X[j].long()]
        u = torch.rand((K, n), generator=gen, device=DEVICE).clamp_(1e-12, 1 - 1e-7)
        return (s - torch.log(-torch.log(u))).argmax(0).float().cpu().numpy(), None
    s = normal(use) @ Z + 0.5 * Z[0] * Z[1]
    if case["objective"] == "regression":
        return (s + 0.5 * normal(n)).cpu().numpy(), None
    if case["objective"] == "binary":
        u = torch.rand(n, generator=gen, device=DEVICE)
        return (u < torch.sigmoid(s + 0.1 * normal(n))).float().cpu().numpy(), None
    s += 0.5 * s.std() * normal(n)
    edges = torch.sort(s[:200000]).values
    edges = edges[(torch.tensor([0.2, 0.4, 0.6, 0.8]) * (len(edges) - 1)).long().to(DEVICE)]
    y = torch.bucketize(s, edges).float().cpu().numpy()
    sizes = np.random.default_rng(seed).poisson(case["query"], 2 * n // case["query"] + 64)
    ends = np.cumsum(np.clip(sizes, 1, None))
    return y, np.concatenate([[0], ends[ends < n], [n]]).astype(np.int32)


def _mappers(case, X):
    """One BinMapper per numerical feature, from a sample of the rows."""
    n = case["rows"]
    idx = torch.from_numpy(sample_indices(n, BIN_SAMPLE, 1).astype(np.int64)).to(DEVICE)
    S = X[:, idx].cpu().numpy().astype(np.float64)
    return [BinMapper.from_sampled_column(col, n, max_bin=case["max_bin"],
                                          min_data_in_leaf=MIN_DATA,
                                          bin_construct_sample_cnt=BIN_SAMPLE) for col in S]


def _plain(case):
    """A training that `exact` can follow: numerical columns, f32 gradients, one score."""
    return (case["kind"] == "train" and case["quant"] == 0 and case["classes"] == 1
            and case["fraction"] == 1.0 and case["cats"] == 0
            and case["objective"] != "lambdarank")


def _binned(case, X):
    """A table without missing values as a program that bins for itself hands it over:
    uint8 bins [features, rows] on the device, and per feature its descriptor and bin
    values.  Numerical columns get equal-frequency bins of their nonzero values and a bin
    of zeros, categorical ones a bin per level after the one kept for unknown levels."""
    F, cats = case["features"], case["cats"]
    out = torch.empty(X.shape, dtype=torch.uint8, device=DEVICE)
    meta, values = [], []
    zero = torch.tensor([-1e-35, 1e-35], device=DEVICE)
    for f in range(F):
        if f >= F - cats:
            out[f] = X[f] + 1
            meta.append(feature_meta(case["levels"] + 1, 1, 0, 1, f, bin_type=1))
            values.append(torch.arange(-1, case["levels"], dtype=torch.float64, device=DEVICE))
            continue
        s = X[f, :BIN_SAMPLE]
        s = torch.sort(s[s != 0]).values
        k = case["max_bin"] - 2
        edges = s[torch.arange(1, k, device=DEVICE) * len(s) // k]
        edges = torch.unique(torch.cat([edges, zero if edges[0] < 0 else zero[1:]]))
        out[f] = torch.bucketize(X[f], edges)
        at = int(torch.searchsorted(edges, zero[1]))
        meta.append(feature_meta(len(edges) + 1, at, 0, at, f))
        values.append(torch.cat([edges.double(), torch.full((1,), math.inf, device=DEVICE)]))
    return out, meta, torch.cat(values).cpu().numpy()


def _config():
    return GainConfig.make(min_data_in_leaf=MIN_DATA, min_sum_hessian_in_leaf=MIN_HESSIAN)


def _forest(case, seed):
    """Random trees grown like a leaf-wise learner grows them: the heavier of two random
    leaves is split on a feature (low positions more often) at a random quantile of the
    range it has left there.  Each tree is a dict of the arrays a model is made from, with
    `sets`, the levels that go left at its categorical nodes."""
    rng = np.random.default_rng(seed)
    cols, cats, nl = case["cols"], case["cats"], case["leaves"]
    num = cols - cats
    sparse = case["source"] == "csr"
    trees = []
    for _ in range(case["trees"] * case["classes"]):
        u = rng.random((nl, 6))
        sets = rng.random((nl, case["levels"])) < 0.5
        sets[:, 0], sets[:, 1] = True, False
        mass, box, at = [1.0], [{}], [None]
        feat, quant, left, right, dt = [], [], [], [], []
        for node in range(nl - 1):
            a, b = int(u[node, 0] * len(mass)), int(u[node, 1] * len(mass))
            leaf = a if mass[a] >= mass[b] else b
            f = int(u[node, 2] ** 2 * num)
            is_cat = cats > 0 and u[node, 3] < 0.15
            if is_cat:
                f, p, q = num + f % cats, 0.5, 0.5
            else:
                lo, hi = box[leaf].get(f, (0.0, 1.0))
                p = 0.2 + 0.6 * u[node, 4]
                q = lo + p * (hi - lo)
            if at[leaf] is not None:
                side, parent = at[leaf]
                side[parent] = node
            feat.append(f)
            quant.append(q)
            # decision type: categorical; else the missing type (zero for a sparse
            # matrix, NaN where the column has any) and a default direction
            dt.append(1 if is_cat else ((1 if sparse else 2) << 2) + (2 if u[node, 5] < 0.5 else 0))
            left.append(~leaf)
            right.append(~len(mass))
            at.append((right, node))
            at[leaf] = (left, node)
            mass.append(mass[leaf] * (1 - p))
            mass[leaf] *= p
            old = box[leaf]
            box.append(old if is_cat else {**old, f: (q, hi)})
            box[leaf] = old if is_cat else {**old, f: (lo, q)}
        q = torch.tensor(quant, dtype=torch.float64).clamp_(1e-6, 1 - 1e-6)
        thr = torch.special.ndtri(q).numpy()
        dt = np.array(dt, np.int8)
        is_cat = (dt & 1) > 0
        thr[is_cat] = np.arange(int(is_cat.sum()))
        weight = np.maximum(1, np.round(np.array(mass) * 1e6)).astype(np.int32)
        cover = np.zeros(nl - 1, np.int32)
        for node in range(nl - 2, -1, -1):  # children have higher numbers
            cover[node] = sum(cover[k] if k >= 0 else weight[~k] for k in (left[node], right[node]))
        trees.append(dict(
            num_leaves=nl, split_feature=np.array(feat, np.int32), threshold=thr,
            decision_type=dt, left_child=np.array(left, np.int32),
            right_child=np.array(right, np.int32),
            internal_count=cover, leaf_value=rng.normal(0.0, 0.1, nl), leaf_count=weight, num_cat=int(is_cat.sum()),
            sets=sets[:nl - 1][is_cat]))
    return trees


def _objective(case):
    return "multiclass num_class:%d" % case["classes"] if case["classes"] > 1 else "binary sigmoid:1"


def _model(case, forest):
    """The forest as the model text that a program loads."""
    words = -(-case["levels"] // 32)

    def line(key, values):
        return "%s=%s" % (key, " ".join(map(repr, np.asarray(values).tolist())))

    text = ["tree", "version=v4", "num_class=%d" % case["classes"],
            "num_tree_per_iteration=%d" % case["classes"], "label_index=0",
            "max_feature_idx=%d" % (case["cols"] - 1), "objective=" + _objective(case),
            "feature_names=" + " ".join("Column_%d" % f for f in range(case["cols"])),
            "feature_infos=" + " ".join(["none"] * case["cols"]), ""]
    for i, t in enumerate(forest):
        text += ["Tree=%d" % i, "num_leaves=%d" % t["num_leaves"], "num_cat=%d" % t["num_cat"]]
        text += [line(k, v) for k, v in t.items() if k not in ("num_leaves", "num_cat", "sets")]
        if t["num_cat"]:
            bits = np.zeros((t["num_cat"], 32 * words), np.uint64)
            bits[:, :case["levels"]] = t["sets"]
            packed = (bits.reshape(-1, words, 32) << np.arange(32, dtype=np.uint64)).sum(2)
            text += [line("cat_boundaries", np.arange(t["num_cat"] + 1) * words),
                     line("cat_threshold", packed.ravel())]
        text += ["is_linear=0", "shrinkage=1", "", ""]
    return Model("\n".join(text + ["end of trees", ""]))


def _rows(case, seed):
    """Rows to predict, float32 [rows, cols] on the device."""
    gen = _generator(seed + 7)
    n, cols, cats = case["rows"], case["cols"], case["cats"]
    X = torch.randn((n, cols), generator=gen, device=DEVICE)
    if cats:
        X[:, cols - cats:] = torch.randint(0, case["levels"], (n, cats), generator=gen, device=DEVICE).float()
    if case["density"] < 1:
        X[torch.rand((n, cols), generator=gen, device=DEVICE) >= case["density"]] = 0.0
    if case["nans"] > 0:
        X[torch.rand((n, cols), generator=gen, device=DEVICE) < case["nans"]] = math.nan
    return X


# ---- a program's state ----------------------------------------------------------------

def prepare(case, seed):
    state = {"case": case, "be": HipBackend(0)}
    if case["kind"] == "predict":
        X = _rows(case, seed)
        state["model"] = _model(case, _forest(case, seed))
        if case["source"] == "device":
            state["x"] = X
            leaf = case["what"] == "leaf"
            state["out"] = torch.empty((case["rows"], case["classes"] * (case["trees"] if leaf else 1)),
                                       device=DEVICE, dtype=torch.int32 if leaf else torch.float64)
        elif case["source"] == "csr":
            row, col = torch.nonzero(X, as_tuple=True)
            ends = torch.cumsum(torch.bincount(row, minlength=case["rows"]), 0).cpu().numpy()
            state["csr"] = (np.concatenate([[0], ends]).astype(np.int64),
                            col.int().cpu().numpy(), X[row, col].cpu().numpy())
        else:
            state["x"] = X.cpu().numpy()
        torch.cuda.synchronize()
        return state
    X = _table(case, seed)
    y, queries = _target(case, X, seed)
    state.update(labels=y, queries=queries, config=_config())
    be, n = state["be"], case["rows"]
    torch.cuda.synchronize()  # the library works on a stream of its own
    if case["kind"] == "fit":
        state.update(x=X.t().contiguous(), mappers=_mappers(case, X))
    elif case["kind"] == "seam":
        be.upload_raw_device(X.data_ptr(), np.float32, n, case["features"], _mappers(case, X),
                             col_major=True)
    else:
        bins, meta, values = _binned(case, X)
        be.upload_resident_bins(bins.cpu().numpy(), meta, values)
    if case["kind"] == "seam":
        p = 1.0 / (1.0 + np.exp(-0.5 * np.random.default_rng(seed).standard_normal(n)))
        state.update(grad=(p - y).astype(np.float32), hess=(p * (1 - p)).astype(np.float32))
    else:
        be.set_lookahead(case["classes"] == 1)
    if case["classes"] > 1:
        prior = np.bincount(y.astype(np.int64), minlength=case["classes"]) / n
        state["init"] = np.log(np.maximum(prior, EPS))
    elif case["kind"] != "seam":
        init = boost_from_score(case["objective"], y)
        state["init"] = init if abs(init) > EPS else 0.0
    torch.cuda.synchronize()
    return state


def _joined(trees, leaves):
    """The trees' arrays, one after another and zeros up to what full trees hold (a level
    set fits a word), and their leaf counts."""
    out = {"num_leaves": np.array([t["num_leaves"] for t in trees])}
    for k in TREE_FIELDS:
        a = np.concatenate([t[k] for t in trees])
        a.resize(len(trees) * leaves)
        out[k] = a
    return out


def _train(state):
    case, be = state["case"], state["be"]
    cfg, leaves, quant = state["config"], case["leaves"], case["quant"]
    trees = []
    if case["classes"] > 1:
        be.set_labels_multiclass(state["labels"], case["classes"], state["init"])
        for i in range(case["iters"]):
            trees += be.train_iter_multiclass(i, cfg, leaves, -1, LEARNING_RATE, quant)
    else:
        be.set_labels(state["labels"], state["init"])
        if case["objective"] == "lambdarank":
            be.set_lambdarank(state["queries"])
        else:
            be.set_objective(case["objective"])
        if case["fraction"] < 1:
            be.set_col_sampler(case["fraction"], 1.0, COL_SEED)
        for i in range(case["iters"]):
            trees.append(be.train_iter(i, cfg, leaves, -1, LEARNING_RATE, quant))
    return {"trees": _joined(trees, leaves), "scores": be.scores()}


def run(state):
    case, be = state["case"], state["be"]
    if case["kind"] == "train":
        return _train(state)
    if case["kind"] == "fit":
        x = state["x"]
        be.upload_raw_device(x.data_ptr(), np.float32, x.shape[0], x.shape[1], state["mappers"])
        return _train(state)
    if case["kind"] == "seam":
        be.upload_resident_grad_hess(state["grad"], state["hess"])
        scales, _, _ = be.discretize_dequantize_in_place(case["quant"], True, 1)
        tree, layout = be.grow_tree_on_device_with_cfg(state["config"], case["leaves"])
        return {"scales": scales, "trees": _joined([tree], case["leaves"]),
                "layout": layout}
    m = state["model"]
    if case["source"] == "device":
        be.predict_device(m, state["x"].data_ptr(), case["rows"], case["cols"],
                          state["out"].data_ptr(), case["what"])
        return state["out"]
    if case["source"] == "csr":
        return be.predict_csr(m, *state["csr"], case["cols"], case["what"])
    return be.predict(m, state["x"], case["what"])


# ---- the same in 64 bits ----------------------------------------------------------------

def _walk64(case, forest, X):
    """Leaf of every row in every tree, [trees, rows]."""
    out = []
    rows = torch.arange(len(X), device=DEVICE)
    for t in forest:
        feat, left, right, thr, dt = (torch.from_numpy(t[k]).to(DEVICE) for k in (
            "split_feature", "left_child", "right_child", "threshold", "decision_type"))
        sets = torch.from_numpy(t["sets"]).to(DEVICE) if t["num_cat"] else torch.ones(
            (1, case["levels"]), dtype=torch.bool, device=DEVICE)
        node = torch.zeros(len(X), dtype=torch.int64, device=DEVICE)
        while bool((node >= 0).any()):
            i = node.clamp_min(0)
            v, d = X[rows, feat[i].long()].double(), dt[i]
            cat, missing = (d & 1) > 0, d >> 2
            nan = v.isnan()
            v = torch.where(nan & (missing != 2), 0.0, v)
            by_default = ((missing == 1) & (v.abs() <= 1e-35)) | ((missing == 2) & nan)
            go = torch.where(by_default, (d & 2) > 0, v <= thr[i])
            k = torch.where(cat, thr[i], 0.0).long()
            level = torch.nan_to_num(v).clamp(0, case["levels"] - 1).long()
            go = torch.where(cat, sets[k, level], go)
            node = torch.where(node < 0, node, torch.where(go, left[i], right[i]).long())
        out.append(~node)
    return torch.stack(out)


def _contrib64(case, forest, X):
    """TreeSHAP (path-dependent) from its definition: a leaf on a path of m distinct
    features, z_j the cover share it keeps when feature j is not known and o_j whether the
    row satisfies the path's conditions on j, gives feature i its value times (o_i - z_i)
    times sum over k of k! (m - k - 1)! / m! times the coefficient of x^k in
    prod_{j != i} (z_j + o_j x)."""
    phi = torch.zeros((len(X), case["cols"] + 1), dtype=torch.float64, device=DEVICE)
    for t in forest:
        cover, count = t["internal_count"].astype(float), t["leaf_count"].astype(float)
        thr, dt = t["threshold"], t["decision_type"]
        phi[:, -1] += float((t["leaf_value"] * count).sum() / count.sum())
        stack = [(0, {})]
        while stack:
            node, path = stack.pop()
            if node >= 0:
                f = int(t["split_feature"][node])
                v = X[:, f].double()
                go = torch.where(v.isnan(), bool(dt[node] & 2), v <= thr[node])
                for child, ok in ((int(t["left_child"][node]), go), (int(t["right_child"][node]), ~go)):
                    share = (cover[child] if child >= 0 else count[~child]) / cover[node]
                    z, o = path.get(f, (1.0, None))
                    stack.append((child, {**path, f: (z * share, ok if o is None else o & ok)}))
                continue
            m, names = len(path), list(path)
            zs = torch.tensor([path[f][0] for f in names], dtype=torch.float64, device=DEVICE)
            os_ = torch.stack([path[f][1] for f in names]).double()
            poly = torch.zeros((m, m, len(X)), dtype=torch.float64, device=DEVICE)  # [i, k, row]
            poly[:, 0] = 1.0
            for j in range(m):
                keep = poly[j].clone()
                up = torch.cat([torch.zeros_like(poly[:, :1]), poly[:, :-1]], 1)
                poly = poly * zs[j] + up * os_[j]
                poly[j] = keep
            w = torch.tensor([math.factorial(k) * math.factorial(m - k - 1) / math.factorial(m)
                              for k in range(m)], dtype=torch.float64, device=DEVICE)
            total = (poly * w[None, :, None]).sum(1)
            phi[:, torch.tensor(names, device=DEVICE)] += (
                total * (os_ - zs[:, None]) * float(t["leaf_value"][~node])).t()
    return phi


def _predict64(case, seed):
    forest, X = _forest(case, seed), _rows(case, seed)
    if case["what"] == "leaf":
        return None
    if case["what"] == "contrib":
        return _contrib64(case, forest, X)
    leaf = _walk64(case, forest, X)
    K = case["classes"]
    score = torch.zeros((case["rows"], K), dtype=torch.float64, device=DEVICE)
    for i, t in enumerate(forest):
        score[:, i % K] += torch.from_numpy(t["leaf_value"]).to(DEVICE)[leaf[i]]
    if case["what"] == "raw":
        return score
    return torch.softmax(score, 1) if K > 1 else torch.sigmoid(score)


class _Leaf:
    """A leaf of the 64-bit learner: its rows, histogram [2, features, bins], sums, the
    features it may still split on, and its best split."""

    def __init__(self, rows, hist, g, h, can):
        self.rows, self.hist, self.g, self.h, self.can = rows, hist, g, h, can
        self.gain, self.split = -math.inf, None

    def scan(self, counts):
        """Best threshold of every feature, high thresholds first, as a numerical scan
        without missing values finds it."""
        n, h = len(self.rows), self.h + 2 * EPS
        G, H = self.hist
        C = torch.floor(H * (n / h) + 0.5)
        g_r, h_r, n_r = (v.flip(1).cumsum(1)[:, :-1] for v in (G, H, C))
        h_r = h_r + EPS
        g_l, h_l, n_l = self.g - g_r, h - h_r, n - n_r
        gain = g_l * g_l / h_l + g_r * g_r / h_r
        B = G.shape[1]
        t = torch.arange(B - 2, -1, -1, device=DEVICE)[None, :]  # bins <= t go left
        ok = ((t < counts[:, None] - 1) & (n_r >= MIN_DATA) & (n_l >= MIN_DATA)
              & (h_r >= MIN_HESSIAN) & (h_l >= MIN_HESSIAN) & self.can[:, None])
        shift = self.g * self.g / h
        gain = torch.where(ok & (gain > shift), gain, torch.full_like(gain, -math.inf))
        best, pos = gain.max(1)
        first = (gain == best[:, None]).int().argmax(1)
        self.can = best > -math.inf
        best, f = (best - shift).max(0)
        f = int((best == torch.where(self.can, gain.max(1).values - shift, -math.inf)).int().argmax())
        if not bool(self.can[f]):
            return
        at = int(first[f])
        self.gain = float(best)
        self.split = (f, B - 2 - at, float(g_l[f, at]), float(h_l[f, at]) - EPS,
                      float(g_r[f, at]), float(h_r[f, at]) - EPS)


def _grow64(bins, counts, g, h, leaves):
    """One leaf-wise tree over u8 bins [features, rows] in 64 bits: the leaves in the
    learner's order (a split's left child keeps its number, the right child is the next)."""
    F, B = len(bins), int(counts.max())
    base = torch.arange(F, device=DEVICE)[:, None] * B

    def histogram(rows):
        at = (bins[:, rows].long() + base).reshape(-1)
        return torch.stack([torch.bincount(at, v[rows].repeat(F), F * B).view(F, B) for v in (g, h)])

    rows = torch.arange(bins.shape[1], device=DEVICE)
    can = torch.ones(F, dtype=torch.bool, device=DEVICE)
    tree = [_Leaf(rows, histogram(rows), float(g.sum()), float(h.sum()), can)]
    if len(rows) >= 2 * MIN_DATA:
        tree[0].scan(counts)
    while len(tree) < leaves:
        i = max(range(len(tree)), key=lambda k: (tree[k].gain, -k))
        p = tree[i]
        if not p.gain > 0:
            break
        f, t, gl, hl, gr, hr = p.split
        left = bins[f, p.rows] <= t
        rl, rr = p.rows[left], p.rows[~left]
        small = histogram(rl if len(rl) < len(rr) else rr)
        other = p.hist - small
        hists = (small, other) if len(rl) < len(rr) else (other, small)
        tree[i] = _Leaf(rl, hists[0], gl, hl, p.can)
        tree.append(_Leaf(rr, hists[1], gr, hr, p.can))
        if max(len(rl), len(rr)) >= 2 * MIN_DATA:
            tree[i].scan(counts)
            tree[-1].scan(counts)
    return tree


def _train64(case, seed):
    X = _table(case, seed)
    y, _ = _target(case, X, seed)
    bins, meta, _ = _binned(case, X)
    counts = torch.tensor([m.num_bin for m in meta], device=DEVICE)
    y = torch.from_numpy(y).to(DEVICE).double()
    mean = float(y.mean())
    binary = case["objective"] == "binary"
    score = torch.full_like(y, math.log(mean / (1 - mean)) if binary else mean)
    values = []
    for _ in range(case["iters"]):
        if binary:
            sign = torch.where(y > 0, 1.0, -1.0)
            r = -sign / (1 + torch.exp(sign * score))
            g, h = r.float().double(), (r.abs() * (1 - r.abs())).float().double()
        else:
            g, h = (score - y).float().double(), torch.ones_like(y)
        for leaf in (tree := _grow64(bins, counts, g, h, case["leaves"])):
            out = -leaf.g / (leaf.h + 2 * EPS) * LEARNING_RATE
            values.append(out)
            if len(tree) > 1:
                score[leaf.rows] += out
    values = np.array(values)
    values.resize(case["iters"] * case["leaves"])
    return {"trees": dict(dict.fromkeys(TREE_FIELDS + ("num_leaves",)), leaf_value=values),
            "scores": score}


def exact(case, seed):
    """The outputs in 64 bits.  Quantized trainings have none of their own: their trees and
    scores follow from whole numbers and are compared bit for bit.  The wide, multiclass
    and lambdarank trainings would take minutes."""
    if case["kind"] == "predict":
        return _predict64(case, seed)
    if _plain(case) and case["rows"] * case["features"] * case["iters"] <= 600_000_000:
        return _train64(case, seed)
    return None


# ---- what a pass cannot do without ------------------------------------------------------

def work(case):
    n = case["rows"]
    if case["kind"] == "predict":
        K, walks = case["classes"], n * case["trees"] * case["classes"]
        depth = max(1.0, math.log2(case["leaves"]))
        width = {"leaf": 4 * case["trees"] * K, "contrib": 8 * (case["cols"] + 1) * K}.get(case["what"], 8 * K)
        cell = 4 if case["source"] != "csr" else 8 * case["density"]
        forest = case["trees"] * K * case["leaves"] * 32
        # a comparison a level; contributions: every leaf's path, quadratic in its length
        ops = walks * (depth if case["what"] != "contrib" else 6 * case["leaves"] * depth ** 2)
        return {"bytes": n * (case["cols"] * cell + width) + forest, "flops": ops}
    # each tree reads every row's bins and gradients once and updates its score; a level of
    # the tree adds half the rows' bins to the smaller children's histograms
    F, trees = case["features"], case["iters"] * case["classes"]
    row = F + (2 if case["quant"] else 8)
    per_tree = n * (row + 4 + 16)
    adds = 2 * n * F * (1 + 0.5 * math.log2(case["leaves"]))
    if case["kind"] == "fit":
        return {"bytes": trees * per_tree + n * F * 5, "flops": trees * adds}
    if case["kind"] == "seam":
        return {"bytes": n * (row + 8 + 4), "flops": adds}
    return {"bytes": trees * per_tree + n * 8 * case["classes"], "flops": trees * adds}


def tolerance(case):
    if case["kind"] == "predict":
        # f64 sums of the same leaf values: 1e-16 apart in another order; exp and the
        # path products of the contributions a few ulps more
        return "exact" if case["what"] == "leaf" else {"rel": 1e-14, "max": 1e-12}
    if case["quant"] == 4:
        return "exact"  # whole-number histograms: every later value follows from them
    # f32 gradients summed in f64 or 64-bit fixed point: the same splits, leaf values and
    # gains within the rounding of the sums and of their cancellation in small leaves
    return {"rel": 1e-9, "max": 1e-7}
