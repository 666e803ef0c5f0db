"""The packed trees of k_predict_lds (model_pack_trees), without a GPU: which models get
them, and that a model for which memory is short goes without instead of failing.  The
entries are walked here as the kernel walks them and compared with the nodes."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "lightgbm_rs_amd", "csrc")
SRC = r"""
#include <sys/resource.h>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <sstream>
#include "model.h"

// Leaf by the packed entries, as pred_walk goes; a set of several words by its index.
static int walk(const PredEntry* w, const float* x, const lgbm_hip_model& m) {
  for (uint32_t e = 0;;) {
    const PredEntry n = w[e];
    if ((n.word & 0xffffu) == 0u) { int l; std::memcpy(&l, &n.threshold, 4); return l; }
    float v = x[(n.word >> 16) & 0xfffu];
    uint32_t bits; std::memcpy(&bits, &n.threshold, 4);
    bool second;
    if (n.word & PRED_CATEGORICAL) {
      const bool some = v > -1.0f && v < 2147483648.0f;
      const int32_t c = some ? (int32_t)v : 0;
      if (n.word & PRED_SET) {
        const int32_t lo = m.cat_bounds[bits], words = m.cat_bounds[bits + 1] - lo;
        second = !(some && c / 32 < words && ((m.cat_words[lo + c / 32] >> (c % 32)) & 1u));
      } else {
        second = !(some && c < 32 && ((bits >> c) & 1u));
      }
    } else {
      if ((n.word & PRED_ZERO_MISSING) && std::fabs((double)v) <= 1e-35) v = NAN;
      second = ((n.word & PRED_FLIP) ? -v : v) > n.threshold;
    }
    e = (n.word & 0xffffu) + (second ? 1u : 0u);
  }
}

int main(int argc, char** argv) {
  std::ifstream f(argv[1]);
  std::stringstream ss;
  ss << f.rdbuf();
  std::string text = ss.str(), err;
  lgbm_hip_model m;
  if (!parse_model_text(text.data(), text.size(), &m, &err)) { std::puts(err.c_str()); return 1; }
  if (argc > 2 && !std::strcmp(argv[2], "short")) {
    rlimit r{1 << 20, 1 << 20};  // no more address space than there is
    setrlimit(RLIMIT_AS, &r);
  }
  PredPacked p;
  const bool ok = model_pack_trees(m, &p);
  std::printf("%d %zu %d %d\n", ok ? 1 : 0, p.words.size(), p.stride, p.values);
  if (ok && argc > 3) {
    std::ifstream rows(argv[3], std::ios::binary);
    std::vector<float> x((size_t)m.max_feature_idx + 1);
    while (rows.read((char*)x.data(), x.size() * 4)) {
      for (size_t t = 0; t < m.tree_index.size(); ++t) {
        const PredEntry* w = p.words.data() + t * p.stride;
        const int l = walk(w, x.data(), m);
        double v; std::memcpy((void*)&v, (const void*)(w + p.values + l), 8);
        std::printf("%d %a\n", l, v);
      }
    }
  }
}
"""


@pytest.fixture(scope="module")
def pack(tmp_path_factory):
    d = tmp_path_factory.mktemp("pack_trees")
    (d / "t.cpp").write_text(SRC)
    exe = str(d / "t")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "t.cpp"),
                    os.path.join(CSRC, "model.cpp"), "-o", exe], check=True)

    def run(text, *args, rows=None):
        (d / "m.txt").write_text(text)
        cmd = [exe, str(d / "m.txt"), *args]
        if rows is not None:
            rows.astype(np.float32).tofile(d / "x.bin")
            cmd += ["-", str(d / "x.bin")]
        out = subprocess.run(cmd, capture_output=True, text=True)
        assert out.returncode == 0, out.stdout + out.stderr
        lines = out.stdout.splitlines()
        return tuple(map(int, lines[0].split())), lines[1:]

    return run


def _stump(i):
    return (f"Tree={i}\nnum_leaves=2\nnum_cat=0\nsplit_feature=0\nthreshold=0.5\ndecision_type=2\n"
            "left_child=-1\nright_child=-2\nleaf_value=1 2\nis_linear=0\nshrinkage=1\n\n\n")


def _chain(i, leaves):
    n = leaves - 1
    return (f"Tree={i}\nnum_leaves={leaves}\nnum_cat=0\nsplit_feature={' '.join(['0'] * n)}\n"
            f"threshold={' '.join(str(k / n) for k in range(n))}\ndecision_type={' '.join(['2'] * n)}\n"
            f"left_child={' '.join(str(~k) for k in range(n))}\n"
            f"right_child={' '.join(str(k + 1) if k + 1 < n else str(~n) for k in range(n))}\n"
            f"leaf_value={' '.join(str(k) for k in range(leaves))}\nis_linear=0\nshrinkage=1\n\n\n")


def _model(trees, features=1):
    return ("tree\nversion=v4\nnum_class=1\nnum_tree_per_iteration=1\nlabel_index=0\n"
            f"max_feature_idx={features - 1}\nobjective=regression\n"
            f"feature_names={' '.join(f'c{i}' for i in range(features))}\n"
            f"feature_infos={' '.join(['none'] * features)}\n\n" + "".join(trees) + "end of trees\n")


# (stumps beside one tree of `leaves`, whether the model is packed): every tree takes the
# largest one's 3 * leaves - 1 words, up to 2^23 words whatever the padding
@pytest.mark.parametrize("stumps,leaves,packed", [
    (0, 2, True), (3, 1365, True), (3, 1366, False), (2040, 1365, True), (2060, 1365, False),
    (16000, 1365, False), (16000, 13, True)])
def test_padding_is_bounded(pack, stumps, leaves, packed):
    (ok, words, stride, values), _ = pack(_model([_chain(0, leaves)] + [_stump(i + 1) for i in range(stumps)]))
    assert ok == int(packed)
    if packed:
        assert (words, stride, values) == ((stumps + 1) * (3 * leaves - 1), 3 * leaves - 1, 2 * leaves - 1)
    else:
        assert words == 0


def test_short_memory_leaves_the_model_unpacked(pack):
    text = _model([_chain(0, 1000)] + [_stump(i + 1) for i in range(1500)])  # 36 MB packed
    assert pack(text)[0][0] == 1
    assert pack(text, "short")[0] == (0, 0, 0, 0)


@pytest.mark.parametrize("leaves,cat", [(2, False), (31, False), (31, True), (255, True)])
def test_entries_walk_like_the_nodes(pack, leaves, cat):
    from oracle import predict as P
    from tests.test_gpu_predict_lds import _rows, _text
    rng = np.random.default_rng(leaves)
    text = _text(rng, leaves, 7, 1, 4, cat)
    X = _rows(rng, 300, 7)
    (ok, *_), lines = pack(text, rows=X)
    assert ok == 1
    pm = P.parse_model(text)
    ref = np.asarray(P.predict(pm, X, kind="leaf")).reshape(300, -1)
    got = np.array([int(v.split()[0]) for v in lines]).reshape(300, -1)
    assert np.array_equal(got, ref)
    value = [float.fromhex(v.split()[1]) for v in lines]
    leaf_value = [np.atleast_1d(t["leaf_value"]) for t in pm["trees"]]
    assert value == [leaf_value[k % len(leaf_value)][v] for k, v in enumerate(ref.ravel())]
