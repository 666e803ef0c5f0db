"""The leaf paths behind feature contributions (model_shap_paths), without a GPU: those of a
range of trees are the ones that the whole model has, and nothing beyond the range is made."""
import os
import subprocess

import numpy as np
import pytest

from lightgbm_rs_amd import Model
from tests.test_gpu_contrib_paths import _tree

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "lightgbm_rs_amd", "csrc")
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <sstream>
#include "model.h"
int main(int, char** argv) {
  std::ifstream f(argv[1]);
  std::stringstream ss;
  ss << f.rdbuf();
  std::string text = ss.str(), err;
  lgbm_hip_model m;
  if (!parse_model_text(text.data(), text.size(), &m, &err)) return 1;
  ShapPaths p;
  model_shap_paths(m, std::atoi(argv[2]), std::atoi(argv[3]), &p);
  std::printf("%zu %zu %zu\n", p.leaves.size(), p.steps.size(), p.feats.size());
  for (const ShapLeaf& l : p.leaves) {
    std::printf("%d %d", l.tree, l.dm);
    for (int j = 0; j < (l.dm & 0xffff); ++j)
      std::printf(" %d:%d", p.steps[l.path0 + j].node, p.steps[l.path0 + j].other);
    for (int j = 0; j < l.dm >> 16; ++j) std::printf(" %d", p.feats[l.feat0 + j]);
    std::printf("\n");
  }
}
"""


@pytest.fixture(scope="module")
def paths(tmp_path_factory):
    d = tmp_path_factory.mktemp("shap_paths")
    (d / "t.cpp").write_text(SRC)
    exe = str(d / "t")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "t.cpp"),
                    os.path.join(CSRC, "model.cpp"), "-o", exe], check=True)
    rng = np.random.default_rng(4)
    leaves = [5, 1, 30, 2, 32, 9]
    m = Model.create(num_class=1, max_feature_idx=6)
    for i, n in enumerate(leaves):
        m.add_tree(_tree(rng, n, 7, i == 4))
    (d / "m.txt").write_text(m.to_text())

    def run(t0, t1):
        out = subprocess.run([exe, str(d / "m.txt"), str(t0), str(t1)], capture_output=True,
                             text=True, check=True).stdout.splitlines()
        return tuple(map(int, out[0].split())), out[1:]

    return leaves, run


@pytest.mark.parametrize("t0,t1", [(0, 1), (1, 2), (2, 3), (1, 5), (5, 6), (0, 6)])
def test_a_range_of_the_whole(paths, t0, t1):
    leaves, run = paths
    _, whole = run(0, len(leaves))
    (n_leaves, n_steps, n_feats), got = run(t0, t1)
    assert got == whole[sum(leaves[:t0]):sum(leaves[:t1])] and n_leaves == sum(leaves[t0:t1])
    assert n_steps == sum(":" in v for line in got for v in line.split())
    assert n_feats == sum(":" not in v for line in got for v in line.split()[2:])
