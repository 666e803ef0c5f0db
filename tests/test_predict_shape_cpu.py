"""The choice between k_predict_lds and k_predict (predict_shape.h), without a GPU: blocks
that fit what the kernel assumes over the whole range of calls, and calls of which one
kernel was measured clearly faster going to that one."""
import itertools
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "lightgbm_rs_amd", "csrc")
SRC = r"""
#include <cstdio>
#include "predict_shape.h"
int main() {
  long long rows; int width, words, trees, form, transformed; double leaves, entries;
  while (std::scanf("%lld %d %d %d %lf %d %lf %d", &rows, &width, &words, &trees, &leaves, &form, &entries, &transformed) == 8) {
    const lgbm::PredShape s = lgbm::predict_lds_shape({rows, width, words, trees, leaves, (lgbm::PredForm)form, entries, transformed});
    std::printf("%d %d %zu\n", s.rb, s.nb, s.lds);
  }
}
"""


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    d = tmp_path_factory.mktemp("predict_shape")
    (d / "t.cpp").write_text(SRC)
    exe = str(d / "t")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "t.cpp"), "-o", exe], check=True)

    def run(calls):
        text = "\n".join(" ".join(map(str, c)) for c in calls)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


def _call(rows, cols, leaves, trees, form=0, entries=0, transformed=0):
    return (rows, cols, 3 * leaves - 1, trees, leaves, form, entries, transformed)


def test_blocks_fit_the_kernel(shape):
    calls = [_call(*c) for c in itertools.product(
        (1, 7, 255, 2048, 2049, 65537, 10 ** 6, 10 ** 8, 2 ** 33), (1, 2, 63, 64, 500, 4095),
        (1, 2, 31, 700, 1365, 1366), (0, 1, 3, 100, 20000), (0, 1, 2))]
    taken = 0
    for c, (rb, nb, lds) in zip(calls, shape(calls)):
        rows, width, words, trees, *_ = c
        if rb == 0:
            continue
        taken += 1
        groups = 1024 // rb
        assert 8 <= rb <= 1024 and rb & (rb - 1) == 0 and 1 <= nb <= trees
        assert words <= 4096 and nb * words <= 4096  # a thread stages 4 words of a batch
        assert lds <= 156 * 1024
        assert lds >= rb * (width | 1) * 4 + 16 * nb * words + (16 * nb * rb if groups > 1 else 0)
        assert rb == 8 or rows >= rb * 256  # a block a CU
    assert taken > 300


def test_what_does_not_fit_is_refused(shape):
    assert all(rb == 0 for rb, _, _ in shape([
        _call(100, 28, 1366, 50), _call(100, 28, 31, 0), _call(100, 5000, 31, 50),
        _call(100, 0, 31, 50)]))


# (rows, columns, leaves, trees, CSR, entries a row, outputs transformed): k_predict and k_predict_lds, us
@pytest.mark.parametrize("call,walk,lds", [
    ((200000, 120, 31, 1), 27, 46), ((200000, 500, 31, 1), 31, 134), ((200000, 500, 31, 3), 59, 127),
    ((200000, 1000, 31, 3), 66, 229), ((200000, 1000, 31, 10), 195, 241), ((200000, 3900, 31, 1), 33, 840),
    ((200000, 3900, 31, 30), 613, 1100), ((200000, 1000, 255, 10), 306, 455), ((20000, 3900, 255, 10), 101, 182),
    ((200000, 2000, 255, 100), 3096, 4905), ((200000, 3900, 255, 300), 9850, 30360),
    ((60000, 1400, 900, 200), 2960, 7534), ((1000000, 160, 15, 1), 78, 226),
    ((60000, 3900, 255, 100, 1, 78), 1499, 2980), ((60000, 3900, 255, 20, 1, 78), 618, 823),
    ((64, 28, 31, 100), 270, 14), ((1000, 28, 31, 1), 19, 16), ((1000, 3900, 255, 300), 2277, 324),
    ((200000, 28, 255, 300), 1530, 390), ((200000, 120, 255, 10), 194, 79), ((200000, 200, 31, 10), 142, 83),
    ((200000, 500, 255, 30), 809, 469), ((20000, 1000, 31, 10), 69, 39), ((200000, 1000, 31, 30), 540, 290),
    ((20000, 2000, 255, 30), 276, 192), ((200000, 3900, 31, 300), 5849, 3923),
    ((250000, 500, 31, 1, 1, 10), 179, 149), ((2000, 3900, 31, 1, 1, 78), 98, 14),
    ((250000, 60, 255, 100, 1, 1.2), 665, 294), ((60000, 500, 31, 1, 1, 50), 128, 59), ((600000, 28, 31, 60, 0, 0, 60), 1741, 2078),
    ((600000, 28, 31, 60), 755, 513), ((600000, 28, 31, 600, 0, 0, 60), 5785, 5372),
    ((600000, 200, 31, 60, 0, 0, 60), 4744, 1341), ((100000, 28, 31, 1), 19, 21)])
def test_measured_calls_take_the_faster_kernel(shape, call, walk, lds):
    assert (shape([_call(*call)])[0][0] > 0) == (lds < walk)


def test_a_call_left_to_k_predict_stays_there(shape):
    """Rows made dense for k_predict are not given to k_predict_lds after all."""
    calls = [c[:-3] for c in (_call(*c) for c in itertools.product(
        (64, 8000, 60000, 200000), (12, 63, 64, 350, 2000, 4000), (15, 63, 255, 900), (1, 5, 20, 200)))]
    csr, made = shape([c + (1, 0.05 * c[1], 0) for c in calls]), shape([c + (2, 0, 0) for c in calls])
    assert all(b[0] == 0 for a, b in zip(csr, made) if a[0] == 0)
