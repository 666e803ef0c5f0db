// predict_shape.h — which prediction kernel a call takes, and the shape of k_predict_lds's
// blocks (host only).
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace lgbm {

constexpr int32_t PRED_TREE_WORDS = 4096;   // packed words of a tree at most, and of a staged batch
constexpr int32_t PRED_THREADS = 1024;      // of a k_predict_lds block
constexpr size_t PRED_LDS = 156 * 1024;     // its LDS at most
constexpr int64_t PRED_FILL = 256;          // blocks before a block takes more rows
constexpr int32_t PRED_STAGE_COLS = 63;     // k_predict stages rows of up to this many columns

struct PredShape {
  int32_t rb, nb;  // rows and staged trees of a block; rb = 0: the call is k_predict's
  size_t lds;
};

// What a call's kernel depends on.
enum PredForm { PRED_DENSE, PRED_CSR, PRED_MADE_DENSE };  // the last: sparse input's rows
struct PredCall {
  int64_t rows;
  int32_t width;       // columns of a row (CSR: the model's, which it is made dense to)
  int32_t tree_words;  // of a packed tree
  int32_t n_trees;
  double leaves;       // of a tree on average
  PredForm form;
  double entries;      // PRED_CSR: of a row on average
  int32_t transformed; // outputs of a row that ConvertOutput goes over again, or 0
};

// Times of the two kernels in microseconds, a launch included.  The constants are fits to 828 dense calls (64 to 1M rows x 12 to 3900
// columns, 1 to 300 trees of 15 to 900 leaves): the kernel that the sums name took at most
// 1.1 times the other's time and a microsecond more, in all but 2 (1.14 and 1.21 times).
inline double predict_time(const PredCall& c) {
  const bool sparse = c.form != PRED_DENSE, staged = c.width <= PRED_STAGE_COLS;
  // rows of mostly zeros take the same shorter walks
  const double levels = c.n_trees * std::log2(std::max(c.leaves, 2.0)) *
                        (!sparse ? 1.0 : staged ? 0.75 : 0.9);
  // nodes past an XCD's L2 are read from further away
  const double far = !sparse && c.n_trees * c.leaves * 32.0 > 4e6 ? 1.4 : 1.0;
  if (staged)
    return 15.0 + (double)c.rows * c.width * 4.0 / 3.3e6 +
           levels * std::max(0.45 * far, 0.25 + 1.9e-6 * (double)c.rows);
  // a line of its row a level: a chain of loads, and the lines of all rows past the caches
  const double bytes = (double)c.rows * std::min(c.width * 4.0, levels * 64.0);
  return 13.5 + levels * ((bytes <= 32e6 ? 0.6 : 1.0) * far +
                          1.4e-5 * (double)c.rows * std::min(1.0, bytes / 300e6));
}
inline double predict_lds_time(const PredCall& c, const PredShape& s) {
  const double rounds = (double)(((c.rows + s.rb - 1) / s.rb + PRED_FILL - 1) / PRED_FILL);
  const int32_t groups = PRED_THREADS / s.rb;
  const double batches = (c.n_trees + s.nb - 1) / s.nb, side = (s.nb + groups - 1) / groups;
  // the rows' staging: latency, or the memory's rate
  const double stage = std::max(rounds * s.rb * c.width / 8192.0,
                                (double)c.rows * c.width * 4.0 / 3.7e6);
  // where each thread has a row, no other block of the CU goes on beside the rows' transform
  const double transform =
      groups == 1 && c.transformed > 1 ? 1.1e-5 * (double)c.rows * c.transformed : 0.0;
  // and a batch's load and its walks
  return 15.0 + stage + transform +
         rounds * batches * (0.8 + 0.2 * side * std::log2(std::max(c.leaves, 2.0)));
}

// Rows and trees a block of k_predict_lds takes: among the row counts that leave the chip a
// block a CU, the one with the most walks side by side (the block's LDS holds fewer trees
// beside more or wider rows), the larger where they tie.
//
// rb = 0 leaves the call to k_predict, where rows or trees do not fit or where it is the
// faster one.  Staging copies all of a row, of which a walk reads a few values, so few trees
// over wide rows are k_predict's: 200k rows x 1000 columns, trees of 31 leaves, k_predict
// and k_predict_lds 1 tree 32 and 231 us, 10 trees 195 and 241, 30 trees 540 and 290.  And
// wide rows leave LDS for few large trees, so that a block's walks are few: 200k rows x 3900
// columns, 300 trees of 255 leaves 9.8 and 30.4 ms (2000 columns 9.1 and 14.3, 1000 columns
// 8.4 and 7.3).  One iteration of many classes, transformed, is k_predict's on many narrow
// rows: 600k x 28, 60 classes 1.74 and 2.08 ms (ten iterations 5.8 and 5.4).
inline PredShape predict_lds_shape(const PredCall& c) {
  PredShape best{0, 0, 0};
  if (c.n_trees < 1 || c.width < 1 || c.tree_words > PRED_TREE_WORDS) return best;
  const size_t tree = (size_t)c.tree_words * 8;
  int32_t walks = 0;
  for (int32_t rb = PRED_THREADS; rb >= 8; rb /= 2) {
    if (rb > 8 && c.rows < (int64_t)rb * PRED_FILL) continue;
    const int32_t groups = PRED_THREADS / rb;
    const size_t x = (size_t)rb * (size_t)(c.width | 1) * 4;
    const size_t per_tree = 2 * tree + (groups > 1 ? (size_t)rb * 16 : 0);
    if (x + per_tree > PRED_LDS) continue;
    int64_t nb = std::min((int64_t)((PRED_LDS - x) / per_tree), (int64_t)PRED_TREE_WORDS / c.tree_words);
    nb = std::min<int64_t>(std::min<int64_t>(nb, c.n_trees), std::max(groups, 8));
    if (rb * (int32_t)std::min<int64_t>(nb, groups) <= walks) continue;
    walks = rb * (int32_t)std::min<int64_t>(nb, groups);
    best = {rb, (int32_t)nb, x + per_tree * (size_t)nb};
  }
  if (best.rb == 0) return best;
  // made dense first: the dense rows' write, or a thread a row that takes its entries in turn
  const double dense = c.form != PRED_CSR ? 0.0 : 15.0 +
      std::max((double)c.rows * c.width * 4.0 / 3.2e6, 1.15 * c.entries);
  if (predict_lds_time(c, best) > 1.05 * (predict_time(c) + dense) - 1.0) return PredShape{0, 0, 0};
  return best;
}

}  // namespace lgbm
