// predict.hip — batch prediction of a LightGBM model over f32 rows, dense or CSR.
//
// A row walks every tree of the requested iteration range on its raw feature values (no
// binning), as the reference predictor does:
//   Tree::get_leaf / numerical_decision / categorical_decision (tree.rs:160-340),
//   GbdtModel::predict_raw (ensemble.rs:75-102): per class an f64 sum over the
//   iterations in order, starting from 0.0 — here each class's trees are added in that
//   order, whichever class comes first,
//   ConvertOutput (objective.rs:241-340) for the transformed kind.
// k_predict_lds walks trees from LDS, several of a row side by side; k_predict, a thread a
// row, has what that does not take and the calls where it is the faster (predict_shape.h).
// Feature contributions (TreeSHAP) go by leaf paths (k_shap_items, k_shap_rows) or, past
// their limits, a thread a row (k_contrib).
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "model.h"

namespace lgbm {

struct PredModelDev {
  const PredNode* nodes;
  const PredTree* trees;
  const double* leaves;
  const int32_t* cat_bounds;
  const uint32_t* cat_words;
  const PredLinLeaf* lin_leaves;
  const int32_t* lin_features;
  const double* lin_coeffs;
};

// The node's fields arrive as values: selecting between members of a struct held by
// reference makes the compiler keep the struct in scratch memory.
__device__ __forceinline__ int32_t pred_next(double thr, int32_t dtype, int32_t left,
                                             int32_t right, double fval, const PredModelDev& M,
                                             int32_t cat0) {
  bool go_left;
  if (dtype & 1) {  // CategoricalDecision (tree.rs:212-237)
    go_left = false;
    if (!isnan(fval)) {
      const int32_t iv = fval >= 2147483647.0 ? 2147483647
                         : fval <= -2147483648.0 ? (int32_t)(-2147483647 - 1)
                                                 : (int32_t)fval;  // saturating `as i32`
      if (iv >= 0) {
        const int32_t ci = (int32_t)thr;  // checked at load: 0 <= ci < num_cat
        const int32_t lo = M.cat_bounds[cat0 + ci], hi = M.cat_bounds[cat0 + ci + 1];
        const int32_t w = iv >> 5;
        go_left = w < hi - lo && ((M.cat_words[lo + w] >> (iv & 31)) & 1u) != 0u;
      }
    }
  } else {  // NumericalDecision (tree.rs:193-210)
    const int32_t mt = (dtype >> 2) & 3;
    if (isnan(fval) && mt != 2) fval = 0.0;
    if ((mt == 1 && fval >= -1e-35 && fval <= 1e-35) || (mt == 2 && isnan(fval)))
      go_left = (dtype & 2) != 0;
    else
      go_left = fval <= thr;
  }
  return go_left ? left : right;
}

// Leaf of tree t for the row at x (a path visits fewer than num_leaves nodes: the
// structure was checked at load).
__device__ __forceinline__ int32_t pred_leaf(const PredModelDev& M, int32_t t, const float* x) {
  const PredTree T = M.trees[t];
  if (T.num_leaves <= 1) return 0;
  int32_t node = 0;
  for (int32_t d = 0; d < T.num_leaves && node >= 0; ++d) {
    const PredNode* nd = M.nodes + T.node0 + node;
    const double thr = nd->threshold;
    const int32_t feat = nd->feature, left = nd->left, right = nd->right, dtype = nd->dtype;
    node = pred_next(thr, dtype, left, right, (double)x[feat], M, T.cat0);
  }
  return node < 0 ? ~node : 0;
}

// Tree::predict (tree.rs:279-316): the leaf's value, or for a linear tree the leaf's
// `leaf_const + sum coeff * x[feature]` in term order (f64, no fused multiply-add),
// falling back to the leaf's value when any of its features is NaN.
__device__ __forceinline__ double pred_tree(const PredModelDev& M, int32_t t, const float* x) {
  const int32_t leaf = pred_leaf(M, t, x);
  const PredTree T = M.trees[t];
  const double lv = M.leaves[T.leaf0 + leaf];
  if (T.lin0 < 0) return lv;
  const PredLinLeaf L = M.lin_leaves[T.lin0 + leaf];
  double v = L.c;
  for (int32_t j = 0; j < L.count; ++j) {
    const double xv = (double)x[M.lin_features[L.start + j]];
    if (isnan(xv)) return lv;
    v += M.lin_coeffs[L.start + j] * xv;
  }
  return v;
}

__device__ __forceinline__ double pred_sigmoid(double x, double s) { return 1.0 / (1.0 + exp(-s * x)); }

// ConvertOutput of one row's raw scores in place.
__device__ __forceinline__ void pred_transform(double* o, int32_t ntpi, int32_t iterations,
                                               int32_t objective, double sigmoid,
                                               int32_t average_output) {
  if (average_output && iterations > 0)  // RF: raw sum / iterations before ConvertOutput
    for (int32_t k = 0; k < ntpi; ++k) o[k] /= (double)iterations;
  switch (objective) {
    case OBJ_REGRESSION_SQRT: {
      const double v = o[0];
      o[0] = (v > 0.0 ? 1.0 : (v < 0.0 ? -1.0 : 0.0)) * v * v;
      break;
    }
    case OBJ_BINARY:
      o[0] = pred_sigmoid(o[0], sigmoid);
      break;
    case OBJ_XENTROPY:
      o[0] = pred_sigmoid(o[0], 1.0);
      break;
    case OBJ_XENTLAMBDA:
      o[0] = log1p(exp(o[0]));
      break;
    case OBJ_EXP:
      o[0] = exp(o[0]);
      break;
    case OBJ_MULTICLASS: {  // Common::Softmax: max subtraction, sum in class order
      double wmax = o[0];
      for (int32_t k = 1; k < ntpi; ++k) wmax = o[k] > wmax ? o[k] : wmax;
      double wsum = 0.0;
      for (int32_t k = 0; k < ntpi; ++k) {
        o[k] = exp(o[k] - wmax);
        wsum += o[k];
      }
      for (int32_t k = 0; k < ntpi; ++k) o[k] /= wsum;
      break;
    }
    case OBJ_MULTICLASS_OVA:
      for (int32_t k = 0; k < ntpi; ++k) o[k] = pred_sigmoid(o[k], sigmoid);
      break;
    default:
      break;
  }
}

// STAGE: rows of up to PRED_STAGE_COLS columns are staged in LDS (256 rows x an odd stride
// of at most 63 floats = 63 KiB): one coalesced load of the block's rows, then every tree
// walk reads its feature values from LDS instead of one cache line per node visit.
template <bool STAGE>
__global__ __launch_bounds__(256) void k_predict(PredModelDev M, const float* __restrict__ X,
                                                 int64_t rows, int32_t cols, int32_t it0,
                                                 int32_t it1, int32_t ntpi, int32_t kind,
                                                 int32_t objective, double sigmoid,
                                                 int32_t average_output, int32_t es_freq,
                                                 double es_margin, int32_t* __restrict__ es_iters,
                                                 double* __restrict__ out,
                                                 int32_t* __restrict__ leaf_out) {
  extern __shared__ float s_x[];
  const int64_t r0 = (int64_t)blockIdx.x * blockDim.x;
  const int64_t r = r0 + threadIdx.x;
  const float* x;
  if (STAGE) {
    const int32_t stride = cols | 1;  // odd: lanes' rows fall in different banks
    const int32_t total = (int32_t)(min((int64_t)blockDim.x, rows - r0) * cols);
    const float* src = X + r0 * cols;
    for (int32_t i = threadIdx.x; i < total; i += blockDim.x) {
      const int32_t rr = i / cols;
      s_x[rr * stride + (i - rr * cols)] = src[i];
    }
    __syncthreads();
    if (r >= rows) return;
    x = s_x + threadIdx.x * stride;
  } else {
    if (r >= rows) return;
    x = X + r * cols;
  }
  if (kind == 2) {
    const int64_t nt = (int64_t)(it1 - it0) * ntpi;
    for (int32_t i = it0; i < it1; ++i)
      for (int32_t k = 0; k < ntpi; ++k)
        leaf_out[r * nt + (int64_t)(i - it0) * ntpi + k] = pred_leaf(M, i * ntpi + k, x);
    return;
  }
  double* o = out + r * ntpi;
  if (es_freq > 0) {
    // GbdtModel::predict_raw_early_stop (ensemble.rs:120-151): iterations in order,
    // each adding its trees class by class; every es_freq iterations the margin
    // test of pred_early_stop_should_stop (ensemble.rs:337-356) may end the row
    for (int32_t k = 0; k < ntpi; ++k) o[k] = 0.0;
    int32_t counter = 0, evaluated = 0;
    for (int32_t i = it0; i < it1; ++i) {
      for (int32_t k = 0; k < ntpi; ++k) {
        const int32_t t = i * ntpi + k;
        o[k] += pred_tree(M, t, x);
      }
      ++evaluated;
      if (++counter == es_freq) {
        bool stop;
        if (ntpi == 1) {
          stop = 2.0 * fabs(o[0]) > es_margin;
        } else {
          double top1 = -__builtin_inf(), top2 = -__builtin_inf();
          for (int32_t k = 0; k < ntpi; ++k) {
            const double v = o[k];
            if (v > top1) {
              top2 = top1;
              top1 = v;
            } else if (v > top2) {
              top2 = v;
            }
          }
          stop = (top1 - top2) > es_margin;
        }
        if (stop) break;
        counter = 0;
      }
    }
    es_iters[r] = evaluated;
    return;
  }
  for (int32_t k = 0; k < ntpi; ++k) {
    double acc = 0.0;
    for (int32_t i = it0; i < it1; ++i) {
      const int32_t t = i * ntpi + k;
      acc += pred_tree(M, t, x);
    }
    o[k] = acc;
  }
  if (kind == 1) pred_transform(o, ntpi, it1 - it0, objective, sigmoid, average_output);
}

// ---- trees and rows in LDS --------------------------------------------------------------
// The usual prediction (no early stop, constant leaves, trees that fit): a block stages
// `rb` rows and walks the trees, a few at a time, from LDS too.  A node is one 8-byte
// word pair (model.h) and its children are neighbours, so a step is two LDS reads (the
// node, the row's value) and 15 VALU instructions, where k_predict gathers 24 bytes a
// node from L2.  Thresholds are f32: for an f32 value v, v <= thr exactly when v <= the
// largest float not above thr.
//
// The 1024 threads are rb rows x 1024 / rb groups of trees.  With one group a row's thread
// walks the trees class by class and adds their values as k_predict does.  With few rows,
// or wide ones, a group walks every (1024 / rb)-th tree of a batch and leaves the leaf
// values in LDS, from which a thread per row and class adds the batch's in tree order,
// while the next batch is walked.
//
// Measured against k_predict: 2M rows x 28 columns, 100 trees of 255 leaves 3.31 -> 1.53
// ms, now bound by the chain of a walk's reads, which four waves a SIMD do not cover (of the
// CUs' busy cycles VALU 67 %, LDS 35 %, four tenths of it conflicts; waves wait 59 % of
// theirs); 64 rows, 100 trees of 31 leaves 273 -> 14 us (one thread walked all trees); 200003 CSR
// rows x 500 columns, 200 trees of 63 leaves 3.84 (with the densify) -> 1.00 ms.  Blocks
// of half the LDS, two a CU, took 2.55 ms on the first and 2.10 on the third.
constexpr int32_t PRED_WORDS = PRED_TREE_WORDS / PRED_THREADS;  // a thread stages of a batch

// NODES: 0 nodes without these flags only, 1 PRED_ZERO_MISSING ones too, 2 any.  Branch-
// free but for sets of more than a word: a wave's lanes meet all kinds at every step.
template <int NODES>
__device__ __forceinline__ int32_t pred_walk(const uint2* nodes, const float* x,
                                             const PredModelDev& M, bool sets) {
  // one 8-byte read an entry: as two words the compiler would read them apart
  auto entry = [&](uint32_t i) { return *(const unsigned long long*)(nodes + i); };
  unsigned long long e = entry(0);
  for (;;) {
    const uint32_t t = (uint32_t)e, w = (uint32_t)(e >> 32);
    if ((w & 0xffffu) == 0u) return (int32_t)t;
    const float v = x[(w >> 16) & 0xfffu];
    float u = v;
    if constexpr (NODES >= 1) {
      // the smallest float above 1e-35, or 0 (below which nothing is)
      const uint32_t tiny = (uint32_t)((int32_t)(w << 1) >> 31) & 0x0554ad2eu;
      if (fabsf(v) < __uint_as_float(tiny)) u = __builtin_nanf("");
    }
    bool second = __uint_as_float(__float_as_uint(u) ^ (w & PRED_FLIP)) > __uint_as_float(t);
    if constexpr (NODES >= 2) {
      // v truncated (above -1 to 0): a NaN, a negative or a larger one is in no set
      const bool in = v > -1.0f && v < 32.0f;
      const uint32_t bit = in ? t >> ((uint32_t)(int32_t)v & 31u) : 0u;
      if (w & PRED_CATEGORICAL) second = (bit & 1u) == 0u;
      if (sets && (w & PRED_SET)) second = pred_next(0.0, 1, 0, 1, (double)v, M, (int32_t)t) != 0;
    }
    e = entry((w & 0xffffu) + (second ? 1u : 0u));
  }
}

// Where the rows come from: a dense matrix, or CSR rows made dense in LDS.  In the CSR
// form a cell first takes the largest position + 1 of its entries (the last of a repeated
// column wins), then that entry's value; a bad indptr pair or column sets its bit of *err
// and the host drops the call's results.
template <bool CSR, int NODES>
__global__ __launch_bounds__(PRED_THREADS) void k_predict_lds(
    PredModelDev M, PredPack K, PredRows R, int64_t rows, int32_t width, int32_t rb, int32_t nb,
    int32_t it0, int32_t it1, int32_t ntpi, int32_t kind, int32_t objective, double sigmoid,
    int32_t average_output, double* __restrict__ out, int32_t* __restrict__ leaf_out) {
  extern __shared__ __align__(16) uint2 pred_lds[];
  const int tid = (int)threadIdx.x;
  const int groups = PRED_THREADS / rb, row = tid & (rb - 1), g = tid / rb;
  const int batch = nb * K.stride;  // words
  double* val = (double*)(pred_lds + 2 * batch);  // [2][nb][rb]
  float* x = (float*)(val + (groups > 1 ? 2 * nb * rb : 0));
  const int stride = width | 1;  // odd: the rows of a wave's lanes start in different banks
  const int64_t r0 = (int64_t)blockIdx.x * rb;
  const int nrow = (int)min((int64_t)rb, rows - r0);
  const int n_it = it1 - it0, total = n_it * ntpi;
  // this thread's words of a batch: (tree of the batch, word of the tree)
  int wt[PRED_WORDS], ww[PRED_WORDS];
  uint2 word[PRED_WORDS];
#pragma unroll
  for (int u = 0; u < PRED_WORDS; ++u) {
    const int q = tid + u * PRED_THREADS;
    wt[u] = q < batch ? q / K.stride : INT32_MAX;
    ww[u] = q < batch ? q - wt[u] * K.stride : 0;
  }
  // the p-th tree walked: in tree order, or class by class where fewer groups than classes
  // leave a thread more than one class to add
  const bool by_class = groups < ntpi;
  auto tree_of = [&](int p) {
    const int k = by_class ? p / n_it : 0;
    return by_class ? (int64_t)(it0 + p - k * n_it) * ntpi + k : (int64_t)it0 * ntpi + p;
  };
  auto load = [&](int p0) {
    const int nt = min(nb, total - p0);
    const uint2* src = K.words + ((int64_t)it0 * ntpi + p0) * K.stride + tid;
#pragma unroll
    for (int u = 0; u < PRED_WORDS; ++u)
      if (wt[u] < nt)
        word[u] = by_class ? K.words[tree_of(p0 + wt[u]) * K.stride + ww[u]] : src[u * PRED_THREADS];
  };
  auto store = [&](int p0, uint2* buf) {
#pragma unroll
    for (int u = 0; u < PRED_WORDS; ++u)
      if (wt[u] < min(nb, total - p0)) buf[tid + u * PRED_THREADS] = word[u];
  };
  load(0);
  if constexpr (CSR) {
    uint32_t* claim = (uint32_t*)x;
    for (int i = tid; i < nrow * stride; i += PRED_THREADS) claim[i] = 0u;
    __syncthreads();
    int64_t lo = 0, hi = 0;
    if (row < nrow) {
      lo = R.indptr[r0 + row];
      hi = R.indptr[r0 + row + 1];
      if (lo < 0 || hi < lo || hi > R.nnz) {
        if (g == 0) atomicOr(R.err, 1u);
        hi = lo;
      }
    }
    for (int64_t k = lo + g; k < hi; k += groups) {
      const int32_t c = R.indices[k];
      if (c < 0 || c >= R.cols)
        atomicOr(R.err, 2u);
      else if (c < width)
        atomicMax(&claim[row * stride + c], (uint32_t)(k - lo + 1));
    }
    __syncthreads();
    const int64_t base = lo;  // a thread fills cells of its own row
    if (row < nrow)
      for (int c = g; c < width; c += groups) {
        const uint32_t u = claim[row * stride + c];
        x[row * stride + c] = u ? R.values[base + (u - 1)] : 0.0f;
      }
  } else {
    // the block's rows are consecutive floats: a thread's (row, column) advance without a
    // division, eight loads in flight
    constexpr int B = 8;
    const float* src = R.dense + r0 * width;
    int rr = tid / width, c = tid - rr * width;
    const int dr = PRED_THREADS / width, dc = PRED_THREADS - dr * width, n = nrow * width;
    for (int i0 = tid; i0 < n; i0 += B * PRED_THREADS) {
      float v[B];
#pragma unroll
      for (int u = 0; u < B; ++u) v[u] = i0 + u * PRED_THREADS < n ? src[i0 + u * PRED_THREADS] : 0.0f;
#pragma unroll
      for (int u = 0; u < B; ++u) {
        if (i0 + u * PRED_THREADS < n) x[rr * stride + c] = v[u];
        rr += dr;
        c += dc;
        if (c >= width) {
          c -= width;
          ++rr;
        }
      }
    }
  }
  store(0, pred_lds);
  __syncthreads();
  const bool live = row < nrow, sets = K.set != 0;
  const float* xr = x + row * stride;
  const int64_t r = r0 + row;
  double acc = 0.0;
  // by class: the class being added and its trees to come
  int32_t cls = 0, todo = n_it;
  auto add = [&](double v) {
    acc += v;
    if (--todo == 0) {
      out[r * ntpi + cls] = acc;
      acc = 0.0;
      ++cls;
      todo = n_it;
    }
  };
  for (int p0 = 0, b = 0; p0 < total; p0 += nb, b ^= 1) {
    const uint2* buf = pred_lds + b * batch;
    double* vals = val + b * nb * rb + row;
    const int nt = min(nb, total - p0);
    load(p0 + nb);
    if (live)
      for (int j = g; j < nt; j += groups) {
        const uint2* tree = buf + j * K.stride;
        const int32_t leaf = pred_walk<NODES>(tree, xr, M, sets);
        if (kind == 2) {
          leaf_out[r * total + tree_of(p0 + j) - (int64_t)it0 * ntpi] = leaf;
          continue;
        }
        const double v = *(const double*)(tree + K.values + leaf);
        if (groups > 1)
          vals[j * rb] = v;
        else
          add(v);
      }
    store(p0 + nb, pred_lds + (b ^ 1) * batch);
    __syncthreads();
    if (groups == 1 || !live || kind == 2) continue;
    if (by_class) {
      if (g == 0)
        for (int j = 0; j < nt; ++j) add(vals[j * rb]);
    } else if (g < ntpi) {
      // class g's trees of the batch, eight reads in flight
      constexpr int B = 8;
      for (int j = (g - p0 % ntpi + ntpi) % ntpi; j < nt; j += B * ntpi) {
        double v[B];
#pragma unroll
        for (int u = 0; u < B; ++u) v[u] = j + u * ntpi < nt ? vals[(j + u * ntpi) * rb] : 0.0;
#pragma unroll
        for (int u = 0; u < B; ++u)
          if (j + u * ntpi < nt) acc += v[u];
      }
    }
  }
  if (groups > 1 && !by_class && kind != 2) {
    if (live && g < ntpi) out[r * ntpi + g] = acc;
    __syncthreads();  // a row's classes, for its transform
  }
  if (kind == 1 && live && g == 0)
    pred_transform(out + r * ntpi, ntpi, n_it, objective, sigmoid, average_output);
}

// Opts the kernels into their LDS; 0 = ok.
int predict_lds_prepare() {
  const void* k[6] = {(const void*)k_predict_lds<false, 0>, (const void*)k_predict_lds<false, 1>,
                      (const void*)k_predict_lds<false, 2>, (const void*)k_predict_lds<true, 0>,
                      (const void*)k_predict_lds<true, 1>, (const void*)k_predict_lds<true, 2>};
  for (const void* f : k)
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)PRED_LDS) != hipSuccess)
      return 1;
  return 0;
}

// `csr`: the rows are R's CSR entries made `width` columns wide, else R.dense's.
void launch_predict_lds(const PredShape& S, const PredPack& K, const int32_t* cat_bounds,
                        const uint32_t* cat_words, const PredRows& R, bool csr, int64_t rows,
                        int32_t width, int32_t it0, int32_t it1, int32_t ntpi, int32_t kind,
                        int32_t objective, double sigmoid, int32_t average_output, double* out,
                        int32_t* leaf_out, hipStream_t s, const KernelEvents* ev) {
  const PredModelDev M{nullptr, nullptr, nullptr, cat_bounds, cat_words, nullptr, nullptr, nullptr};
  const dim3 g((unsigned)((rows + S.rb - 1) / S.rb)), b(PRED_THREADS);
  const int nodes = K.cat ? 2 : K.zero ? 1 : 0;
#define PRED_LDS_LAUNCH(C, N)                                                                \
  if (csr == C && nodes == N)                                                                 \
  KLAUNCH(ev, (k_predict_lds<C, N>), g, b, S.lds, s, M, K, R, rows, width, S.rb, S.nb, it0, it1, \
          ntpi, kind, objective, sigmoid, average_output, out, leaf_out)
  PRED_LDS_LAUNCH(false, 0);
  PRED_LDS_LAUNCH(false, 1);
  PRED_LDS_LAUNCH(false, 2);
  PRED_LDS_LAUNCH(true, 0);
  PRED_LDS_LAUNCH(true, 1);
  PRED_LDS_LAUNCH(true, 2);
#undef PRED_LDS_LAUNCH
}

// ---- feature contributions (TreeSHAP) ------------------------------------------------
// Lundberg et al., arXiv:1706.06060, Algorithm 2, as the reference computes it
// (Tree::predict_contrib / extend_path / unwind_path / unwound_path_sum / tree_shap,
// tree.rs:400-583): one thread per row, the recursion turned into a loop over the hot
// child with a stack of pending cold calls (popped in the recursion's order, so every
// f64 update happens in the same sequence), and every product and quotient in the
// reference's association (this file is built without fused multiply-add).
//
// Each thread's unique paths live in one flat buffer of (D+1)(D+2)/2 elements for the
// deepest tree D, as in the reference: a call's frame starts `d` elements after its
// parent's and copies the parent's first `d` elements; the cold call reads its parent's
// frame after the hot subtree returns, which wrote only past it.  The buffers are
// workspace memory laid out element-major (element k of thread i at k * stride + i), so
// a wave's accesses to one element are contiguous.
struct ShapWork {
  int32_t* feat;
  double* zero;
  double* one;
  double* pw;
  int32_t* s_node;  // pending cold calls: node, parent frame base, depth, split feature
  int32_t* s_base;
  int32_t* s_depth;
  int32_t* s_feat;
  double* s_zero;
  int64_t stride;  // threads of the launch
};

struct ShapModelDev {
  const double* node_cover;
  const double* leaf_cover;
  const double* expected;
};

__device__ __forceinline__ void shap_extend(const ShapWork& W, int64_t i0, int32_t b, int32_t d,
                                            double zf, double of, int32_t feat) {
  const int64_t e = (int64_t)(b + d) * W.stride + i0;
  W.feat[e] = feat;
  W.zero[e] = zf;
  W.one[e] = of;
  W.pw[e] = d == 0 ? 1.0 : 0.0;
  const double dd = (double)d;
  for (int32_t i = d - 1; i >= 0; --i) {
    const int64_t ei = (int64_t)(b + i) * W.stride + i0;
    const double prev = W.pw[ei];
    W.pw[ei + W.stride] += of * prev * ((double)i + 1.0) / (dd + 1.0);
    W.pw[ei] = zf * prev * (dd - (double)i) / (dd + 1.0);
  }
}

__device__ __forceinline__ void shap_unwind(const ShapWork& W, int64_t i0, int32_t b, int32_t d,
                                            int32_t k) {
  const int64_t ek = (int64_t)(b + k) * W.stride + i0;
  const double of = W.one[ek], zf = W.zero[ek];
  double next = W.pw[(int64_t)(b + d) * W.stride + i0];
  const double dd = (double)d;
  for (int32_t i = d - 1; i >= 0; --i) {
    const int64_t ei = (int64_t)(b + i) * W.stride + i0;
    if (of != 0.0) {
      const double tmp = W.pw[ei];
      W.pw[ei] = next * (dd + 1.0) / (((double)i + 1.0) * of);
      next = tmp - W.pw[ei] * zf * (dd - (double)i) / (dd + 1.0);
    } else {
      W.pw[ei] = (W.pw[ei] * (dd + 1.0)) / (zf * (dd - (double)i));
    }
  }
  for (int32_t i = k; i < d; ++i) {
    const int64_t ei = (int64_t)(b + i) * W.stride + i0;
    W.feat[ei] = W.feat[ei + W.stride];
    W.zero[ei] = W.zero[ei + W.stride];
    W.one[ei] = W.one[ei + W.stride];
  }
}

__device__ __forceinline__ double shap_unwound_sum(const ShapWork& W, int64_t i0, int32_t b,
                                                   int32_t d, int32_t k) {
  const int64_t ek = (int64_t)(b + k) * W.stride + i0;
  const double of = W.one[ek], zf = W.zero[ek];
  double next = W.pw[(int64_t)(b + d) * W.stride + i0];
  double total = 0.0;
  const double dd = (double)d;
  for (int32_t i = d - 1; i >= 0; --i) {
    const double pwi = W.pw[(int64_t)(b + i) * W.stride + i0];
    if (of != 0.0) {
      const double tmp = next * (dd + 1.0) / (((double)i + 1.0) * of);
      total += tmp;
      next = pwi - tmp * zf * ((dd - (double)i) / (dd + 1.0));
    } else {
      total += (pwi / zf) / ((dd - (double)i) / (dd + 1.0));
    }
  }
  return total;
}

__global__ __launch_bounds__(256) void k_contrib(PredModelDev M, ShapModelDev S, ShapWork W,
                                                 const float* __restrict__ X, int64_t r0,
                                                 int64_t rows, int32_t cols, int32_t nf,
                                                 int32_t it0, int32_t it1, int32_t ntpi,
                                                 double* __restrict__ out) {
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t r = r0 + i0;
  if (i0 >= W.stride || r >= rows) return;
  const float* x = X + r * cols;
  const int32_t block = nf + 1;
  double* o = out + r * (int64_t)ntpi * block;
  for (int32_t j = 0; j < ntpi * block; ++j) o[j] = 0.0;
  for (int32_t it = it0; it < it1; ++it) {
    for (int32_t k = 0; k < ntpi; ++k) {
      const int32_t t = it * ntpi + k;
      double* phi = o + k * block;
      phi[nf] += S.expected[t];
      const PredTree T = M.trees[t];
      if (T.num_leaves <= 1) continue;
      int32_t node = 0, pb = 0, d = 0, pf = -1, sp = 0;
      double pz = 1.0, po = 1.0;
      for (;;) {
        const int32_t b = pb + d;
        for (int32_t i = 0; i < d; ++i) {
          const int64_t src = (int64_t)(pb + i) * W.stride + i0, dst = (int64_t)(b + i) * W.stride + i0;
          W.feat[dst] = W.feat[src];
          W.zero[dst] = W.zero[src];
          W.one[dst] = W.one[src];
          W.pw[dst] = W.pw[src];
        }
        shap_extend(W, i0, b, d, pz, po, pf);
        if (node < 0) {
          const double lv = M.leaves[T.leaf0 + ~node];
          for (int32_t i = 1; i <= d; ++i) {
            const double w = shap_unwound_sum(W, i0, b, d, i);
            const int64_t ei = (int64_t)(b + i) * W.stride + i0;
            phi[W.feat[ei]] += w * (W.one[ei] - W.zero[ei]) * lv;
          }
          if (sp == 0) break;
          --sp;
          const int64_t es = (int64_t)sp * W.stride + i0;
          node = W.s_node[es];
          pb = W.s_base[es];
          d = W.s_depth[es];
          pf = W.s_feat[es];
          pz = W.s_zero[es];
          po = 0.0;
          continue;
        }
        const PredNode* nd = M.nodes + T.node0 + node;
        const double thr = nd->threshold;
        const int32_t f = nd->feature, left = nd->left, right = nd->right, dtype = nd->dtype;
        const int32_t hot = pred_next(thr, dtype, left, right, (double)x[f], M, T.cat0);
        const int32_t cold = hot == left ? right : left;
        const double w = S.node_cover[T.node0 + node];
        const double hc = hot >= 0 ? S.node_cover[T.node0 + hot] : S.leaf_cover[T.leaf0 + ~hot];
        const double cc = cold >= 0 ? S.node_cover[T.node0 + cold] : S.leaf_cover[T.leaf0 + ~cold];
        const double hz = hc / w, cz = cc / w;
        double iz = 1.0, io = 1.0;
        int32_t pi = 0;
        while (pi <= d && W.feat[(int64_t)(b + pi) * W.stride + i0] != f) ++pi;
        int32_t nd1 = d;
        if (pi != d + 1) {
          const int64_t ep = (int64_t)(b + pi) * W.stride + i0;
          iz = W.zero[ep];
          io = W.one[ep];
          shap_unwind(W, i0, b, d, pi);
          nd1 -= 1;
        }
        const int64_t es = (int64_t)sp * W.stride + i0;
        W.s_node[es] = cold;
        W.s_base[es] = b;
        W.s_depth[es] = nd1 + 1;
        W.s_feat[es] = f;
        W.s_zero[es] = cz * iz;
        ++sp;
        node = hot;
        pb = b;
        d = nd1 + 1;
        pz = hz * iz;
        po = io;
        pf = f;
      }
    }
  }
}

// ---- feature contributions by leaf paths ---------------------------------------------
// What a leaf adds to a row's contributions depends on the row only through the ancestors
// at which the row goes the leaf's way: the unique path's features and zero fractions are
// the leaf's own, its one fractions are 0 or 1.  So the work is done per (leaf, item) and
// not per (leaf, row): an item is one of the 2^depth outcomes of the leaf's ancestors, or
// a row where the rows are fewer.  k_shap_items runs the recursion's own sequence of
// extends and unwinds along one root-to-leaf path per item and writes the m values
// `w * (one - zero) * leaf_value` of the path's m features; k_shap_rows adds them up for
// every row in the recursion's order.
//
// The recursion visits leaves hot child first, and each feature's f64 sum keeps that
// order: a leaf's position in it is the number of leaves in the hot siblings of those of
// its ancestors' children that the row does not take.  Every f64 operation is the
// recursion's, so the sums are too.
//
// 50000 rows x 100 trees of 31 leaves (28 features): the one-thread-per-row kernel
// (k_contrib, kept for deeper and wider trees) took 201.5 ms, bound by its path buffers
// in memory, 28 bytes an element and quadratic in the depth.  Here the values take 0.10
// ms and the sums 2.45 ms, bound by the latency of the gathers per leaf (waves wait 71 % of
// their cycles) and by LDS (57 % of the CUs' busy cycles, seven tenths of it conflicts).
constexpr int32_t SHAP_LANES = 8;  // lanes a row: unique paths are mostly this short
constexpr size_t SHAP_LDS = 64 * 1024;

// LDS stores of the wave's lanes before, loads after (one wave, in order).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Block = one wave: leaf leaf0 + blockIdx.x, 64 items at a time.  Everything but the path
// weights and the one fractions (a bit per element) is the same in all lanes.
__global__ __launch_bounds__(LGBM_WAVE) void k_shap_items(
    PredModelDev M, ShapModelDev S, const ShapLeaf* __restrict__ leaves,
    const ShapStep* __restrict__ steps, const ShapPlan* __restrict__ plan, int32_t leaf0,
    const float* __restrict__ X, int64_t rows, int32_t cols, double* __restrict__ tab) {
  constexpr int D = SHAP_MAX_DEPTH + 1;
  __shared__ double pw[D][LGBM_WAVE];
  __shared__ double zero[D], ratio[D];
  __shared__ int32_t feat[D];
  const int32_t leaf = leaf0 + (int32_t)blockIdx.x;
  const ShapLeaf L = leaves[leaf];
  const ShapPlan P = plan[leaf];
  const int32_t depth = L.dm & 0xffff, m = L.dm >> 16;
  const bool by_row = (P.items & SHAP_BY_ROW) != 0u;
  // the plan's row chunk can be larger than the last one
  const int64_t items = by_row ? min((int64_t)(P.items & ~SHAP_BY_ROW), rows) : (int64_t)P.items;
  const int lane = (int)threadIdx.x;
  const int32_t cat0 = M.trees[L.tree].cat0;
  const double lv = M.leaves[leaf];
  for (int64_t i0 = (int64_t)blockIdx.y * LGBM_WAVE; i0 < items; i0 += (int64_t)gridDim.y * LGBM_WAVE) {
    const int64_t item = i0 + lane;
    uint32_t hot = (uint32_t)item;  // bit j: the row goes the leaf's way at ancestor j
    if (by_row) {
      hot = 0u;
      const float* x = X + min(item, items - 1) * cols;
      for (int32_t j = 0; j < depth; ++j) {
        const ShapStep st = steps[L.path0 + j];
        const PredNode nd = M.nodes[st.node];
        const int32_t next = pred_next(nd.threshold, nd.dtype, nd.left, nd.right,
                                       (double)x[nd.feature], M, cat0);
        hot |= (next == ((st.other & 1) ? nd.right : nd.left) ? 1u : 0u) << j;
      }
    }
    int32_t d = 0;
    uint32_t one = 1u;  // bit i: the one fraction of element i
    feat[0] = -1;
    zero[0] = 1.0;
    pw[0][lane] = 1.0;
    for (int32_t j = 0; j < depth; ++j) {
      const int32_t node = steps[L.path0 + j].node;
      const int32_t f = M.nodes[node].feature;
      const double cover = j + 1 < depth ? S.node_cover[steps[L.path0 + j + 1].node] : S.leaf_cover[leaf];
      const double share = cover / S.node_cover[node];
      wave_lds_sync();
      double iz = 1.0;
      uint32_t io = 1u;
      int32_t pi = 0;
      while (pi <= d && feat[pi] != f) ++pi;
      if (pi <= d) {  // UnwindPath of the feature's earlier element
        iz = zero[pi];
        io = (one >> pi) & 1u;
        const double dd = (double)d;
        double next = pw[d][lane];
        for (int32_t i = d - 1; i >= 0; --i) {
          if (io) {
            const double tmp = pw[i][lane];
            const double v = next * (dd + 1.0) / (((double)i + 1.0) * 1.0);
            pw[i][lane] = v;
            next = tmp - v * iz * (dd - (double)i) / (dd + 1.0);
          } else {
            pw[i][lane] = (pw[i][lane] * (dd + 1.0)) / (iz * (dd - (double)i));
          }
        }
        for (int32_t i = pi; i < d; ++i) {
          feat[i] = feat[i + 1];
          zero[i] = zero[i + 1];
        }
        one = (one & ((1u << pi) - 1u)) | ((one >> (pi + 1)) << pi);
        d -= 1;
      }
      // ExtendPath
      d += 1;
      const double zf = share * iz;
      const bool is_hot = ((hot >> j) & 1u) != 0u;
      const uint32_t of = is_hot ? io : 0u;
      wave_lds_sync();
      feat[d] = f;
      zero[d] = zf;
      one = (one & ((1u << d) - 1u)) | (of << d);
      pw[d][lane] = 0.0;
      const double dd = (double)d, o = of ? 1.0 : 0.0;
      for (int32_t i = d - 1; i >= 0; --i) {
        const double prev = pw[i][lane];
        pw[i + 1][lane] += o * prev * ((double)i + 1.0) / (dd + 1.0);
        pw[i][lane] = zf * prev * (dd - (double)i) / (dd + 1.0);
      }
    }
    if (lane < d) ratio[lane] = ((double)d - (double)lane) / ((double)d + 1.0);
    wave_lds_sync();
    if (item < items) {
      double* out = tab + P.off + item * m;
      for (int32_t k = 1; k <= d; ++k) {  // UnwoundPathSum of each element
        const double zf = zero[k], dd = (double)d;
        const bool of = ((one >> k) & 1u) != 0u;
        double total = 0.0;
        if (of) {
          double next = pw[d][lane];
          for (int32_t i = d - 1; i >= 0; --i) {
            const double tmp = next * (dd + 1.0) / (((double)i + 1.0) * 1.0);
            total += tmp;
            next = pw[i][lane] - tmp * zf * ratio[i];
          }
        } else {
          for (int32_t i = d - 1; i >= 0; --i) total += (pw[i][lane] / zf) / ratio[i];
        }
        out[k - 1] = total * ((of ? 1.0 : 0.0) - zf) * lv;
      }
    }
    wave_lds_sync();
  }
}

// LDS of a row of k_shap_rows: its sums (one class), the leaves in the recursion's order,
// and the outcome of every node.
__host__ __device__ inline size_t shap_row_lds(int32_t nf, int32_t max_leaves) {
  return (size_t)(nf + 1) * 8 + (size_t)max_leaves * 8 + ((size_t)max_leaves + 7) / 8 * 8;
}

// SHAP_LANES lanes a row.  Per tree: the lanes evaluate its nodes (a ballot keeps the
// outcomes), place its leaves in the recursion's order with the offset of the row's
// values, and then add leaf after leaf, a lane a feature, four leaves' loads in flight.
__global__ __launch_bounds__(256) void k_shap_rows(
    PredModelDev M, ShapModelDev S, const ShapLeaf* __restrict__ leaves,
    const ShapStep* __restrict__ steps, const int32_t* __restrict__ feats,
    const ShapPlan* __restrict__ plan, const double* __restrict__ tab,
    const float* __restrict__ X, int64_t rows, int32_t cols, int32_t nf, int32_t max_leaves,
    int32_t t0, int32_t t1, int32_t ntpi, int32_t first, double* __restrict__ out) {
  extern __shared__ __align__(16) char shap_lds[];
  constexpr int G = SHAP_LANES;
  const int gl = (int)threadIdx.x & (G - 1), slot = (int)threadIdx.x / G;
  const int shift = (int)lane_id() & ~(G - 1);
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x / G) + slot;
  const bool live = row < rows;
  const int64_t r = live ? row : rows - 1;  // a stand-in, written nowhere
  char* mine = shap_lds + (size_t)slot * shap_row_lds(nf, max_leaves);
  double* phi = (double*)mine;
  uint2* order = (uint2*)(phi + nf + 1);
  uint8_t* left = (uint8_t*)(order + max_leaves);
  const float* x = X + r * cols;
  const int32_t block = nf + 1;
  for (int32_t k = 0; k < ntpi; ++k) {
    double* o = out + (r * ntpi + k) * (int64_t)block;
    for (int32_t j = gl; j < block; j += G) phi[j] = first ? 0.0 : o[j];
    for (int32_t t = t0 + (k - t0 % ntpi + ntpi) % ntpi; t < t1; t += ntpi) {
      wave_lds_sync();
      if (gl == 0) phi[nf] += S.expected[t];
      const PredTree T = M.trees[t];
      const int32_t nl = T.num_leaves;
      if (nl <= 1) continue;
      for (int32_t b = 0; b < nl - 1; b += G) {
        const int32_t n = b + gl;
        bool go = false;
        if (n < nl - 1) {
          const PredNode nd = M.nodes[T.node0 + n];
          go = pred_next(nd.threshold, nd.dtype, 1, 0, (double)x[nd.feature], M, T.cat0) != 0;
        }
        const unsigned long long m = __ballot(go);
        if (gl == 0) left[b / G] = (uint8_t)(m >> shift);
      }
      wave_lds_sync();
      for (int32_t l = gl; l < nl; l += G) {
        const ShapLeaf L = leaves[T.leaf0 + l];
        const ShapPlan P = plan[T.leaf0 + l];
        const int32_t depth = L.dm & 0xffff;
        uint32_t hot = 0u, rank = 0u;
        for (int32_t j = 0; j < depth; ++j) {
          const ShapStep st = steps[L.path0 + j];
          const int32_t n = st.node - T.node0;
          const bool h = (((left[n / G] >> (n & (G - 1))) & 1) != 0) != ((st.other & 1) != 0);
          hot |= (h ? 1u : 0u) << j;
          rank += h ? 0u : (uint32_t)(st.other >> 1);
        }
        const uint32_t m = (uint32_t)(L.dm >> 16);
        const uint32_t item = (P.items & SHAP_BY_ROW) ? (uint32_t)r : hot;
        order[rank] = make_uint2(P.off + item * m, ((uint32_t)L.feat0 << 5) | m);
      }
      wave_lds_sync();
      constexpr int B = 4;
      for (int32_t q0 = 0; q0 < nl; q0 += B) {
        uint2 e[B];
        double c[B];
        int32_t f[B];
#pragma unroll
        for (int u = 0; u < B; ++u) e[u] = q0 + u < nl ? order[q0 + u] : make_uint2(0u, 0u);
#pragma unroll
        for (int u = 0; u < B; ++u) {
          const bool in = gl < (int)(e[u].y & 31u);
          c[u] = in ? tab[e[u].x + gl] : 0.0;
          f[u] = in ? feats[(e[u].y >> 5) + gl] : -1;
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
          // a leaf's features are its path's own, but the leaf before may have met one of
          // them in another lane: its adds come first
          wave_lds_sync();
          if (f[u] >= 0) phi[f[u]] += c[u];
          for (int i = gl + G; i < (int)(e[u].y & 31u); i += G)
            phi[feats[(e[u].y >> 5) + i]] += tab[e[u].x + i];
        }
      }
    }
    wave_lds_sync();
    if (live)
      for (int32_t j = gl; j < block; j += G) o[j] = phi[j];
  }
}

// Rows a block of k_shap_rows, 0 where a row's LDS is too large for it.
int32_t shap_rows_per_block(int32_t nf, int32_t max_leaves) {
  for (int32_t rpb = 256 / SHAP_LANES; rpb * SHAP_LANES >= LGBM_WAVE; rpb /= 2)
    if (shap_row_lds(nf, max_leaves) * (size_t)rpb <= SHAP_LDS) return rpb;
  return 0;
}

// Trees [t0, t1) whose leaves are [leaf0, leaf1), over rows [0, rows) of X: their values
// into `tab`, then the rows' sums (continued from `out` unless `first`).  `leaves` and `plan`
// are indexed by a leaf's number in the model; only those leaves' are read.
void launch_shap_paths(const PredNode* nodes, const PredTree* trees, const double* leaf_values,
                       const int32_t* cat_bounds, const uint32_t* cat_words,
                       const double* node_cover, const double* leaf_cover, const double* expected,
                       const ShapLeaf* leaves, const ShapStep* steps, const int32_t* feats,
                       const ShapPlan* plan, int64_t max_items, const float* X, int64_t rows,
                       int32_t cols, int32_t nf, int32_t max_leaves, int32_t t0, int32_t t1,
                       int32_t leaf0, int32_t leaf1, int32_t ntpi, int first, double* tab,
                       double* out, hipStream_t s) {
  const PredModelDev M{nodes, trees, leaf_values, cat_bounds, cat_words, nullptr, nullptr, nullptr};
  const ShapModelDev S{node_cover, leaf_cover, expected};
  // a few waves share a leaf's items where they are many
  const int64_t gy = std::min<int64_t>(std::max<int64_t>((max_items + 255) / 256, 1), 64);
  k_shap_items<<<dim3((unsigned)(leaf1 - leaf0), (unsigned)gy), dim3(LGBM_WAVE), 0, s>>>(
      M, S, leaves, steps, plan, leaf0, X, rows, cols, tab);
  const int32_t rpb = shap_rows_per_block(nf, max_leaves);
  k_shap_rows<<<dim3((unsigned)((rows + rpb - 1) / rpb)), dim3(rpb * SHAP_LANES),
                shap_row_lds(nf, max_leaves) * (size_t)rpb, s>>>(
      M, S, leaves, steps, feats, plan, tab, X, rows, cols, nf, max_leaves, t0, t1, ntpi, first, out);
}

// Path elements and stack entries one thread needs for trees of depth at most `depth`.
int64_t shap_path_elems(int32_t depth) { return (int64_t)(depth + 1) * (depth + 2) / 2; }
int64_t shap_bytes_per_row(int32_t depth) {
  return shap_path_elems(depth) * (4 + 8 + 8 + 8) + (int64_t)(depth + 1) * (4 * 4 + 8);
}

// Runs TreeSHAP for rows [r0, r0 + n) with `ws` holding shap_bytes_per_row(depth) * n
// bytes (n a multiple of 256 or the tail of the rows).
void launch_contrib(const PredNode* nodes, const PredTree* trees, const double* leaves,
                    const int32_t* cat_bounds, const uint32_t* cat_words, const double* node_cover,
                    const double* leaf_cover, const double* expected, const float* X, int64_t r0,
                    int64_t n, int64_t rows, int32_t cols, int32_t nf, int32_t it0, int32_t it1,
                    int32_t ntpi, int32_t depth, void* ws, double* out, hipStream_t s,
                    const KernelEvents* ev) {
  if (n <= 0) return;
  const PredModelDev M{nodes, trees, leaves, cat_bounds, cat_words, nullptr, nullptr, nullptr};
  const ShapModelDev S{node_cover, leaf_cover, expected};
  const int64_t pe = shap_path_elems(depth), se = depth + 1;
  char* p = (char*)ws;
  ShapWork W;
  W.stride = n;
  W.pw = (double*)p;
  p += pe * n * 8;
  W.zero = (double*)p;
  p += pe * n * 8;
  W.one = (double*)p;
  p += pe * n * 8;
  W.s_zero = (double*)p;
  p += se * n * 8;
  W.feat = (int32_t*)p;
  p += pe * n * 4;
  W.s_node = (int32_t*)p;
  p += se * n * 4;
  W.s_base = (int32_t*)p;
  p += se * n * 4;
  W.s_depth = (int32_t*)p;
  p += se * n * 4;
  W.s_feat = (int32_t*)p;
  KLAUNCH(ev, k_contrib, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, M, S, W, X, r0, rows,
          cols, nf, it0, it1, ntpi, out);
}

// ---- sparse rows ------------------------------------------------------------------
// scatter_csr_row + validate_indptr_pair (predict.rs:772-870): one thread per row
// writes its entries in order into its zeroed dense row of `width` (=
// max_feature_idx + 1) floats (a repeated column keeps the last value; columns in
// [width, cols) are dropped).  A row whose indptr pair leaves [0, nnz] or runs backwards sets bit 0
// of *err, a column outside [0, cols) bit 1; the host refuses the call on either.
__global__ __launch_bounds__(256) void k_csr_dense(const int64_t* __restrict__ indptr,
                                                   const int32_t* __restrict__ indices,
                                                   const float* __restrict__ values, int64_t nnz,
                                                   int64_t rows, int32_t cols, int32_t width,
                                                   float* __restrict__ dense,
                                                   uint32_t* __restrict__ err) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  float* row = dense + r * width;
  const int64_t lo = indptr[r], hi = indptr[r + 1];
  if (lo < 0 || hi < lo || hi > nnz) {
    atomicOr(err, 1u);
    return;
  }
  for (int64_t k = lo; k < hi; ++k) {
    const int32_t c = indices[k];
    if (c < 0 || c >= cols) {
      atomicOr(err, 2u);
      return;
    }
    if (c < width) row[c] = values[k];
  }
}

// scatter_csc_dense (predict.rs:868-894) over the entries in parallel.  The dense
// rows are zeroed; a repeated row of a column keeps the column's last value; columns
// past `width` are only checked.  Bit 0 of *err: a column's indptr pair leaves
// [0, nnz] or runs backwards; bit 1: a row index outside [0, rows) (the host refuses
// the call on either, so the dense rows are then never read).
//   k_csc_check: one thread per column checks its indptr pair;
//   k_csc_claim: one thread per entry finds its column (the last c with indptr[c] <=
//     k; entries outside every column's range are skipped), checks its row and takes
//     its dense cell with a 32-bit atomic maximum of k + 1, so the last entry wins;
//     the claims live in the dense buffer itself (zeroed first);
//   k_csc_fill: one thread per cell replaces its claim by the claimed value (0: none).
__global__ __launch_bounds__(256) void k_csc_check(const int64_t* __restrict__ indptr,
                                                   int64_t nnz, int32_t cols,
                                                   uint32_t* __restrict__ err) {
  const int32_t c = (int32_t)(blockIdx.x * blockDim.x + threadIdx.x);
  if (c >= cols) return;
  const int64_t lo = indptr[c], hi = indptr[c + 1];
  if (lo < 0 || hi < lo || hi > nnz) atomicOr(err, 1u);
}
__global__ __launch_bounds__(256) void k_csc_claim(const int64_t* __restrict__ indptr,
                                                   const int32_t* __restrict__ indices,
                                                   int64_t nnz, int64_t rows, int32_t cols,
                                                   int32_t width, uint32_t* __restrict__ claim,
                                                   uint32_t* __restrict__ err) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  int32_t lo = 0, hi = cols + 1;  // first position in [0, cols] with indptr > k
  while (lo < hi) {
    const int32_t mid = lo + (hi - lo) / 2;
    if (indptr[mid] > k)
      hi = mid;
    else
      lo = mid + 1;
  }
  const int32_t c = lo - 1;
  if (c < 0 || c >= cols || k < indptr[c] || k >= indptr[c + 1]) return;
  const int32_t r = indices[k];
  if (r < 0 || (int64_t)r >= rows) {
    atomicOr(err, 2u);
    return;
  }
  if (c < width) atomicMax(&claim[(int64_t)r * width + c], (uint32_t)(k + 1));
}
__global__ __launch_bounds__(256) void k_csc_fill(const float* __restrict__ values, int64_t cells,
                                                  float* dense) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cells) return;
  const uint32_t u = ((const uint32_t*)dense)[i];
  dense[i] = u ? values[u - 1] : 0.0f;
}

void launch_csc_dense(const int64_t* indptr, const int32_t* indices, const float* values,
                      int64_t nnz, int64_t rows, int32_t cols, int32_t width, float* dense,
                      uint32_t* err, hipStream_t s) {
  if (cols <= 0) return;
  k_csc_check<<<dim3((unsigned)((cols + 255) / 256)), dim3(256), 0, s>>>(indptr, nnz, cols, err);
  if (nnz > 0)
    k_csc_claim<<<dim3((unsigned)((nnz + 255) / 256)), dim3(256), 0, s>>>(
        indptr, indices, nnz, rows, cols, width, (uint32_t*)dense, err);
  const int64_t cells = rows * (int64_t)width;
  if (cells > 0)
    k_csc_fill<<<dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, s>>>(values, cells, dense);
}

void launch_csr_dense(const int64_t* indptr, const int32_t* indices, const float* values,
                      int64_t nnz, int64_t rows, int32_t cols, int32_t width, float* dense,
                      uint32_t* err, hipStream_t s) {
  if (rows <= 0) return;
  k_csr_dense<<<dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, s>>>(
      indptr, indices, values, nnz, rows, cols, width, dense, err);
}

void launch_predict(const PredNode* nodes, const PredTree* trees, const double* leaves,
                    const int32_t* cat_bounds, const uint32_t* cat_words,
                    const PredLinLeaf* lin_leaves, const int32_t* lin_features,
                    const double* lin_coeffs, const float* X, int64_t rows, int32_t cols, int32_t it0, int32_t it1, int32_t ntpi, int32_t kind,
                    int32_t objective, double sigmoid, int32_t average_output, int32_t es_freq,
                    double es_margin, int32_t* es_iters, double* out, int32_t* leaf_out,
                    hipStream_t s, const KernelEvents* ev) {
  if (rows <= 0) return;
  const PredModelDev M{nodes,      trees,        leaves,    cat_bounds,
                       cat_words,  lin_leaves,   lin_features, lin_coeffs};
  const int64_t blocks = (rows + 255) / 256;
  if (cols <= PRED_STAGE_COLS)
    KLAUNCH(ev, k_predict<true>, dim3((unsigned)blocks), dim3(256),
            (size_t)256 * (cols | 1) * sizeof(float), s, M, X, rows, cols, it0, it1, ntpi, kind,
            objective, sigmoid, average_output, es_freq, es_margin, es_iters, out, leaf_out);
  else
    KLAUNCH(ev, k_predict<false>, dim3((unsigned)blocks), dim3(256), 0, s, M, X, rows, cols, it0,
            it1, ntpi, kind, objective, sigmoid, average_output, es_freq, es_margin, es_iters, out,
            leaf_out);
}

}  // namespace lgbm
