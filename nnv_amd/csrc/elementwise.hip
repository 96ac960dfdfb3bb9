// Affine layers that act row by row or through small fixed windows; all are single passes over
// the generator matrix (HBM bound):
//   * per-row affine programs: BatchNormalizationLayer (nn/layers/BatchNormalizationLayer.m:247-351),
//     ImageInputLayer normalisation (nn/layers/ImageInputLayer.m:121-166), ImageStar.affineMap
//     (set/ImageStar.m:431-460) -- the steps are applied in the reference's order so results
//     round the same way;
//   * AveragePooling2DLayer (nn/layers/AveragePooling2DLayer.m:229-247, 424-436; the arithmetic is
//     MatConvNet's vl_nnpool 'avg': mean over the part of the window inside the image);
//   * row permutations: the C-style FlattenLayer variants (nn/layers/FlattenLayer.m:118-170).
// Geometry of every kernel: a lane owns two adjacent rows, the eight waves of a block interleave
// columns; grid = (row blocks, column chunks, sets).
#include <algorithm>
#include <cmath>
#include <map>
#include <memory>
#include <vector>

#include "internal.h"
#include "relu_sort.h"

struct nnvhip_rowmap {
  nnvhip_ctx* ctx = nullptr;
  int64_t N = 0, ld = 0;
  int32_t n_steps = 0;
  int32_t op[8] = {0}, scope[8] = {0};
  bool keeps_zeros = true;   // the steps on all columns leave a zero generator entry zero (products and quotients by finite
                             // numbers, divisors not zero)
  bool may_flip = false;     // ... and some of them are negative
  nnvhip::BufRef params;  // ld x n_steps, zero padded rows
};

struct nnvhip_avgpool2d {
  nnvhip_ctx* ctx = nullptr;
  int64_t pool[2] = {1, 1}, stride[2] = {1, 1}, pad[4] = {0, 0, 0, 0};
};

namespace nnvhip {

constexpr int kEwWaves = 8;
constexpr int kEwRows = 128;  // rows per wave: 64 lanes x 2
constexpr int kMaxSteps = 8;

struct SetDesc {
  const double* in;
  double* out;
  int32_t ncols;
  int32_t pad_;
  // columns [box_from, box_to) are zero outside their windows box[j], whatever the memory holds there (images of HW positions, H a
  // column; permute_rows_lds_kernel only; null: none)
  const ColBox* box;
  int32_t box_from, box_to, H, HW;
};

struct RowmapArgs {
  const double* params;
  int64_t ld;      // leading dimension of in, out and params
  int32_t n_steps;
  int32_t cols_per_chunk;
  int32_t op[kMaxSteps];
  int32_t scope[kMaxSteps];
};

__device__ __forceinline__ double apply_op(int op, double v, double p) {
  switch (op) {
    case NNVHIP_OP_ADD: return __dadd_rn(v, p);
    case NNVHIP_OP_SUB: return __dsub_rn(v, p);
    case NNVHIP_OP_MUL: return __dmul_rn(v, p);
    default: return __ddiv_rn(v, p);
  }
}

__global__ __launch_bounds__(64 * kEwWaves) void rowmap_kernel(const SetDesc* __restrict__ table, SetDesc one,
                                                               RowmapArgs a) {
  const SetDesc d = table ? table[blockIdx.z] : one;
  const int j0 = blockIdx.y * a.cols_per_chunk;
  if (j0 >= d.ncols) return;
  const int j1 = min(d.ncols, j0 + a.cols_per_chunk);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t r0 = (int64_t)blockIdx.x * kEwRows + 2 * lane;
  if (r0 >= a.ld) return;
  double2 p[kMaxSteps];
#pragma unroll
  for (int s = 0; s < kMaxSteps; ++s)
    if (s < a.n_steps) p[s] = *reinterpret_cast<const double2*>(a.params + (int64_t)s * a.ld + r0);
  for (int jb = j0 + 4 * wave; jb < j1; jb += 4 * kEwWaves) {
    double2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (jb + u < j1) v[u] = *reinterpret_cast<const double2*>(d.in + r0 + (int64_t)(jb + u) * a.ld);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = jb + u;
      if (j >= j1) break;
      double2 x = v[u];
#pragma unroll
      for (int s = 0; s < kMaxSteps; ++s) {
        if (s >= a.n_steps) break;
        if (a.scope[s] == NNVHIP_SCOPE_ALL || j == 0) {
          x.x = apply_op(a.op[s], x.x, p[s].x);
          x.y = apply_op(a.op[s], x.y, p[s].y);
        }
      }
      *reinterpret_cast<double2*>(d.out + r0 + (int64_t)j * a.ld) = x;
    }
  }
}

// ---- generators that are known to be sparse --------------------------------------------------------------------
// The generator images behind a normalisation or an average pooling are as sparse as the ones in front of it: a row map
// scales them where they are, a pooling moves a window to the positions whose cells reach it.  The kernels below work
// inside the windows (nnvhip_star::box) and leave the zeros around them to a reader of whole columns (ColSource::win_*),
// as a convolution does.  A block takes a few columns and its threads their window places (position and channel), so a
// column costs eh * ew * C elements instead of the image; column 0, the centre, is a whole image and has the first blocks.
// What bounds them is the latency of scattered 16-40 byte pieces, not bytes.  A 32x32x3 CNN with
// normalisation and pooling (3073-3362 columns): batch normalisation 63 -> 9 us, row reset and pooling 48 + 51 -> 13 and
// 30 + 41 -> 22 us, and the convolutions in between stay inside windows too (162 -> 24, 83 -> 14 us).
struct WinSet {            // one set of a call (blockIdx.y)
  const double* in;
  double* out;
  const ColBox* box;       // windows of the output's columns
  int32_t eh, area;        // bound on a window: eh rows, area = eh * ew positions
  int32_t C, H, HW;        // channels; the input's image
  int32_t ncols;           // columns of the output
  int32_t cols_per_block;  // generator columns of a block
  // What a pooling reads besides whole columns: windows of the input's dense columns, the classes of a pending row reset
  // (rows other than kKeep read as zero), the list of unit-vector columns.
  int32_t dense;
  const ColBox* in_box;    // by input column, for 1 <= j < dense; or null (dense == 1)
  const int32_t* cls;      // or null
  const int32_t* idx;      // column dense + t is scale[idx[t]] (1 without scales) at row idx[t]
  const double* scale;
};
struct WinArgs {
  int64_t ldin, ldout;
  int32_t centre_blocks;   // the first blocks of a set do column 0, 256 rows each, the others a few generator columns each
};

__global__ __launch_bounds__(256) void rowmap_window_kernel(const WinSet* __restrict__ table, WinSet one, WinArgs g, RowmapArgs a) {
  const WinSet w = table ? table[blockIdx.y] : one;
  if ((int)blockIdx.x < g.centre_blocks) {
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= g.ldout) return;
    double x = w.in[r];
    for (int s = 0; s < a.n_steps; ++s) x = apply_op(a.op[s], x, a.params[(int64_t)s * a.ld + r]);
    w.out[r] = x;
    return;
  }
  const int j0 = 1 + ((int)blockIdx.x - g.centre_blocks) * w.cols_per_block;
  const int per = w.area * w.C, items = per * min(w.cols_per_block, w.ncols - j0);
  for (int f = threadIdx.x; f < items; f += 256) {
    const int jj = f / per, e = f - jj * per, j = j0 + jj;
    const int c = e / w.area, t = e - c * w.area;
    const int dw = t / w.eh, dh = t - dw * w.eh;
    const ColBox b = w.box[j];
    const int h = b.h0 + dh, x = b.w0 + dw;
    if (h > b.h1 || x > b.w1) continue;
    const int64_t r = (int64_t)c * w.HW + x * w.H + h;
    double v = w.in[r + (int64_t)j * g.ldin];
    for (int s = 0; s < a.n_steps; ++s)
      if (a.scope[s] == NNVHIP_SCOPE_ALL) v = apply_op(a.op[s], v, a.params[(int64_t)s * a.ld + r]);
    w.out[r + (int64_t)j * g.ldout] = v;
  }
}

// Centre and scales of boxes of which nothing else is in memory: blockIdx.y = vector (sets' centres, then scale vectors).
struct VecMap {
  const double* in;
  double* out;
  int32_t centre;  // 1: every step applies
};
__global__ __launch_bounds__(256) void rowmap_vectors_kernel(const VecMap* __restrict__ table, RowmapArgs a) {
  const VecMap d = table[blockIdx.y];
  const int64_t r = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (r >= a.ld) return;
  double x = d.in[r];
  for (int s = 0; s < a.n_steps; ++s)
    if (d.centre || a.scope[s] == NNVHIP_SCOPE_ALL) x = apply_op(a.op[s], x, a.params[(int64_t)s * a.ld + r]);
  d.out[r] = x;
}

struct PoolArgs {
  int64_t ldin, ldout;
  int32_t H, W, C, Ho, Wo;
  int32_t ph, pw, sh, sw, pt, pl;
  int32_t cols_per_chunk;
};

// One thread per output row (ho fastest, then wo, then channel); the waves of a block interleave
// columns.  Sum order: window columns outer, window rows inner, then one multiplication by
// 1 / (number of window cells inside the image).
__global__ __launch_bounds__(64 * kEwWaves) void avgpool_kernel(const SetDesc* __restrict__ table, SetDesc one,
                                                                PoolArgs a) {
  const SetDesc d = table ? table[blockIdx.z] : one;
  const int j0 = blockIdx.y * a.cols_per_chunk;
  if (j0 >= d.ncols) return;
  const int j1 = min(d.ncols, j0 + a.cols_per_chunk);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t r = (int64_t)blockIdx.x * 64 + lane;
  if (r >= a.ldout) return;
  const int64_t Nout = (int64_t)a.Ho * a.Wo * a.C;
  const bool real = r < Nout;
  int y1 = 0, y2 = 0, x1 = 0, x2 = 0;
  int64_t base = 0;
  double scale = 0.0;
  if (real) {
    const int ho = (int)(r % a.Ho);
    const int wo = (int)((r / a.Ho) % a.Wo);
    const int c = (int)(r / ((int64_t)a.Ho * a.Wo));
    y1 = ho * a.sh - a.pt;
    x1 = wo * a.sw - a.pl;
    y2 = min(y1 + a.ph, a.H);
    x2 = min(x1 + a.pw, a.W);
    y1 = max(y1, 0);
    x1 = max(x1, 0);
    base = (int64_t)c * a.H * a.W;
    scale = 1.0 / (double)((y2 - y1) * (x2 - x1));
  }
  // each wave takes 4 consecutive columns per step: four independent sums keep more loads in flight
  for (int jb = j0 + 4 * wave; jb < j1; jb += 4 * kEwWaves) {
    const int nu = min(4, j1 - jb);
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (real) {
      const double* col = d.in + (int64_t)jb * a.ldin + base;
      if (nu == 4) {
        for (int x = x1; x < x2; ++x)
          for (int y = y1; y < y2; ++y) {
            const double* p = col + y + (int64_t)x * a.H;
            const double v0 = p[0], v1 = p[a.ldin], v2 = p[2 * a.ldin], v3 = p[3 * a.ldin];
            acc[0] = __dadd_rn(acc[0], v0);
            acc[1] = __dadd_rn(acc[1], v1);
            acc[2] = __dadd_rn(acc[2], v2);
            acc[3] = __dadd_rn(acc[3], v3);
          }
      } else {
        for (int u = 0; u < nu; ++u)
          for (int x = x1; x < x2; ++x)
            for (int y = y1; y < y2; ++y) acc[u] = __dadd_rn(acc[u], col[y + (int64_t)x * a.H + (int64_t)u * a.ldin]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] = __dmul_rn(acc[u], scale);
    }
    for (int u = 0; u < nu; ++u) d.out[r + (int64_t)(jb + u) * a.ldout] = acc[u];  // padding rows stay zero
  }
}

// The cells of a window of up to kPoolAhead rows are asked for together, kPoolAhead columns at a time: one after the other, with
// the row's class in front of each, a 3 x 3 pooling of 3360 images of 16 x 16 x 16 took 23.3 us, now 16.9.
constexpr int kPoolAhead = 3;
// Sums run as in avgpool_kernel (window columns outer, rows inner); what lies outside an input window adds an exact zero
// and is left out.
__global__ __launch_bounds__(256) void avgpool_window_kernel(const WinSet* __restrict__ table, WinSet one, WinArgs g, PoolArgs a) {
  const WinSet w = table ? table[blockIdx.y] : one;
  const int HW = a.H * a.W, P = a.Ho * a.Wo;
  auto cell = [&](int ho, int wo, int& y1, int& y2, int& x1, int& x2) {
    y1 = ho * a.sh - a.pt;
    x1 = wo * a.sw - a.pl;
    y2 = min(y1 + a.ph, a.H);
    x2 = min(x1 + a.pw, a.W);
    y1 = max(y1, 0);
    x1 = max(x1, 0);
    return 1.0 / (double)((y2 - y1) * (x2 - x1));
  };
  if ((int)blockIdx.x < g.centre_blocks) {
    const int r = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (r >= P * w.C) return;
    const int c = r / P, p = r - c * P, wo = p / a.Ho, ho = p - wo * a.Ho;
    int y1, y2, x1, x2;
    const double scale = cell(ho, wo, y1, y2, x1, x2);
    double acc = 0.0;
    for (int x = x1; x < x2; ++x)
      for (int y = y1; y < y2; ++y) {
        const int64_t q = (int64_t)c * HW + x * a.H + y;
        acc = __dadd_rn(acc, w.cls == nullptr || w.cls[q] == kKeep ? w.in[q] : 0.0);
      }
    w.out[r] = __dmul_rn(acc, scale);
    return;
  }
  const int j0 = 1 + ((int)blockIdx.x - g.centre_blocks) * w.cols_per_block;
  const int per = w.area * w.C, items = per * min(w.cols_per_block, w.ncols - j0);
  for (int f = threadIdx.x; f < items; f += 256) {
    const int jj = f / per, e = f - jj * per, j = j0 + jj;
    const int c = e / w.area, t = e - c * w.area;
    const int dw = t / w.eh, dh = t - dw * w.eh;
    const ColBox b = w.box[j];
    const int ho = b.h0 + dh, wo = b.w0 + dw;
    if (ho > b.h1 || wo > b.w1) continue;
    int y1, y2, x1, x2;
    const double scale = cell(ho, wo, y1, y2, x1, x2);
    double acc = 0.0;
    if (j < w.dense) {
      const ColBox q = w.in_box[j];
      const double* col = w.in + (int64_t)j * g.ldin + (int64_t)c * HW;
      const int xa = max(x1, (int)q.w0), xb = min(x2, q.w1 + 1), ya = max(y1, (int)q.h0), yb = min(y2, q.h1 + 1);
      if (a.ph <= kPoolAhead) {
        // kPoolAhead window columns at a time, all their cells asked for together (one behind the window: its last again)
        for (int x = xa; x < xb && ya < yb; x += kPoolAhead) {
          double v[kPoolAhead][kPoolAhead];
          int cl[kPoolAhead][kPoolAhead];
#pragma unroll
          for (int u = 0; u < kPoolAhead; ++u)
#pragma unroll
            for (int t = 0; t < kPoolAhead; ++t) {
              const int at = min(x + u, xb - 1) * a.H + min(ya + t, yb - 1);
              v[u][t] = col[at];
              cl[u][t] = w.cls != nullptr ? w.cls[(int64_t)c * HW + at] : kKeep;
            }
#pragma unroll
          for (int u = 0; u < kPoolAhead; ++u)
#pragma unroll
            for (int t = 0; t < kPoolAhead; ++t)
              if (x + u < xb && ya + t < yb) acc = __dadd_rn(acc, cl[u][t] == kKeep ? v[u][t] : 0.0);
        }
      } else {
        for (int x = xa; x < xb; ++x)
          for (int y = ya; y < yb; ++y)
            acc = __dadd_rn(acc, w.cls == nullptr || w.cls[(int64_t)c * HW + x * a.H + y] == kKeep ? col[x * a.H + y] : 0.0);
      }
    } else {
      const int src = w.idx[j - w.dense];
      const int sc = src / HW, sp = src - sc * HW, sx = sp / a.H, sy = sp - sx * a.H;
      if (sc == c && sx >= x1 && sx < x2 && sy >= y1 && sy < y2) acc = w.scale != nullptr ? w.scale[src] : 1.0;
    }
    w.out[(int64_t)c * P + wo * a.Ho + ho + (int64_t)j * g.ldout] = __dmul_rn(acc, scale);
  }
}

struct PermArgs {
  const int32_t* src_row;  // ldout entries; -1 = padding row (written as zero)
  int64_t ldin, ldout;
  int32_t cols_per_chunk;
};

__global__ __launch_bounds__(64 * kEwWaves) void permute_rows_kernel(const SetDesc* __restrict__ table, SetDesc one,
                                                                     PermArgs a) {
  const SetDesc d = table ? table[blockIdx.z] : one;
  const int j0 = blockIdx.y * a.cols_per_chunk;
  if (j0 >= d.ncols) return;
  const int j1 = min(d.ncols, j0 + a.cols_per_chunk);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t r0 = (int64_t)blockIdx.x * kEwRows + 2 * lane;
  if (r0 >= a.ldout) return;
  const int2 src = *reinterpret_cast<const int2*>(a.src_row + r0);
  for (int jb = j0 + 4 * wave; jb < j1; jb += 4 * kEwWaves) {
    double2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      v[u] = make_double2(0.0, 0.0);
      if (jb + u < j1) {
        const double* col = d.in + (int64_t)(jb + u) * a.ldin;
        if (src.x >= 0) v[u].x = col[src.x];
        if (src.y >= 0) v[u].y = col[src.y];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (jb + u < j1) *reinterpret_cast<double2*>(d.out + r0 + (int64_t)(jb + u) * a.ldout) = v[u];
  }
}

// Short columns (N <= kPermLdsRows): a block stages whole columns in LDS with coalesced loads and
// gathers from there, so global memory sees only contiguous traffic.  Images that are in memory inside their windows only
// (SetDesc::box) are read there and zero elsewhere: 3400 images of 8 x 8 x 16 10.4 us of zeros written + 13.7 -> 15.8.
// Grid: (1, column chunks, sets).
constexpr int kPermLdsRows = 4096;
__host__ __device__ constexpr int perm_stride(int n_rows) { return n_rows + n_rows / 32 + 1; }
// columns staged per step: four where four blocks of them fit a CU, two within 64 KB
constexpr int perm_columns(int n_rows) { return n_rows <= 1024 ? 4 : n_rows <= 3968 ? 2 : 1; }

__global__ __launch_bounds__(64 * kEwWaves) void permute_rows_lds_kernel(const SetDesc* __restrict__ table, SetDesc one,
                                                                         PermArgs a, int n_rows, int step) {
  const SetDesc d = table ? table[blockIdx.z] : one;
  const int j0 = blockIdx.y * a.cols_per_chunk;
  if (j0 >= d.ncols) return;
  const int j1 = min(d.ncols, j0 + a.cols_per_chunk);
  // (a place left free behind every 32: the rows that neighbouring outputs come from are often a multiple of 32 apart, 64 lanes on
  // one bank)
  extern __shared__ double stage[];
  const int stride = perm_stride(n_rows);
  const int tid = threadIdx.x;
  for (int jb = j0; jb < j1; jb += step) {
    const int nc = min(step, j1 - jb);
    // a row's place in the image serves all columns; four columns' entries are asked for together
    for (int r = tid; r < n_rows; r += 64 * kEwWaves) {
      int h = 0, w = 0;
      if (d.box != nullptr) {
        const int p = r % d.HW;
        w = p / d.H, h = p - w * d.H;
      }
      for (int u0 = 0; u0 < nc; u0 += 4) {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int j = jb + u0 + u;
          bool in = u0 + u < nc;
          if (in && d.box != nullptr && j >= d.box_from && j < d.box_to) {
            const ColBox b = d.box[j];
            in = h >= b.h0 && h <= b.h1 && w >= b.w0 && w <= b.w1;
          }
          v[u] = in ? d.in[r + (int64_t)j * a.ldin] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (u0 + u < nc) stage[(u0 + u) * stride + r + r / 32] = v[u];
      }
    }
    __syncthreads();
    for (int64_t r = tid; r < a.ldout; r += 64 * kEwWaves) {
      const int src = a.src_row[r];
      const double* from = stage + max(src, 0) + max(src, 0) / 32;
      for (int u = 0; u < nc; ++u) d.out[r + (int64_t)(jb + u) * a.ldout] = src >= 0 ? from[u * stride] : 0.0;
    }
    __syncthreads();
  }
}

// Common launch plumbing: output handles, descriptor table, grid with a few thousand blocks.
template <class Launch>
static int run_row_layer(nnvhip_ctx* c, int64_t count, nnvhip_star* const* in, nnvhip_star** out, int64_t Nout,
                         int64_t rows_per_block, int min_cols_per_chunk, Launch launch, bool reads_windows = false) {
  if (count > 65535) NNV_FAIL(NNVHIP_ERR_SHAPE, "at most 65535 sets per call");
  for (int64_t i = 0; i < count; ++i) {
    if (in[i]->N != in[0]->N || in[i]->ld != in[0]->ld)
      NNV_FAIL(NNVHIP_ERR_SHAPE, "sets of one array must have the same dimension");
  }
  // These passes read every column.  (reads_windows: the launch knows how to read a set of which nothing is missing but the zeros
  // around its images' windows.)
  auto only_zeros_missing = [&](const nnvhip_star* s) {
    return reads_windows && s->cs.win_pending() && !s->cs.in_pixels() && !s->rows_pending && s->stored_cols() == s->n + 1 && !s->cs.pending &&
           s->cs.zero_to <= 1 && !s->cs.delta_pending() && s->cs.win_rows == s->N;
  };
  std::vector<nnvhip_star*> whole;
  for (int64_t i = 0; i < count; ++i)
    if (!only_zeros_missing(in[i])) whole.push_back(in[i]);
  if (!whole.empty()) NNV_TRY(ensure_dense_batch(c, (int64_t)whole.size(), whole.data()));
  std::vector<nnvhip_star*> outs;
  bool contig = false;
  int64_t cols = 0;
  NNV_TRY(c->begin_op());
  int st = make_affine_outputs(c, count, in, Nout, &outs, &contig, &cols);
  if (st == NNVHIP_OK) {
    std::vector<SetDesc> descs((size_t)count);
    int64_t max_cols = 0;
    for (int64_t i = 0; i < count; ++i) {
      descs[i].in = in[i]->V;
      descs[i].out = outs[i]->V;
      descs[i].ncols = (int32_t)(in[i]->n + 1);
      descs[i].pad_ = 0;
      descs[i].box = nullptr;
      if (only_zeros_missing(in[i])) {
        const ColSource& cs = in[i]->cs;
        descs[i].box = cs.win_box;
        descs[i].box_from = (int32_t)cs.win_from;
        descs[i].box_to = (int32_t)cs.win_to;
        descs[i].H = cs.win_H;
        descs[i].HW = cs.win_H * cs.win_W;
        ++c->routes[NNVHIP_ROUTE_PERMUTE_WINDOW];
      }
      max_cols = std::max<int64_t>(max_cols, in[i]->n + 1);
    }
    const SetDesc* table = nullptr;
    BufRef tab;
    if (count > 1) {
      st = c->upload_table(descs.data(), sizeof(SetDesc) * descs.size(), &tab);
      if (st == NNVHIP_OK) table = tab->as<SetDesc>();
    }
    if (st == NNVHIP_OK) {
      const int64_t ldout = outs[0]->ld;
      const int64_t row_blocks = ceil_div(ldout, rows_per_block);
      int64_t chunks = std::max<int64_t>(1, std::min<int64_t>(ceil_div(8192, row_blocks * count),
                                                               ceil_div(max_cols, min_cols_per_chunk)));
      const int64_t cpc = ceil_div(max_cols, chunks);
      chunks = ceil_div(max_cols, cpc);
      double bytes = 0.0;  // algorithmic: every input element read once, every output element written once
      for (int64_t i = 0; i < count; ++i) bytes += 8.0 * (double)(in[i]->N + Nout) * (double)(in[i]->n + 1);
      st = c->kernel_timer_begin(c->kernel_timing);
      launch(dim3((unsigned)row_blocks, (unsigned)chunks, (unsigned)count), table, descs[0], (int32_t)cpc, outs[0]->ld);
      if (st == NNVHIP_OK) st = c->kernel_timer_end(c->kernel_timing, 4, bytes);
      if (hipGetLastError() != hipSuccess) {
        set_error("kernel launch failed");
        st = NNVHIP_ERR_HIP;
      }
    }
  }
  if (st == NNVHIP_OK) st = c->end_op();
  if (st != NNVHIP_OK) {
    release_all(outs);
    return st;
  }
  for (int64_t i = 0; i < count; ++i) out[i] = outs[i];
  return NNVHIP_OK;
}

// Marks the generator columns of a call's outputs as written inside their windows only; the padding rows are zeroed (the
// outputs lie back to back: one launch).
static int leave_outside_windows(nnvhip_ctx* c, const std::vector<nnvhip_star*>& outs, int64_t total_cols) {
  for (auto* o : outs) {
    o->cs.win_box_buf = o->box_buf;
    o->cs.win_box = o->box;
    o->cs.win_from = 1;
    o->cs.win_to = o->n + 1;
    o->cs.win_rows = o->N;
    o->cs.win_H = o->box_H;
    o->cs.win_W = o->box_W;
    if (c->poison_pending)  // debugging aid: NaNs where nothing will be written
      NNV_HIP_TRY(hipMemsetAsync(o->V + o->ld, 0xff, sizeof(double) * o->ld * o->n, c->stream));
  }
  return launch_zero_pad_rows(c, outs[0]->V, outs[0]->ld, outs[0]->N, total_cols);
}

// The sets of a call (all but the pooling's own fields), its arguments and its grid.
struct WinCall {
  std::vector<WinSet> sets;
  WinArgs g{};
  dim3 grid;
  double places = 0.0;  // window places of all generator columns
  const WinSet* table = nullptr;
  BufRef tab;
};
static WinCall win_call(int64_t count, nnvhip_star* const* in, const std::vector<nnvhip_star*>& outs, int64_t HW) {
  WinCall w;
  w.g.ldin = in[0]->ld;
  w.g.ldout = outs[0]->ld;
  w.g.centre_blocks = (int32_t)ceil_div(outs[0]->ld, 256);
  int64_t column_blocks = 0;
  w.sets.resize((size_t)count);
  for (int64_t i = 0; i < count; ++i) {
    const nnvhip_star* o = outs[(size_t)i];
    WinSet& s = w.sets[(size_t)i];
    s = WinSet{};
    s.in = in[i]->V;
    s.out = o->V;
    s.box = o->box;
    s.eh = o->box_eh;
    s.area = o->box_eh * o->box_ew;
    s.H = o->box_H;
    s.HW = (int32_t)(HW > 0 ? HW : (int64_t)o->box_H * o->box_W);
    s.C = (int32_t)(in[i]->N / s.HW);
    s.ncols = (int32_t)(o->n + 1);
    // a block: the columns that make two to four elements a thread, one column at least
    s.cols_per_block = (int32_t)std::max<int64_t>(1, 1024 / std::max<int64_t>(1, (int64_t)s.area * s.C));
    column_blocks = std::max<int64_t>(column_blocks, ceil_div(o->n, s.cols_per_block));
    w.places += (double)s.area * s.C * (double)o->n;
  }
  w.grid = dim3((unsigned)(w.g.centre_blocks + column_blocks), (unsigned)count);
  return w;
}
static int upload_sets(nnvhip_ctx* c, WinCall* w) {
  if (w->sets.size() < 2) return NNVHIP_OK;
  NNV_TRY(c->upload_table(w->sets.data(), sizeof(WinSet) * w->sets.size(), &w->tab));
  w->table = w->tab->as<WinSet>();
  return NNVHIP_OK;
}

static bool small_windows(int64_t eh, int64_t ew, int64_t P) { return eh > 0 && ew > 0 && 2 * eh * ew <= P; }
static bool windows_allowed(const nnvhip_ctx* c) { return !c->eager_cols && !c->dense_affine && !c->no_conv_boxes; }

// Row map of an image set whose generator images are zero outside small windows, every column of which is in memory there.
static bool rowmap_in_windows(const nnvhip_ctx* c, const nnvhip_rowmap* m, const nnvhip_star* s) {
  if (!windows_allowed(c) || !m->keeps_zeros || s->rows_pending || s->stored_cols() != s->n + 1 || s->n < 1) return false;
  if (s->box == nullptr || s->box_cols < s->n + 1 || s->box_H <= 0 || s->box_W <= 0) return false;
  const int64_t P = (int64_t)s->box_H * s->box_W;
  return s->N % P == 0 && small_windows(s->box_eh, s->box_ew, P) && !s->cs.pending && s->cs.zero_to <= 1 && !s->cs.delta_pending() &&
         !s->cs.in_pixels() && s->n < 1000000;
}

// One launch for all sets of a call, here and in pool_windows.  (With a launch or three per image, 100 images of 12 x 12
// through two poolings, a batch normalisation, a convolution and two FC layers took 5.9 ms a pass, 4.7 ms over whole columns;
// now 2.7 ms.  64 images of 28 x 28: 4.2, 4.3 and 1.8 ms.)
static int rowmap_windows(nnvhip_ctx* c, const RowmapArgs& a, int64_t N, int64_t count, nnvhip_star* const* in, nnvhip_star** out) {
  if (count > 65535) NNV_FAIL(NNVHIP_ERR_SHAPE, "at most 65535 sets per call");
  std::vector<nnvhip_star*> outs;
  bool contig = false;
  int64_t cols = 0;
  NNV_TRY(c->begin_op());
  int st = make_affine_outputs(c, count, in, N, &outs, &contig, &cols);
  if (st == NNVHIP_OK) {
    for (int64_t i = 0; i < count; ++i) {
      nnvhip_star* o = outs[(size_t)i];
      o->box_buf = in[i]->box_buf;
      o->box = in[i]->box;
      o->box_cols = in[i]->box_cols;
      o->box_H = in[i]->box_H;
      o->box_W = in[i]->box_W;
      o->box_eh = in[i]->box_eh;
      o->box_ew = in[i]->box_ew;
    }
    st = leave_outside_windows(c, outs, cols);
  }
  if (st == NNVHIP_OK) {
    WinCall w = win_call(count, in, outs, 0);
    st = upload_sets(c, &w);
    if (st == NNVHIP_OK) {
      NNV_LAUNCH(c, c->kernel_timing, rowmap_window_kernel, w.grid, dim3(256), 0, w.table, w.sets[0], w.g, a);
      st = c->kernel_timer_end(c->kernel_timing, 4, 16.0 * (w.places + (double)N * (double)count));
    }
    if (st == NNVHIP_OK && hipGetLastError() != hipSuccess) {
      set_error("kernel launch failed");
      st = NNVHIP_ERR_HIP;
    }
  }
  if (st == NNVHIP_OK) st = c->end_op();
  if (st != NNVHIP_OK) {
    release_all(outs);
    return st;
  }
  c->routes[NNVHIP_ROUTE_ROWMAP_WINDOW] += count;
  for (int64_t i = 0; i < count; ++i) out[i] = outs[(size_t)i];
  return NNVHIP_OK;
}

// Row map of boxes of which only the centres are in memory: the same boxes with mapped centres and scales (a scale vector
// shared by several sets is mapped once and stays shared).
static int rowmap_boxes(nnvhip_ctx* c, const RowmapArgs& a, bool may_flip, int64_t N, int64_t count, nnvhip_star* const* in,
                        nnvhip_star** out) {
  const int64_t ld = a.ld;
  double whole = 0.0;  // (mapped boxes whose matrices no reader could be given are refused here, as where they are made)
  for (int64_t i = 0; i < count; ++i) whole += 8.0 * (double)ld * (double)(in[i]->n + 1);
  NNV_TRY(c->check_room((size_t)whole));
  NNV_TRY(c->begin_op());
  std::map<const double*, int64_t> scale_at;
  for (int64_t i = 0; i < count; ++i) scale_at.emplace(in[i]->oh_scale, (int64_t)scale_at.size());
  BufRef buf, tab;
  NNV_TRY(c->alloc(sizeof(double) * ld * (count + (int64_t)scale_at.size()), &buf));
  std::vector<VecMap> vm((size_t)(count + (int64_t)scale_at.size()));
  for (int64_t i = 0; i < count; ++i) vm[(size_t)i] = VecMap{in[i]->V, buf->as<double>() + i * ld, 1};
  for (const auto& sc : scale_at) vm[(size_t)(count + sc.second)] = VecMap{sc.first, buf->as<double>() + (count + sc.second) * ld, 0};
  NNV_TRY(c->upload_table(vm.data(), sizeof(VecMap) * vm.size(), &tab));
  for (size_t v0 = 0; v0 < vm.size(); v0 += 65535) {
    const unsigned cnt = (unsigned)std::min<size_t>(65535, vm.size() - v0);
    NNV_LAUNCH(c, c->kernel_timing, rowmap_vectors_kernel, dim3((unsigned)ceil_div(ld, 256), cnt), dim3(256), 0, tab->as<VecMap>() + v0, a);
    NNV_TRY(c->kernel_timer_end(c->kernel_timing, 4, 16.0 * (double)ld * cnt));
  }
  NNV_HIP_TRY(hipGetLastError());
  c->routes[NNVHIP_ROUTE_ROWMAP_BOX] += count;
  for (int64_t i = 0; i < count; ++i) {
    nnvhip_star* o = new_star(c);
    o->N = N;
    o->n = in[i]->n;
    o->ld = ld;
    o->Vbuf = buf;
    o->V = vm[(size_t)i].out;
    o->vcols = 1;
    o->pbuf = in[i]->pbuf;
    o->plb = in[i]->plb;
    o->pub = in[i]->pub;
    o->ptails = in[i]->ptails;
    o->pslot = in[i]->pslot;
    o->pcap = in[i]->pcap;
    o->cons = in[i]->cons;
    o->oh_from = 1;
    o->oh_idx_buf = in[i]->oh_idx_buf;
    o->oh_idx = in[i]->oh_idx;
    o->oh_scale_buf = buf;
    o->oh_scale = vm[(size_t)(count + scale_at[in[i]->oh_scale])].out;
    o->oh_scale_neg = in[i]->oh_scale_neg || may_flip;
    o->oh_inv_buf = in[i]->oh_inv_buf;
    o->oh_inv = in[i]->oh_inv;
    out[i] = o;
  }
  return c->end_op();
}

// Average pooling inside windows: the input's dense images have small windows (or there is nothing dense but the centre),
// its other columns are unit vectors by list, and the output's windows are small.
struct PoolPlan {
  int64_t dense = 0, m = 0, eh = 0, ew = 0;
};
static bool pool_in_windows(const nnvhip_ctx* c, const nnvhip_avgpool2d* p, const nnvhip_star* s, int64_t H, int64_t W, int64_t Ho, int64_t Wo,
                            PoolPlan* pl) {
  if (!windows_allowed(c) || s->n < 1 || H >= 32768 || W >= 32768) return false;
  const int64_t nc = s->n + 1;
  pl->dense = (s->oh_from > 0 && s->oh_from < nc) ? s->oh_from : nc;
  pl->m = nc - pl->dense;
  if (pl->dense > s->stored_cols() || (pl->m > 0 && s->oh_idx == nullptr)) return false;
  if (s->cs.pending || s->cs.zero_to > 1 || s->cs.delta_pending() || s->cs.in_pixels() || (s->rows_pending && s->cls == nullptr)) return false;
  if (pl->dense > 1 && !(s->box != nullptr && s->box_H == H && s->box_W == W && s->box_cols >= pl->dense)) return false;
  auto extent = [&](int d, int64_t e, int64_t size) { return std::min<int64_t>(size, (e - 1 + p->pool[d] - 1) / p->stride[d] + 1); };
  pl->eh = pl->ew = 0;
  if (pl->dense > 1) {
    pl->eh = extent(0, s->box_eh, Ho);
    pl->ew = extent(1, s->box_ew, Wo);
  }
  if (pl->m > 0) {
    pl->eh = std::max(pl->eh, extent(0, 1, Ho));
    pl->ew = std::max(pl->ew, extent(1, 1, Wo));
  }
  return small_windows(pl->eh, pl->ew, Ho * Wo) && s->n < 1000000;
}

static int pool_windows(nnvhip_ctx* c, const nnvhip_avgpool2d* p, PoolArgs a, int64_t count, nnvhip_star* const* in, const PoolPlan* plans,
                        nnvhip_star** out) {
  if (count > 65535) NNV_FAIL(NNVHIP_ERR_SHAPE, "at most 65535 sets per call");
  const int64_t Nout = (int64_t)a.Ho * a.Wo * a.C;
  std::vector<nnvhip_star*> outs;
  bool contig = false;
  int64_t cols = 0;
  NNV_TRY(c->begin_op());
  int st = make_affine_outputs(c, count, in, Nout, &outs, &contig, &cols);
  BufRef boxes;
  if (st == NNVHIP_OK) st = c->alloc(sizeof(ColBox) * (size_t)cols, &boxes);
  if (st == NNVHIP_OK) {
    std::vector<ConvSetup> setup((size_t)count);
    ColBox* at = boxes->as<ColBox>();
    for (int64_t i = 0; i < count; ++i) {
      nnvhip_star* o = outs[(size_t)i];
      const PoolPlan& pl = plans[i];
      setup[(size_t)i] = ConvSetup{pl.dense > 1 ? in[i]->box : nullptr, in[i]->oh_idx, at, nullptr, (int32_t)pl.dense, (int32_t)pl.m, 0, nullptr, nullptr};
      o->box_buf = boxes;
      o->box = at;
      o->box_cols = o->n + 1;
      o->box_H = a.Ho;
      o->box_W = a.Wo;
      o->box_eh = (int32_t)pl.eh;
      o->box_ew = (int32_t)pl.ew;
      at += o->n + 1;
    }
    st = launch_pool_setup(c, a.H, a.W, a.Ho, a.Wo, p->pool, p->stride, p->pad[0], p->pad[2], count, setup.data());
  }
  if (st == NNVHIP_OK) st = leave_outside_windows(c, outs, cols);
  if (st == NNVHIP_OK) {
    WinCall w = win_call(count, in, outs, (int64_t)a.H * a.W);
    for (int64_t i = 0; i < count; ++i) {
      WinSet& s = w.sets[(size_t)i];
      s.H = a.H;
      s.in_box = plans[i].dense > 1 ? in[i]->box : nullptr;
      s.cls = in[i]->rows_pending ? in[i]->cls : nullptr;
      s.idx = in[i]->oh_idx;
      s.scale = in[i]->oh_scale;
      s.dense = (int32_t)plans[i].dense;
    }
    st = upload_sets(c, &w);
    if (st == NNVHIP_OK) {
      NNV_LAUNCH(c, c->kernel_timing, avgpool_window_kernel, w.grid, dim3(256), 0, w.table, w.sets[0], w.g, a);
      st = c->kernel_timer_end(c->kernel_timing, 4, 8.0 * (w.places * 2.0 + (double)(in[0]->N + Nout) * (double)count));
    }
    if (st == NNVHIP_OK && hipGetLastError() != hipSuccess) {
      set_error("kernel launch failed");
      st = NNVHIP_ERR_HIP;
    }
  }
  if (st == NNVHIP_OK) st = c->end_op();
  if (st != NNVHIP_OK) {
    release_all(outs);
    return st;
  }
  c->routes[NNVHIP_ROUTE_POOL_WINDOW] += count;
  for (int64_t i = 0; i < count; ++i) out[i] = outs[(size_t)i];
  return NNVHIP_OK;
}

}  // namespace nnvhip

using namespace nnvhip;

extern "C" {

int nnvhip_rowmap_create(nnvhip_ctx* c, int64_t N, int32_t n_steps, const int32_t* op, const int32_t* scope,
                         const double* params, nnvhip_rowmap** out) {
  if (!c) NNV_FAIL(NNVHIP_ERR_ARG, "null context");
  NNV_TRY(nnvhip::enter_ctx(c));
  if (!op || !scope || !params || !out) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  if (N <= 0 || n_steps <= 0 || n_steps > kMaxSteps) NNV_FAIL(NNVHIP_ERR_SHAPE, "a row map has 1 to 8 steps");
  std::unique_ptr<nnvhip_rowmap> m(new nnvhip_rowmap());
  m->ctx = c;
  m->N = N;
  m->ld = round_up(N, kLdAlign);
  m->n_steps = n_steps;
  for (int s = 0; s < n_steps; ++s) {
    if (op[s] < NNVHIP_OP_ADD || op[s] > NNVHIP_OP_DIV || (scope[s] != NNVHIP_SCOPE_CENTRE && scope[s] != NNVHIP_SCOPE_ALL))
      NNV_FAIL(NNVHIP_ERR_ARG, "invalid step %d", s);
    m->op[s] = op[s];
    m->scope[s] = scope[s];
  }
  for (int s = 0; s < n_steps; ++s) {
    if (m->scope[s] != NNVHIP_SCOPE_ALL) continue;
    if (m->op[s] != NNVHIP_OP_MUL && m->op[s] != NNVHIP_OP_DIV) m->keeps_zeros = false;
    for (int64_t r = 0; r < N; ++r) {
      const double v = params[s * N + r];
      if (!std::isfinite(v) || (m->op[s] == NNVHIP_OP_DIV && v == 0.0)) m->keeps_zeros = false;
      if (std::signbit(v)) m->may_flip = true;
    }
  }
  // padding rows get the neutral operand of their step so that they stay exactly zero
  std::vector<double> host((size_t)(m->ld * n_steps));
  for (int s = 0; s < n_steps; ++s) {
    const double neutral = (op[s] == NNVHIP_OP_MUL || op[s] == NNVHIP_OP_DIV) ? 1.0 : 0.0;
    for (int64_t r = 0; r < m->ld; ++r) host[(size_t)(s * m->ld + r)] = r < N ? params[s * N + r] : neutral;
  }
  NNV_TRY(c->alloc(sizeof(double) * host.size(), &m->params));
  NNV_HIP_TRY(hipMemcpyAsync(m->params->ptr, host.data(), sizeof(double) * host.size(), hipMemcpyHostToDevice, c->stream));
  c->h2d_bytes += (int64_t)(sizeof(double) * host.size());
  NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  *out = m.release();
  return NNVHIP_OK;
}

int nnvhip_rowmap_destroy(nnvhip_rowmap* m) {
  delete m;
  return NNVHIP_OK;
}

int nnvhip_affine_rowmap(nnvhip_ctx* c, const nnvhip_rowmap* m, int64_t count, nnvhip_star* const* in,
                         nnvhip_star** out) {
  if (!c) NNV_FAIL(NNVHIP_ERR_ARG, "null context");
  NNV_TRY(nnvhip::enter_ctx(c));
  if (!m || m->ctx != c) NNV_FAIL(NNVHIP_ERR_ARG, "invalid layer handle");
  NNV_TRY(check_set_array(c, count, in, out));
  for (int64_t i = 0; i < count; ++i)
    if (in[i]->N != m->N)
      NNV_FAIL(NNVHIP_ERR_SHAPE, "Inconsistent number of channels between scale array and the ImageStar");
  RowmapArgs a{};
  a.params = m->params->as<double>();
  a.ld = m->ld;
  a.n_steps = m->n_steps;
  for (int s = 0; s < kMaxSteps; ++s) {
    a.op[s] = m->op[s];
    a.scope[s] = m->scope[s];
  }
  {
    bool windows = true, boxes = m->keeps_zeros && windows_allowed(c);
    for (int64_t i = 0; i < count; ++i) {
      windows = windows && in[i]->ld == in[0]->ld && rowmap_in_windows(c, m, in[i]);
      boxes = boxes && is_unwritten_box(in[i]) && in[i]->ld == m->ld;
    }
    if (windows) return rowmap_windows(c, a, m->N, count, in, out);
    if (boxes) return rowmap_boxes(c, a, m->may_flip, m->N, count, in, out);
  }
  return run_row_layer(c, count, in, out, m->N, kEwRows, 4 * kEwWaves,
                       [&](dim3 grid, const SetDesc* table, const SetDesc& one, int32_t cpc, int64_t) {
                         a.cols_per_chunk = cpc;
                         NNV_LAUNCH(c, c->kernel_timing, rowmap_kernel, grid, dim3(64 * kEwWaves), 0, table, one, a);
                       });
}

int nnvhip_avgpool2d_create(nnvhip_ctx* c, const int64_t pool[2], const int64_t stride[2], const int64_t padding[4],
                            nnvhip_avgpool2d** out) {
  if (!c) NNV_FAIL(NNVHIP_ERR_ARG, "null context");
  if (!pool || !stride || !padding || !out) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  if (pool[0] < 1 || pool[1] < 1) NNV_FAIL(NNVHIP_ERR_SHAPE, "Invalid pool size");
  if (stride[0] < 1 || stride[1] < 1) NNV_FAIL(NNVHIP_ERR_SHAPE, "Invalid stride");
  for (int i = 0; i < 4; ++i)
    if (padding[i] < 0) NNV_FAIL(NNVHIP_ERR_SHAPE, "Invalide padding size");
  // a window that lies entirely in the padding would have no cell to average
  if (padding[0] >= pool[0] || padding[1] >= pool[0] || padding[2] >= pool[1] || padding[3] >= pool[1])
    NNV_FAIL(NNVHIP_ERR_SHAPE, "Invalide padding size");
  nnvhip_avgpool2d* p = new nnvhip_avgpool2d();
  p->ctx = c;
  for (int i = 0; i < 2; ++i) {
    p->pool[i] = pool[i];
    p->stride[i] = stride[i];
  }
  for (int i = 0; i < 4; ++i) p->pad[i] = padding[i];
  *out = p;
  return NNVHIP_OK;
}

int nnvhip_avgpool2d_destroy(nnvhip_avgpool2d* p) {
  delete p;
  return NNVHIP_OK;
}

int nnvhip_avgpool2d_output_size(const nnvhip_avgpool2d* p, int64_t H, int64_t W, int64_t* Ho, int64_t* Wo) {
  if (!p || !Ho || !Wo) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  // (InputSize + padding - FilterSize)/Stride + 1, rounded down (AveragePooling2DLayer.m:396-418)
  const int64_t h = H + p->pad[0] + p->pad[1] - p->pool[0];
  const int64_t w = W + p->pad[2] + p->pad[3] - p->pool[1];
  if (h < 0 || w < 0) NNV_FAIL(NNVHIP_ERR_SHAPE, "Invalid pool size");
  *Ho = h / p->stride[0] + 1;
  *Wo = w / p->stride[1] + 1;
  return NNVHIP_OK;
}

int nnvhip_affine_avgpool2d(nnvhip_ctx* c, const nnvhip_avgpool2d* p, int64_t H, int64_t W, int64_t count,
                            nnvhip_star* const* in, nnvhip_star** out) {
  if (!c) NNV_FAIL(NNVHIP_ERR_ARG, "null context");
  NNV_TRY(nnvhip::enter_ctx(c));
  if (!p || p->ctx != c) NNV_FAIL(NNVHIP_ERR_ARG, "invalid layer handle");
  NNV_TRY(check_set_array(c, count, in, out));
  if (H <= 0 || W <= 0) NNV_FAIL(NNVHIP_ERR_SHAPE, "The input is not an ImageStar object");
  for (int64_t i = 0; i < count; ++i)
    if (in[i]->N % (H * W) != 0)
      NNV_FAIL(NNVHIP_ERR_SHAPE, "Inconsistent dimension in the ImageStar and the original Star set");
  const int64_t C = in[0]->N / (H * W);
  int64_t Ho = 0, Wo = 0;
  NNV_TRY(nnvhip_avgpool2d_output_size(p, H, W, &Ho, &Wo));
  if (in[0]->N >= (int64_t(1) << 31) || Ho * Wo * C >= (int64_t(1) << 31)) NNV_FAIL(NNVHIP_ERR_SHAPE, "image too large");
  PoolArgs a{};
  a.ldin = in[0]->ld;
  a.H = (int32_t)H;
  a.W = (int32_t)W;
  a.C = (int32_t)C;
  a.Ho = (int32_t)Ho;
  a.Wo = (int32_t)Wo;
  a.ph = (int32_t)p->pool[0];
  a.pw = (int32_t)p->pool[1];
  a.sh = (int32_t)p->stride[0];
  a.sw = (int32_t)p->stride[1];
  a.pt = (int32_t)p->pad[0];
  a.pl = (int32_t)p->pad[2];
  {
    std::vector<PoolPlan> plans((size_t)count);
    bool windows = true;
    for (int64_t i = 0; i < count && windows; ++i)
      windows = in[i]->N == in[0]->N && in[i]->ld == in[0]->ld && pool_in_windows(c, p, in[i], H, W, Ho, Wo, &plans[(size_t)i]);
    if (windows) return pool_windows(c, p, a, count, in, plans.data(), out);
  }
  return run_row_layer(c, count, in, out, Ho * Wo * C, 64, 4 * kEwWaves,
                       [&](dim3 grid, const SetDesc* table, const SetDesc& one, int32_t cpc, int64_t ldout) {
                         a.cols_per_chunk = cpc;
                         a.ldout = ldout;
                         NNV_LAUNCH(c, c->kernel_timing, avgpool_kernel, grid, dim3(64 * kEwWaves), 0, table, one, a);
                       });
}

int nnvhip_permute_rows(nnvhip_ctx* c, int64_t N, const int32_t* src_row, int64_t count, nnvhip_star* const* in,
                        nnvhip_star** out) {
  if (!c) NNV_FAIL(NNVHIP_ERR_ARG, "null context");
  NNV_TRY(nnvhip::enter_ctx(c));
  if (!src_row) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  NNV_TRY(check_set_array(c, count, in, out));
  for (int64_t i = 0; i < count; ++i)
    if (in[i]->N != N) NNV_FAIL(NNVHIP_ERR_SHAPE, "Inconsistent dimension in the ImageStar and the original Star set");
  if (N >= (int64_t(1) << 31)) NNV_FAIL(NNVHIP_ERR_SHAPE, "image too large");
  const int64_t ld = round_up(N, kLdAlign);
  std::vector<int32_t> host((size_t)ld, -1);
  std::vector<char> seen((size_t)N, 0);
  for (int64_t r = 0; r < N; ++r) {
    if (src_row[r] < 0 || src_row[r] >= N || seen[(size_t)src_row[r]]) NNV_FAIL(NNVHIP_ERR_ARG, "not a permutation");
    seen[(size_t)src_row[r]] = 1;
    host[(size_t)r] = src_row[r];
  }
  BufRef perm;
  NNV_TRY(c->upload(host.data(), sizeof(int32_t) * host.size(), &perm));
  PermArgs a{};
  a.src_row = perm->as<int32_t>();
  a.ldin = in[0]->ld;
  if (ld <= kPermLdsRows)
    return run_row_layer(c, count, in, out, N, int64_t(1) << 30, perm_columns((int)N),
                         [&](dim3 grid, const SetDesc* table, const SetDesc& one, int32_t cpc, int64_t ldout) {
                           a.cols_per_chunk = cpc;
                           a.ldout = ldout;
                           const int step = perm_columns((int)N);
                           NNV_LAUNCH(c, c->kernel_timing, permute_rows_lds_kernel, grid, dim3(64 * kEwWaves),
                                      sizeof(double) * step * perm_stride((int)N), table, one, a, (int)N, step);
                         }, true);
  return run_row_layer(c, count, in, out, N, kEwRows, 4 * kEwWaves,
                       [&](dim3 grid, const SetDesc* table, const SetDesc& one, int32_t cpc, int64_t ldout) {
                         a.cols_per_chunk = cpc;
                         a.ldout = ldout;
                         NNV_LAUNCH(c, c->kernel_timing, permute_rows_kernel, grid, dim3(64 * kEwWaves), 0, table, one, a);
                       });
}

}  // extern "C"
