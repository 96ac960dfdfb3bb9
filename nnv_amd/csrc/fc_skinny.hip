// A fully connected layer of at most 32 outputs behind a ReLU step (the last layer of most networks) in one launch, straight
// from what the step recorded:
//   out(:, j) = W(:, kept) * V(kept, j)   for the columns the ReLU's input had (j = 0: plus the bias),
//   out(:, j) = W(:, r)                   for the unit vector e_r of a neuron that crosses zero,
// and the four sums of Star.estimateRanges of every tile of columns.  Columns of V that are themselves weight columns nobody
// has written yet (ColSource::pending) are read from those weights.
//
// What bounds it: the latency of its two trips to memory (row list, operands); the work is a few MFLOP.  So a block takes one
// 16-column tile, its waves every fourth (eighth, sixteenth) group of four kept rows each, and eight groups' operands are asked
// for before the first is multiplied.  The waves' sums meet in the LDS in wave order.  It stands for three to six launches that
// wrote the pending columns, a copy of the matrix with its rows reset and unit vectors appended, a dense product over all of it
// (split along K where it leaves the chip idle) and a scan of the result: 10 outputs of 1024 neurons behind an 845-column set
// 4.7 + 8.0 + 5.0 + 3.1 + 6.0 us in five launches -> 9.3 (and 9.1 with eight waves), of 100 neurons behind 1080 columns 4.0 + 5.9 +
// 5.4 -> 4.6, 25 of those 8.4 + 13.9 + 8.4 + 3.8 + 10.0 -> 11.9 (18.2 with eight waves), 100 sets of 1600 columns through 1024
// neurons 49.4 + 25.8 + 4.5 + 16.2 -> 43.  (Columns staged through the LDS, half a wave to a column along the listed rows,
// touch a quarter of the lines per load and were no faster: 9.2, 5.7, 15.6 us of the first three.)
#include <algorithm>
#include <vector>

#include "internal.h"
#include "mfma_tile.h"

namespace nnvhip {

namespace {

struct SkinnySet {
  const double* V;      // the ReLU's input, column j at V + j * ld
  const int32_t* kept;  // nkept rows, then -1 up to a multiple of 16 (at least 16 entries)
  const int32_t* unit;  // rows of the unit vectors: columns dense .. ncols - 1
  double* out;          // column 0 of the output
  const double* plb;
  const double* pub;
  double* part;         // [chunks][4][Mp]: a chunk per contracted tile, then one per block of unit vectors
  // columns [cfrom, cend) are (0 + cW(:, cidx[j - cfrom]) * cscale[...]) of the layer before (cW null: none)
  const double* cW;
  const int32_t* cidx;
  const double* cscale;
  int64_t ld, cld;
  int32_t nkept, dense, ncols;
  int32_t cfrom, cend;
  int32_t zero_to;      // > 1: columns [1, zero_to) are zero
};

constexpr int kSkinnyRows = 1024;  // entries of the row list in the LDS at a time

// FM: row blocks of 16, NW: waves.  Grid: (contracted tiles, then blocks of 16 NW unit vectors; sets).
template <int FM, int NW>
__global__ __launch_bounds__(64 * NW) void fc_skinny_kernel(const SkinnySet* __restrict__ table, SkinnySet one,
                                                            const double* __restrict__ W, const double* __restrict__ bias) {
  constexpr int Mp = 16 * FM, kAhead = 8;
  SkinnySet S = table ? table[blockIdx.y] : one;
  S.V = in_global(S.V);
  S.kept = in_global(S.kept);
  S.unit = in_global(S.unit);
  S.out = in_global(S.out);
  S.plb = in_global(S.plb);
  S.pub = in_global(S.pub);
  S.part = in_global(S.part);
  S.cW = in_global(S.cW);
  S.cidx = in_global(S.cidx);
  S.cscale = in_global(S.cscale);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  const int tiles = (S.dense + 15) / 16;
  const int tile = blockIdx.x;
  __shared__ double acc_s[NW][FM][4][64];
  __shared__ double red[NW][FM][4][16];
  __shared__ int rows_s[kSkinnyRows];
  double* part = S.part + (int64_t)tile * 4 * Mp;
  if (tile >= tiles) {
    const int j0 = S.dense + 16 * NW * (tile - tiles);
    if (j0 >= S.ncols) return;
    // a wave's sixteen unit vectors: lane (row l16, column q + 4 r) takes four of them and adds their terms
    double s[FM][4];
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int a = 0; a < 4; ++a) s[f][a] = 0.0;
    int src[4];
    double pl[4], pu[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = j0 + 16 * wave + q + 4 * r;
      const bool in = j < S.ncols;
      src[r] = in ? S.unit[j - S.dense] : -1;
      pl[r] = in ? S.plb[j - 1] : 0.0;
      pu[r] = in ? S.pub[j - 1] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = j0 + 16 * wave + q + 4 * r;
#pragma unroll
      for (int f = 0; f < FM; ++f) {
        if (src[r] < 0) continue;
        const double v = __dadd_rn(0.0, W[(int64_t)src[r] * Mp + 16 * f + l16]);
        S.out[(int64_t)j * Mp + 16 * f + l16] = v;
        const double p = fmax(v, 0.0), n = fmin(v, 0.0);
        s[f][0] = fma(p, pl[r], s[f][0]);
        s[f][1] = fma(n, pu[r], s[f][1]);
        s[f][2] = fma(p, pu[r], s[f][2]);
        s[f][3] = fma(n, pl[r], s[f][3]);
      }
    }
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        s[f][a] += __shfl_xor(s[f][a], 16);
        s[f][a] += __shfl_xor(s[f][a], 32);
        if (lane < 16) red[wave][f][a][lane] = s[f][a];
      }
    __syncthreads();
    if (tid < 4 * Mp) {
      const int a = tid / Mp, r = tid % Mp;
      double x = 0.0;
#pragma unroll
      for (int w = 0; w < NW; ++w) x += red[w][r / 16][a][r % 16];
      part[a * Mp + r] = x;
    }
    return;
  }
  // the lane's column, as the matrix product's first operand
  const int j = 16 * tile + l16;
  const double* col = S.V;
  double scale = 1.0;
  const bool zero = j >= S.dense || (j >= 1 && j < S.zero_to);
  if (!zero) {
    if (S.cW != nullptr && j >= S.cfrom && j < S.cend) {
      const int src = S.cidx[j - S.cfrom];
      col = S.cW + (int64_t)src * S.cld;
      if (S.cscale != nullptr) scale = S.cscale[src];
    } else {
      col = S.V + (int64_t)j * S.ld;
    }
  }
  // the column whose results a lane holds at the end: wave w has columns 16 tile + q + 4 (w mod 4), row blocks w / 4, ...
  const int r_out = wave % 4, j_out = 16 * tile + q + 4 * r_out;
  const bool j_in = j_out < S.dense;
  double pl = 0.0, pu = 0.0;
  if (j_in && j_out > 0) pl = S.plb[j_out - 1], pu = S.pub[j_out - 1];
  double4_t acc[FM];
#pragma unroll
  for (int f = 0; f < FM; ++f) acc[f] = double4_t{0.0, 0.0, 0.0, 0.0};
  for (int k0 = 0; k0 < S.nkept; k0 += kSkinnyRows) {
    const int n = min(kSkinnyRows, S.nkept - k0);
    if (k0 > 0) __syncthreads();
    for (int t = tid; t < n; t += 64 * NW) rows_s[t] = S.kept[k0 + t];
    __syncthreads();
    const int groups = (n + 3) / 4;
    for (int g0 = wave; g0 < groups; g0 += NW * kAhead) {
      double w[kAhead][FM], v[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int t = 4 * (g0 + u * NW) + q;
        v[u] = 0.0;
#pragma unroll
        for (int f = 0; f < FM; ++f) w[u][f] = 0.0;
        if (t < n) {
          const int row = rows_s[t];
          if (!zero) v[u] = col[row];
#pragma unroll
          for (int f = 0; f < FM; ++f) w[u][f] = W[(int64_t)row * Mp + 16 * f + l16];
        }
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        if (g0 + u * NW >= groups) break;  // (the same for the whole wave)
        const double x = __dadd_rn(0.0, __dmul_rn(v[u], scale));  // (as the gather pass forms a weight column's entries)
#pragma unroll
        for (int f = 0; f < FM; ++f) acc[f] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, w[u][f], acc[f], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int f = 0; f < FM; ++f)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc_s[wave][f][r][lane] = acc[f][r];
  __syncthreads();
  for (int f = wave / 4; f < FM; f += NW / 4) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) v += acc_s[w][f][r_out][lane];
    if (j_in) S.out[(int64_t)j_out * Mp + 16 * f + l16] = j_out == 0 && bias != nullptr ? v + bias[16 * f + l16] : v;
    if (!j_in || j_out == 0) v = 0.0;  // (the centre takes no part in the sums: an infinite one would leave 0 * Inf there)
    const double p = fmax(v, 0.0), n = fmin(v, 0.0);
    double s[4] = {p * pl, n * pu, p * pu, n * pl};
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      s[a] += __shfl_xor(s[a], 16);
      s[a] += __shfl_xor(s[a], 32);
      if (lane < 16) red[r_out][f][a][lane] = s[a];
    }
  }
  __syncthreads();
  if (tid < 4 * Mp) {
    const int a = tid / Mp, r = tid % Mp;
    double x = 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) x += red[u][r / 16][a][r % 16];
    part[a * Mp + r] = x;
  }
}

}  // namespace

// columns of the set that are contracted: those the step's input had
static int64_t leading_columns(const nnvhip_star* s) { return s->oh_from > 0 ? s->oh_from : s->n + 1; }

// (finite weights: an infinite one times the zero of a reset row is NaN, and the rows left out count then)
bool fc_skinny_layer(const nnvhip_fc* fc) { return fc->Mp <= 32 && fc->finite && fc->K < (int64_t(1) << 30); }

bool fc_skinny_takes(const nnvhip_fc* fc, int64_t count, nnvhip_star* const* in) {
  // (matrices of a shared-product call take the same way whether somebody has had them written or not: ColSource::delta)
  if (!fc_skinny_layer(fc) || count > 65535) return false;
  int64_t empty = 0;
  double gathered = 0.0;
  for (int64_t i = 0; i < count; ++i) {
    const nnvhip_star* s = in[i];
    const int64_t nc = s->n + 1, lead = leading_columns(s);
    if (!s->rows_pending || s->kept_idx == nullptr || s->n_kept < 0 || lead > nc || s->oh_scale != nullptr ||
        (lead < nc && s->oh_idx == nullptr) || s->stored_cols() != lead || s->cs.win_pending() || s->cs.delta ||
        nc >= (int64_t(1) << 30))
      return false;
    empty += s->n_kept == 0;
    gathered = std::max(gathered, (double)fc->Mp * (double)fc->Kp * (double)(nc - lead) * (double)count);
  }
  // Beyond what one launch is bound by, sets without kept rows are left to the gather pass, which fills their zero columns as it
  // goes (1024 sets of 2600 columns, none with kept rows: 1.99 ms a reach there, 2.30 here; 100 of 1300, most of them with some:
  // 3.29 there, 3.21 here).
  return gathered < 4.0e6 || 2 * empty <= count;
}

// Waves of a block, by the longest row list of the call
int fc_skinny_waves(const nnvhip_fc* fc, int64_t count, nnvhip_star* const* in) {
  int64_t kept = 0;
  for (int64_t i = 0; i < count; ++i) kept = std::max(kept, in[i]->n_kept);
  return kept <= 128 ? 4 : fc->Mp == 16 ? 16 : 8;
}

int64_t fc_skinny_chunks(const nnvhip_star* in, int waves) {
  const int64_t lead = leading_columns(in);
  return ceil_div(lead, 16) + ceil_div(in->n + 1 - lead, 16 * waves);
}

int launch_fc_skinny(nnvhip_ctx* ctx, const nnvhip_fc* fc, int64_t count, nnvhip_star* const* in, nnvhip_star* const* out, double* const* part,
                     int waves) {
  std::vector<SkinnySet> sets((size_t)count);
  int64_t blocks = 1;
  double flop = 0.0;
  for (int64_t i = 0; i < count; ++i) {
    const nnvhip_star* s = in[i];
    SkinnySet& d = sets[(size_t)i];
    d = SkinnySet{};
    d.V = s->V;
    d.ld = s->ld;
    d.kept = s->kept_idx;
    d.nkept = (int32_t)s->n_kept;
    d.unit = s->oh_idx;
    d.dense = (int32_t)leading_columns(s);
    d.ncols = (int32_t)(s->n + 1);
    d.out = out[i]->V;
    d.plb = out[i]->plb;
    d.pub = out[i]->pub;
    d.part = part[i];
    if (s->cs.pending) {
      d.cW = s->cs.W;
      d.cld = s->cs.ldw;
      d.cidx = s->cs.idx;
      d.cscale = s->cs.scale;
      d.cfrom = (int32_t)s->cs.from;
      d.cend = (int32_t)(s->cs.from + s->cs.cols);
    }
    d.zero_to = (int32_t)s->cs.zero_to;
    blocks = std::max(blocks, fc_skinny_chunks(s, waves));
    flop += 2.0 * (double)fc->Mp * (double)s->n_kept * (double)d.dense;
  }
  const SkinnySet* table = nullptr;
  BufRef tab;
  if (count > 1) {
    NNV_TRY(ctx->upload_table(sets.data(), sizeof(SkinnySet) * sets.size(), &tab));
    table = tab->as<SkinnySet>();
  }
  const double* bias = fc->bias ? fc->bias->as<double>() : nullptr;
  const dim3 grid((unsigned)blocks, (unsigned)count);
  const double* W = fc->W->as<double>();
  if (fc->Mp == 16 && waves == 4)
    NNV_LAUNCH(ctx, ctx->kernel_timing, (fc_skinny_kernel<1, 4>), grid, dim3(256), 0, table, sets[0], W, bias);
  else if (fc->Mp == 16)
    NNV_LAUNCH(ctx, ctx->kernel_timing, (fc_skinny_kernel<1, 16>), grid, dim3(1024), 0, table, sets[0], W, bias);
  else if (waves == 4)
    NNV_LAUNCH(ctx, ctx->kernel_timing, (fc_skinny_kernel<2, 4>), grid, dim3(256), 0, table, sets[0], W, bias);
  else
    NNV_LAUNCH(ctx, ctx->kernel_timing, (fc_skinny_kernel<2, 8>), grid, dim3(512), 0, table, sets[0], W, bias);
  NNV_TRY(ctx->kernel_timer_end(ctx->kernel_timing, 13, flop));
  NNV_HIP_TRY(hipGetLastError());
  ctx->routes[NNVHIP_ROUTE_FC_SKINNY] += count;
  return NNVHIP_OK;
}

}  // namespace nnvhip
