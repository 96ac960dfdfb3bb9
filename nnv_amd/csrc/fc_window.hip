// affineMap of a fully connected layer behind the convolutional part of a network: C = W * [c V] where every generator
// image of V is zero outside a small window (nnvhip_star::box).
//
// What bounds it: fp64 MFMA where the call is large, the latency of a short chain of stages where it is one small set.
// The dense contraction multiplies whole images; 784 pixels of a 28 x 28 image through two convolutions leave columns of
// 9 .. 16 positions out of 196.  Here the columns are put in order of where their windows start (a counting sort along
// strips two positions wide, walked back and forth), and a tile contracts its columns over the kept rows of the windows'
// union only: about 25 of 196 positions for 64 neighbouring columns of that network.  Rows the union leaves out hold zeros
// in every column of the tile, so a column is the sum of the same products in the same ascending order as the contraction
// over all kept rows; only sums over columns (the range sums) and over the whole image (the centre, whose partial
// products are formed next to the sort) are cut differently.
//
// Two stages of operands are in flight in front of the one that is multiplied, none of them behind a branch: one stage ahead,
// loads under their conditions 42.7 us (32 x 32 x 3 through four convolutions), 18.9 (28 x 28 x 1 through two) and 106 (25 of
// those), now 39.3, 15.4 and 95; the centre's partial products next to the sort likewise (25 sets 24.3 -> 21.1 us).
//
// Measured as it came in, kernels of the layer alone: 25 sets of 28 x 28 x 1 through two convolutions into 100 rows, 25 zero fills and a
// product 875 us -> 142 us; one such set 45 -> 24 us; 32 x 32 x 3 through four convolutions into 512 rows (15 000 columns,
// windows of 16 of 49 positions) 174 -> 65 us.
//
// The images are read inside their windows only, so a set whose zeros around the windows have not been written
// (ColSource::win_box) needs no pass that writes them.
#include <algorithm>

#include "internal.h"
#include "mfma_tile.h"
#include "relu_sort.h"
#include "window_sort.h"

namespace nnvhip {

struct FcWinSet {
  const double* V;            // column 0: the centre; columns 1 .. ncols - 1: the images
  int64_t ld;
  const ColBox* box;          // by column
  const uint32_t* keep_bits;  // one bit per row (1: kept), or null
  const int32_t* cls;         // ... or the rows' classes, or null: every row counts
  const int32_t* kept;        // the rows the centre is multiplied over (null: all nk)
  int32_t* order;             // ncols - 1 column numbers by window start
  double* cpart;              // [cchunks][Mp]: partial products of the centre
  double* out;
  const double* plb;
  const double* pub;
  double* rpart;              // [tiles][4][ldo] range sums
  int32_t ncols, tiles, nk, kper, cchunks;
  // images kept pixel by pixel (ColSource::pix), those of all sets or of none
  const double* pix;
  int64_t pix_ld;
  int32_t pix_eh, pix_ew;
};
struct FcWinArgs {
  const double* W;
  const double* bias;
  int64_t lda, ldo;
  int32_t Mp, H, Wd, C;  // Wd: the image's width
  int32_t shift;         // window starts are told apart in steps of 1 << shift positions
  int32_t buckets;
  int32_t tiles_m;
  int32_t sort_blocks, sort_run;
};

// This block's set.
__device__ __forceinline__ FcWinSet win_set(const FcWinSet* __restrict__ table, const FcWinSet& one) {
  FcWinSet s = table ? in_global(table)[blockIdx.y] : one;
  s.V = in_global(s.V);
  s.box = in_global(s.box);
  s.keep_bits = in_global(s.keep_bits);
  s.cls = in_global(s.cls);
  s.kept = in_global(s.kept);
  s.order = in_global(s.order);
  s.cpart = in_global(s.cpart);
  s.out = in_global(s.out);
  s.plb = in_global(s.plb);
  s.pub = in_global(s.pub);
  s.rpart = in_global(s.rpart);
  s.pix = in_global(s.pix);
  return s;
}

// Place of a window's start on a walk over strips two positions wide, up one strip and down the next, so that columns
// next to one another in the order start next to one another.  An empty window goes first.
__device__ __forceinline__ int window_bucket(ColBox b, const FcWinArgs& a) {
  if (b.h0 > b.h1) return 0;
  const int h = b.h0 >> a.shift, w = b.w0 >> a.shift, hs = ((a.H - 1) >> a.shift) + 1;
  const int strip = w >> 1;
  return min((strip * hs + ((strip & 1) ? hs - 1 - h : h)) * 2 + (w & 1), a.buckets - 1);
}

// The first sort_blocks blocks of a set: the stable counting sort of its columns by window start.  The other blocks: a share
// of the rows of the centre's product each.  Grid: (sort blocks + centre blocks, sets).
__global__ __launch_bounds__(kSortThreads) void fc_window_setup_kernel(const FcWinSet* __restrict__ table, FcWinSet one, FcWinArgs a) {
  const FcWinSet S = win_set(table, one);
  const int tid = threadIdx.x;
  if ((int)blockIdx.x >= a.sort_blocks) {  // rows [k0, k1) of the centre's product; a row of the output per thread, groups of threads interleave
    __shared__ double red[kSortThreads];
    const int chunk = blockIdx.x - a.sort_blocks;
    if (chunk >= S.cchunks) return;
    const int k0 = chunk * S.kper, k1 = min(S.nk, k0 + S.kper);
    const int rp = min(kSortThreads, (a.Mp + 63) / 64 * 64), groups = kSortThreads / rp;
    const int g = tid / rp;
    for (int m0 = 0; m0 < a.Mp; m0 += rp) {
      const int row = m0 + tid % rp;
      double s = 0.0;
      if (g < groups && row < a.Mp)
        for (int kk = k0 + g; kk < k1; kk += 8 * groups) {  // eight rows' loads in flight
          double w[8], v[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const int k = min(kk + u * groups, k1 - 1);
            const int r = S.kept != nullptr ? S.kept[k] : k;
            w[u] = a.W[row + (int64_t)r * a.lda];
            v[u] = S.V[r];
          }
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (kk + u * groups < k1) s = fma(w[u], v[u], s);
        }
      red[tid] = s;
      __syncthreads();
      if (g == 0 && row < a.Mp) {
        for (int q = 1; q < groups; ++q) s += red[q * rp + tid];
        S.cpart[(int64_t)chunk * a.Mp + row] = s;
      }
      __syncthreads();
    }
    return;
  }
  sort_windows(S.ncols - 1, a.buckets, S.order, nullptr, a.sort_run, blockIdx.x, [&](int j) { return window_bucket(S.box[j], a); });
}

__device__ double g_win_zero[1];  // what an element outside its image's window is read from (never written)

// TM x TN output tile per block of WR x WC waves.  Column tiles are dealt to the XCDs (blockIdx.x % 8) with all their row
// tiles, which read the same images.  The last column tile of a set is its centre: the sum of the partial products.
// PIXELS: every set's images are kept pixel by pixel (ColSource::pix).  A listed row then has a place in the image beside its number
// and its position.  As one kernel for both ways, with lists of half the length and eight registers more, a CU held one block of
// 64 x 64 less and unions of windows went through several lists: 25 images of 28 x 28 x 1 and of 40 x 40 x 1, column by column, 119 and
// 245 us, 101 and 213 apart (101 and 206 before there were pixels); pixel by pixel 115 and 232, 101 and 204 now.
constexpr int kWinRows = 2048, kWinPixelRows = 1536;  // rows a stage list holds; a union with more kept rows is walked in several lists
template <int TM, int TN, int WR, int WC, int KT, bool PIXELS>
__global__ __launch_bounds__(64 * WR * WC, TN == 64 ? 6 : 4) void fc_window_kernel(const FcWinSet* __restrict__ table, FcWinSet one, FcWinArgs a) {
  constexpr int NT = 64 * WR * WC, NW = WR * WC;
  constexpr int FM = TM / WR / 16, FN = TN / WC / 16;
  constexpr int LDA_S = TM + kPadRow, LDB_S = KT + kPadK;
  static_assert(NT == TN * KT / 2, "one pair of rows of the image tile per thread");
  __shared__ double Ws[2][KT * LDA_S];
  __shared__ double Vs[2][TN * LDB_S];
  // rows of the union's windows, padded to whole stages: ascending; of images kept pixel by pixel pixel by pixel
  constexpr int kRows = PIXELS ? kWinPixelRows : kWinRows;
  // where they lie in an image (x) and their positions (y): h | w << 16 (-1: none) ...
  __shared__ __attribute__((aligned(16))) int2 s_at[kRows + KT];
  __shared__ int s_row[PIXELS ? kRows + KT : 1];  // ... and their numbers where an image is kept pixel by pixel
  __shared__ int s_col[TN];
  __shared__ double s_pl[TN], s_pu[TN];
  __shared__ int s_u[4];
  __shared__ int s_cnt[NW];
  const FcWinSet S = win_set(table, one);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  // The sets of an array begin on one XCD after the other, and with another of their tiles: an XCD hands its blocks to its four
  // shader engines in turn, which have 24 places each, and the tiles of a set past the last multiple of eight would be the same
  // engines' in every set.  25 sets of 14 tiles, twice 64 rows: 25 blocks each on some - a block of 40 us runs behind
  // the others - and 23 at most this way: 93 -> 75 us (87 with the XCDs alone).
  const int y = blockIdx.y, turned = (slot + y + (y >> 2)) % (int)(gridDim.x >> 3);
  const int mt = turned % a.tiles_m, nt = (turned / a.tiles_m) * 8 + ((xcd + y) & 7);
  if (nt > S.tiles) return;
  const int m0 = mt * TM;

  if (nt == S.tiles) {  // the centre
    constexpr int G = NT / TM;
    double* red = &Ws[0][0];
    const int row = m0 + tid % TM, g = tid / TM;
    double s = 0.0;
    if (row < a.Mp)
      for (int q = g; q < S.cchunks; q += G) s += S.cpart[(int64_t)q * a.Mp + row];
    red[tid] = s;
    __syncthreads();
    if (g == 0 && row < a.Mp) {
      for (int q = 1; q < G; ++q) s += red[q * TM + tid];
      S.out[row] = a.bias != nullptr ? s + a.bias[row] : s;  // newV(:,1) = newV(:,1) + b
    }
    return;
  }

  if (wave == 0) {  // the tile's columns and the union of their windows
    const int j = nt * TN + lane;
    const int col = lane < TN && j < S.ncols - 1 ? S.order[j] : -1;
    int h0 = 0x7fff, h1 = -1, w0 = 0x7fff, w1 = -1;
    if (col >= 0) {
      const ColBox b = S.box[col];
      if (b.h0 <= b.h1) h0 = b.h0, h1 = b.h1, w0 = b.w0, w1 = b.w1;
    }
    if (lane < TN) {
      s_col[lane] = col;
      s_pl[lane] = col >= 0 ? S.plb[col - 1] : 0.0;
      s_pu[lane] = col >= 0 ? S.pub[col - 1] : 0.0;
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      h0 = min(h0, __shfl_xor(h0, off));
      h1 = max(h1, __shfl_xor(h1, off));
      w0 = min(w0, __shfl_xor(w0, off));
      w1 = max(w1, __shfl_xor(w1, off));
    }
    if (lane == 0) s_u[0] = h0, s_u[1] = h1, s_u[2] = w0, s_u[3] = w1;
  }
  __syncthreads();
  const int uh0 = s_u[0], uw0 = s_u[2];
  const int uh = max(0, s_u[1] - uh0 + 1), uw = max(0, s_u[3] - uw0 + 1);
  const int P = uh * uw, total = P * a.C, HW = a.H * a.Wd;

  // the image this thread stages: rows 2 * (tid % 8) and the next of every stage, of column tid / 8
  const int bj = tid / (KT / 2), bk = 2 * (tid % (KT / 2));
  const int bcol = s_col[bj];
  const double* img = PIXELS ? S.pix + (int64_t)max(bcol, 0) * S.pix_ld : S.V + (int64_t)max(bcol, 0) * S.ld;
  ColBox bb = {0x4000, 0x4000, 0, 0};  // (images have at most 8192 rows and columns)
  if (bcol >= 0) {
    const ColBox b = S.box[bcol];
    if (b.h0 <= b.h1 && b.w0 <= b.w1) bb = b;
  }
  const unsigned hspan = bb.h1 - bb.h0, wspan = bb.w1 - bb.w0;
  const double* const zero = g_win_zero;

  double4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};

  constexpr int A_VEC = TM * KT / 2, A_PASS = (A_VEC + NT - 1) / NT;
  // A stage's operands travel through registers while the two stages before it are multiplied.  Every load is issued whatever
  // its row and column are: behind a branch the compiler would wait for all loads in flight.  (An element that is not wanted is
  // read from a zero; a row behind the list, or a row of the tile behind the weights, meets zeros or is not stored.)
  typedef double pair_t __attribute__((ext_vector_type(2)));
  struct Regs {
    pair_t a[A_PASS], b;
  };
  const double* const weights = a.W + min(m0 + 2 * (tid % (TM / 2)), a.Mp - 2);
  auto load_tiles = [&](int k0, Regs& g) {
#pragma unroll
    for (int p = 0; p < A_PASS; ++p) {
      const int k = min((tid + p * NT) / (TM / 2), KT - 1);
      const uint32_t row = PIXELS ? s_row[k0 + k] : s_at[k0 + k].x;
      g.a[p] = *reinterpret_cast<const pair_t*>(weights + (uint64_t)row * (uint32_t)a.lda);
    }
    int4 two = *reinterpret_cast<const int4*>(&s_at[k0 + bk]);
    asm("" : "+v"(two.x), "+v"(two.z));  // (read here, not behind a branch on the window tests)
    auto pixel = [&](int at, int pos) {
      const int h = pos & 0xffff, w = pos >> 16;  // (h past any window where there is no row)
      const bool in = ((unsigned)(h - bb.h0) <= hspan) & ((unsigned)(w - bb.w0) <= wspan);
      return in_global(in ? img + at : zero)[0];
    };
    g.b.x = pixel(two.x, two.y);
    g.b.y = pixel(two.z, two.w);
  };
  auto store_tiles = [&](int buf, const Regs& g) {
#pragma unroll
    for (int p = 0; p < A_PASS; ++p) {
      const int idx = tid + p * NT;
      if (A_PASS * NT == A_VEC || idx < A_VEC) *reinterpret_cast<pair_t*>(&Ws[buf][(idx / (TM / 2)) * LDA_S + 2 * (idx % (TM / 2))]) = g.a[p];
    }
    Vs[buf][bj * LDB_S + bk] = g.b.x;  // odd column stride: two 64-bit stores
    Vs[buf][bj * LDB_S + bk + 1] = g.b.y;
  };
  static_assert(NT % (TM / 2) == 0, "a thread's weights are of the same rows in every pass");

  const int wr = wave % WR, wc = wave / WR;
  for (int cand = 0; cand < total;) {
    int nrow = 0;
    while (cand < total && nrow + NT <= kRows) {  // kept rows among the next NT of the union, ascending
      const int e = cand + tid;
      bool keep = e < total;
      int r = 0, h = 0, w = 0, ch = 0;
      if (keep) {
        int q;
        if (PIXELS) {
          q = e / a.C;
          ch = e - q * a.C;
        } else {
          ch = e / P;
          q = e - ch * P;
        }
        w = q / uh;
        h = uh0 + q - w * uh;
        w += uw0;
        r = ch * HW + w * a.H + h;
        if (S.keep_bits != nullptr) keep = (S.keep_bits[r >> 5] >> (r & 31)) & 1;
        else if (S.cls != nullptr) keep = S.cls[r] == kKeep;
      }
      const unsigned long long m = __ballot(keep);
      if (lane == 0) s_cnt[wave] = __popcll(m);
      __syncthreads();
      int before = nrow;
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        const int c = s_cnt[v];
        before += v < wave ? c : 0;
        nrow += c;
      }
      if (keep) {
        const int at = before + __popcll(m & ((1ull << lane) - 1ull));
        s_at[at] = make_int2(PIXELS ? pix_slot(h, w, S.pix_eh, S.pix_ew) * a.C + ch : r, h | (w << 16));
        if (PIXELS) s_row[at] = r;
      }
      __syncthreads();
      cand += NT;
    }
    const int nk = (nrow + KT - 1) / KT;
    if (tid < nk * KT - nrow) {
      s_at[nrow + tid] = make_int2(0, -1);
      if (PIXELS) s_row[nrow + tid] = 0;
    }
    __syncthreads();
    if (nk == 0) continue;
    Regs g0, g1;
    load_tiles(0, g0);
    load_tiles(KT * min(1, nk - 1), g1);
    store_tiles(0, g0);
    __syncthreads();
    auto multiply = [&](int cur) {
      mfma_tile_k16<FM, FN, KT>(&Ws[cur][wr * (TM / WR)], LDA_S, &Vs[cur][(wc * (TN / WC)) * LDB_S], LDB_S, lane, acc);
    };
    // stage t from LDS half t & 1; `next` holds stage t + 1, `far` receives stage t + 2 (past the end: the last again)
    auto step = [&](int t, Regs& next, Regs& far) {
      load_tiles(KT * min(t + 2, nk - 1), far);
      multiply(t & 1);
      store_tiles((t & 1) ^ 1, next);
      __syncthreads();
    };
    for (int t = 0; t + 1 < nk; t += 2) {
      step(t, g1, g0);
      step(t + 1, g0, g1);
    }
    if (nk & 1) {
      multiply(0);
      __syncthreads();
    }
  }

  const int lrow = lane & 15, lcol = lane >> 4;
  // partial sums of Star.estimateRanges over the tile's columns, as in gemm_f64_kernel
  if (S.rpart != nullptr) {
    __syncthreads();
    double* red = &Ws[0][0];
    static_assert(WC * TM * 4 <= 2 * KT * LDA_S, "the sums of the column waves fit the weight stages");
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = wc * (TN / WC) + j * 16 + lcol + 4 * r;  // (a column past the last one: zeros throughout)
          const double v = acc[i][j][r], pl = s_pl[c], pu = s_pu[c];
          const double p = fmax(v, 0.0), q = fmin(v, 0.0);
          s0 = fma(p, pl, s0);
          s1 = fma(q, pu, s1);
          s2 = fma(p, pu, s2);
          s3 = fma(q, pl, s3);
        }
      s0 += __shfl_xor(s0, 16), s1 += __shfl_xor(s1, 16), s2 += __shfl_xor(s2, 16), s3 += __shfl_xor(s3, 16);
      s0 += __shfl_xor(s0, 32), s1 += __shfl_xor(s1, 32), s2 += __shfl_xor(s2, 32), s3 += __shfl_xor(s3, 32);
      if (lcol == 0) {
        double* dst = red + ((wc * TM) + wr * (TM / WR) + i * 16 + lrow) * 4;
        dst[0] = s0, dst[1] = s1, dst[2] = s2, dst[3] = s3;
      }
    }
    __syncthreads();
    for (int t = tid; t < TM * 4; t += NT) {
      const int row = t >> 2, q = t & 3;
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < WC; ++w) s += red[(w * TM + row) * 4 + q];
      if (m0 + row < a.Mp) S.rpart[((int64_t)nt * 4 + q) * a.ldo + m0 + row] = s;
    }
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int row = m0 + wr * (TM / WR) + i * 16 + lrow;
    if (row >= a.Mp) continue;
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = s_col[wc * (TN / WC) + j * 16 + lcol + 4 * r];
        if (col >= 0) S.out[row + (int64_t)col * a.ldo] = acc[i][j][r];
      }
  }
}

static_assert(kFcWindowColumns == kSortColumns, "the columns' windows are sorted");

bool fc_window_takes(const nnvhip_fc* fc, int64_t H, int64_t W) {
  // (0 * Inf is NaN: the rows the union leaves out count then)
  return fc->finite && H >= 1 && W >= 1 && H <= 8192 && W <= 8192 && fc->K % (H * W) == 0 && fc->K < (int64_t(1) << 31) && fc->Mp < (int64_t(1) << 20);
}

int fc_window_tile(const nnvhip_fc* fc, int64_t count, nnvhip_star* const* in, const int64_t* dense) {
  const nnvhip_star* f = in[0];
  if (f->box == nullptr) return 0;
  const int64_t H = f->box_H, W = f->box_W;
  if (!fc_window_takes(fc, H, W)) return 0;
  int64_t cols = 0;
  for (int64_t i = 0; i < count; ++i) {
    const nnvhip_star* s = in[i];
    const ColSource& cs = s->cs;
    if (s->box == nullptr || s->box_H != H || s->box_W != W || s->box_eh != f->box_eh || s->box_ew != f->box_ew) return 0;
    if (dense[i] < 2 || dense[i] > kFcWindowColumns || dense[i] > s->box_cols || dense[i] > s->stored_cols()) return 0;
    // (unit-vector columns carry their one in a row the step has reset: they are the gather pass's)
    if (s->oh_from > 0 && dense[i] > s->oh_from) return 0;
    if (cs.pending || cs.zero_to > 1 || cs.delta_pending()) return 0;
    if (s->rows_pending && s->kept_idx == nullptr) return 0;
    cols += dense[i] - 1;
  }
  return fc_window_tile_of(fc, count, cols, H, W, f->box_eh, f->box_ew);
}

int fc_window_tile_of(const nnvhip_fc* fc, int64_t count, int64_t cols, int64_t H, int64_t W, int64_t eh, int64_t ew) {
  // The positions a tile walks: its columns' windows plus what the columns' starts spread over two strips.  The contraction
  // over all kept rows multiplies at about twice the rate (its stages need no position tests and its tiles are larger), so
  // the line is half of the image: windows of 16 of 49 positions take 65 us here and 174 us there, and from windows as
  // large as half the image on nothing is left to gain.
  const int64_t tiles_m = ceil_div(fc->Mp, 64);
  const int tn = ceil_div(cols, 64) * tiles_m >= 512 ? 64 : 32;
  const double starts = (double)tn * (double)(H * W) * (double)count / (double)cols;  // distinct starts of a tile's columns
  const double uh = std::min((double)H, (double)eh + 0.5 * starts), uw = std::min((double)W, (double)ew + std::min(1.0, starts));
  return 2.0 * uh * uw <= (double)(H * W) ? tn : 0;
}

int launch_fc_window(nnvhip_ctx* ctx, const nnvhip_fc* fc, int tn, int64_t count, const FcWindowSet* sets) {
  if (count < 1) return NNVHIP_OK;
  if (count > 65535) NNV_FAIL(NNVHIP_ERR_SHAPE, "at most 65535 sets per call");
  FcWinArgs a{};
  const nnvhip_star* f = sets[0].in;
  a.W = fc->W->as<double>();
  a.bias = fc->bias ? fc->bias->as<double>() : nullptr;
  a.lda = fc->Mp;
  a.ldo = sets[0].out->ld;
  a.Mp = (int32_t)fc->Mp;
  a.H = f->box_H;
  a.Wd = f->box_W;
  a.C = (int32_t)(fc->K / ((int64_t)a.H * a.Wd));
  auto buckets = [&](int shift) {
    const int64_t hs = ((a.H - 1) >> shift) + 1, ws = ((a.Wd - 1) >> shift) + 1;
    return ceil_div(ws, 2) * hs * 2;
  };
  while (buckets(a.shift) > kSortBuckets) ++a.shift;
  a.buckets = (int32_t)buckets(a.shift);
  const int tm = fc->Mp <= 32 ? 32 : 64;
  a.tiles_m = (int32_t)ceil_div(fc->Mp, tm);
  std::vector<FcWinSet> tab((size_t)count);
  int64_t orders = 0, parts = 0, max_cols = 0, max_tiles = 0, max_chunks = 0;
  for (int64_t i = 0; i < count; ++i) {
    FcWinSet& d = tab[(size_t)i];
    const nnvhip_star* s = sets[i].in;
    d.ncols = (int32_t)sets[i].dense;
    d.tiles = (int32_t)ceil_div(sets[i].dense - 1, tn);
    const bool listed = s->rows_pending || (s->n_kept >= 0 && s->kept_idx != nullptr);
    d.nk = (int32_t)(listed ? s->n_kept : fc->K);
    d.kept = listed ? s->kept_idx : nullptr;
    // (about 64 blocks for one set; an array's blocks fill the chip once)
    d.kper = (int32_t)std::max<int64_t>(32, ceil_div(d.nk, std::max<int64_t>(4, 64 / ceil_div(count, 8))));
    d.cchunks = (int32_t)ceil_div(d.nk, d.kper);
    orders += sets[i].dense;
    parts += d.cchunks;
    max_tiles = std::max<int64_t>(max_tiles, d.tiles);
    max_chunks = std::max<int64_t>(max_chunks, d.cchunks);
    max_cols = std::max<int64_t>(max_cols, sets[i].dense - 1);
  }
  a.sort_run = sort_window_run(max_cols, count);
  a.sort_blocks = sort_window_blocks(max_cols, a.sort_run);
  BufRef order, cpart, dev;
  NNV_TRY(ctx->alloc(sizeof(int32_t) * orders, &order));
  NNV_TRY(ctx->alloc(sizeof(double) * fc->Mp * std::max<int64_t>(parts, 1), &cpart));
  int64_t o = 0, p = 0;
  double flop = 0.0;
  for (int64_t i = 0; i < count; ++i) {
    FcWinSet& d = tab[(size_t)i];
    const nnvhip_star* s = sets[i].in;
    d.V = s->V;
    d.ld = s->ld;
    d.box = s->box;
    if (s->cs.in_pixels() != f->cs.in_pixels()) NNV_FAIL(NNVHIP_ERR_ARG, "internal: images kept in different ways");
    if (s->cs.in_pixels()) {
      d.pix = s->cs.pix;
      d.pix_ld = s->cs.pix_ld;
      d.pix_eh = s->cs.pix_eh;
      d.pix_ew = s->cs.pix_ew;
    }
    if (s->rows_pending) {
      d.keep_bits = s->keep_bits;
      d.cls = s->cls;
    }
    d.order = order->as<int32_t>() + o;
    d.cpart = cpart->as<double>() + p * fc->Mp;
    d.out = sets[i].out->V;
    d.plb = sets[i].out->plb;
    d.pub = sets[i].out->pub;
    d.rpart = sets[i].rpart;
    flop += 2.0 * (double)fc->Mp * (double)(d.ncols - 1) * s->box_eh * s->box_ew * a.C * ((double)d.nk / (double)fc->K);
    o += sets[i].dense;
    p += d.cchunks;
  }
  const FcWinSet* table = nullptr;
  if (count > 1) {
    NNV_TRY(ctx->upload_table(tab.data(), sizeof(FcWinSet) * tab.size(), &dev));
    table = dev->as<FcWinSet>();
  }
  hipLaunchKernelGGL(fc_window_setup_kernel, dim3((unsigned)(a.sort_blocks + max_chunks), (unsigned)count), dim3(kSortThreads), 0, ctx->stream, table,
                     tab[0], a);
  const dim3 grid((unsigned)(round_up(max_tiles + 1, 8) * a.tiles_m), (unsigned)count);
#define NNV_FC_WINDOW(TM, TN, WR, WC, KT)                                                                                                      \
  do {                                                                                                                                         \
    if (f->cs.in_pixels())                                                                                                                     \
      NNV_LAUNCH(ctx, ctx->kernel_timing, (fc_window_kernel<TM, TN, WR, WC, KT, true>), grid, dim3(64 * WR * WC), 0, table, tab[0], a);  \
    else                                                                                                                                       \
      NNV_LAUNCH(ctx, ctx->kernel_timing, (fc_window_kernel<TM, TN, WR, WC, KT, false>), grid, dim3(64 * WR * WC), 0, table, tab[0], a); \
  } while (0)
  // (one small set: a block or none per CU, nothing to hide a stage's loads behind - stages of 32 rows, half as many)
  if (tm == 32 && tn == 32) NNV_FC_WINDOW(32, 32, 2, 2, 16);
  else if (tm == 32) NNV_FC_WINDOW(32, 64, 2, 4, 16);
  else if (tn == 32) NNV_FC_WINDOW(64, 32, 4, 2, 32);
  else NNV_FC_WINDOW(64, 64, 2, 4, 16);
#undef NNV_FC_WINDOW
  NNV_TRY(ctx->kernel_timer_end(ctx->kernel_timing, 11, flop));
  NNV_HIP_TRY(hipGetLastError());
  ctx->routes[NNVHIP_ROUTE_FC_WINDOW] += count;
  return NNVHIP_OK;
}

}  // namespace nnvhip
