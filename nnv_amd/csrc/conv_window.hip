// The generator images of a convolution whose inputs are zero outside known windows (nnvhip_star::box), by output position:
// a block takes one position (h, w) of the output and the columns whose output window covers it - found through a sort of
// the columns by window start - and multiplies the layer's weights with those columns' pixels under the filter,
//   out(h, w, :, column) = sum over the kept input rows r under the filter of Wk(tap of r, :) * V(r, column),
// a small matrix product of the layer's channels x the columns over the kept rows only.
//
// What bounds it: the scattered 8-byte stores into images that lie column by column (without them 67 of 134 us for 4280
// images of 15 x 15 into 64 channels), then fp64 MFMA and the latency of a block's stages.  The implicit GEMM over
// windows (conv2d_fast_kernel<.., COMPACT>) multiplies every tap of every position of a window, among them the rows a ReLU
// step has reset (half of them) - here they are left out, since a block's columns share the position and with it the list of
// rows.  And because a block holds all values of its position (a share of them where there are many columns), it leaves the
// position's sums for Star.estimateRanges in registers' reach: the pass that read the images back for them is not needed.
//
// The products of an element are added in ascending tap order from +0 over the rows that are kept, which is what the
// implicit GEMM adds up besides exact zeros.  Measured against that launch and the scan behind it: 25 sets of 28 x 28 x 1,
// second layer (784 images each into 32 channels of 14 x 14) 270 -> 138 us; 32 x 32 x 3 network, second to fourth layer 77 ->
// 50, 193 -> 137 and 175 -> 160 us.  (Two neighbouring positions per block, stored together: 141 and 209 us for the last two -
// the registers cost a resident block.)
//
// How the range sums are cut depends on the set and the layer only, not on what
// else is in the call.
#include <algorithm>
#include <cstring>

#include "conv_stamp.h"
#include "internal.h"
#include "mfma_tile.h"
#include "relu_sort.h"
#include "window_sort.h"

namespace nnvhip {

struct ConvWinSet {
  const double* V;  // the input; column j at V + j * ld
  int64_t ld;
  const ColBox* in_box;
  const ColBox* out_box;
  const uint32_t* keep_bits;  // one bit per input row (1: kept), or null
  const int32_t* cls;         // ... or the rows' classes, or null: every row counts
  const int32_t* order;       // columns 1 .. ncols - 1 by the start of their output window, w0 * Ho + h0 ...
  const int32_t* first;       // ... and where every start's columns begin (P + 1 entries)
  double* out;
  const double* plb;
  const double* pub;
  double* part;               // [parts][4][ldo] range sums
  int32_t parts;
  int32_t eh, ew;             // bound on the output windows
  // images kept pixel by pixel (ColSource::pix), or null: those of the input, those of the output
  const double* in_pix;
  double* out_pix;
  int64_t in_pix_ld, out_pix_ld;
  int32_t in_eh, in_ew, out_eh, out_ew;
  StampSet stamps;            // unit-vector columns whose stamps go into the same launch (m: 0: none)
};
struct ConvWinArgs {
  const double* Wk;  // k-major weights: tap k's channels at Wk + k * coutp
  const double* bias;
  int64_t ldo;
  const double* Wt;  // the weights tap by tap of a channel (for the stamps)
  ConvGeom g;
  int32_t coutp;
  int32_t per;       // items (position, part) per XCD
  int32_t list;      // entries of a row list
  int32_t stamp_blocks;
};

// PIXELS: places in an image and positions of a filter that fit one word
constexpr int kPosBits = 26, kNoPosition = 31;
__device__ double g_zero[1];  // (never written)
constexpr int kConvWinTaps = 1024;  // taps of a filter (FH * FW * Cin) at most
constexpr int kConvWinStarts = 256;  // positions of an output window at most
constexpr int kConvWinCols = 128;   // columns of a position listed at a time
// TM channels x TN columns per tile, WR x WC waves.  Consecutive items (positions first) stay on one XCD, so that
// neighbouring positions, whose elements share lines of every image, meet in its L2.  Grid: (items, sets, channel tiles).
// The first stamp_blocks blocks of a set write the stamps of its unit-vector columns (S lanes per output row): bound by
// scattered stores, they share the compute units with the products.
//
// PIXELS: every set's images are kept pixel by pixel (ColSource::pix).  A stage's operands are then half of the vector and LDS
// instructions they are for columns: where a listed row lies in an image and which of the filter's positions it belongs to are
// one word, a column's window is one bit per position, made once a tile, and an element that is not wanted is read from a zero
// instead of being dropped later (a row of padding meets zeros, so its weights need not be).  32 x 32 x 3 network, second to
// fourth layer: 38, 129 and 151 us with columns, 26, 97 and 108 with pixels through the same instructions, 22, 85 and 91 with these.
template <int TM, int TN, int WR, int WC, int S_LANES, bool PIXELS>
__global__ __launch_bounds__(64 * WR * WC, TM == 16 ? 3 : 4) void conv_window_kernel(const ConvWinSet* __restrict__ table, ConvWinSet one, ConvWinArgs a) {
  constexpr int NT = 64 * WR * WC, NW = WR * WC;
  constexpr int KT = 16;
  constexpr int FM = TM / WR / 16, FN = TN / WC / 16;
  constexpr int LDA_S = TM + kPadRow, LDB_S = KT + kPadK;
  constexpr int A_VEC = TM * KT / 2, A_PASS = (A_VEC + NT - 1) / NT;
  constexpr int B_PASS = TN * KT / 2 / NT;
  static_assert(NW * 256 <= 2 * TN * LDB_S, "the stamp blocks' sums fit the image stages");
  static_assert(A_PASS * NT == A_VEC && B_PASS * NT == TN * KT / 2 && kConvWinCols % TN == 0, "whole passes, whole tiles");
  __shared__ double Ws[2][KT * LDA_S];
  __shared__ double Vs[2][TN * LDB_S];
  extern __shared__ __attribute__((aligned(16))) int s_rows[];  // kept input rows under the filter, by tap, -1 padded to whole pairs of stages ...
  int* const s_row = s_rows;
  int* const s_tap = s_rows + a.list;      // ... their taps ...
  int* const s_pos = s_rows + 2 * a.list;  // ... and their positions in the image: h | w << 16
  // PIXELS: s_row and s_pos hold where a row lies in the centre and in the other images, | the filter's position << kPosBits
  // (kNoPosition behind the list); s_tap where its weights lie
  __shared__ int s_col[kConvWinCols];
  __shared__ double s_pl[kConvWinCols], s_pu[kConvWinCols];
  __shared__ int s_from[kConvWinStarts], s_end[kConvWinStarts];
  __shared__ int s_cnt[NW];
  ConvWinSet S = table ? in_global(table)[blockIdx.y] : one;
  S.V = in_global(S.V);
  S.in_box = in_global(S.in_box);
  S.out_box = in_global(S.out_box);
  S.keep_bits = in_global(S.keep_bits);
  S.cls = in_global(S.cls);
  S.order = in_global(S.order);
  S.first = in_global(S.first);
  S.out = in_global(S.out);
  S.plb = in_global(S.plb);
  S.pub = in_global(S.pub);
  S.part = in_global(S.part);
  S.in_pix = in_global(S.in_pix);
  S.out_pix = in_global(S.out_pix);
  S.stamps.pix = in_global(S.stamps.pix);
  S.stamps.idx = in_global(S.stamps.idx);
  S.stamps.scale = in_global(S.stamps.scale);
  S.stamps.out = in_global(S.stamps.out);
  S.stamps.plb = in_global(S.stamps.plb);
  S.stamps.pub = in_global(S.stamps.pub);
  S.stamps.part = in_global(S.stamps.part);
  S.stamps.pixel_col = in_global(S.stamps.pixel_col);
  const int blk = (int)blockIdx.x - a.stamp_blocks;
  if (blk < 0) {
    if (S.stamps.m > 0 && blockIdx.z == 0) {
      if (S.stamps.pix != nullptr)
        conv_stamp_pixels_block<NT>(blockIdx.x, &Vs[0][0], s_cnt, reinterpret_cast<int2*>(s_rows), S.stamps, a.g, a.Wk, a.coutp, S.stamps.pixel_col, a.ldo);
      else
        conv_stamp_rows_block<S_LANES, NT>(blockIdx.x, reinterpret_cast<int2*>(s_rows), S.stamps, a.g, a.Wt, S.stamps.pixel_col, a.ldo);
    }
    return;
  }
  const int item = (blk & 7) * a.per + (blk >> 3);  // (stamp_blocks is a multiple of eight)
  if ((blk >> 3) >= a.per || item >= a.g.P * S.parts) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int part = item / a.g.P, p = item - part * a.g.P;
  const int pw = p / a.g.Ho, ph = p - pw * a.g.Ho;
  const int m0 = blockIdx.z * TM;

  // The columns that may cover the position, window start by window start: first the starts whose row is 0 modulo eh, then 1,
  // ... (one row of each class is in reach of the position), by column of the image within a class.  So the blocks of
  // neighbouring rows come to a column at about the same time, and the elements they store next to one another meet in the L2
  // before the line leaves it.
  const int wlo = max(0, pw - S.ew + 1), nw = pw - wlo + 1, runs = S.eh * nw;
  for (int t = tid; t < runs; t += NT) {
    const int c = t / nw, h0 = ph - (ph + S.eh - c) % S.eh;
    const int s = (wlo + t - c * nw) * a.g.Ho + h0;
    s_from[t] = h0 >= 0 ? S.first[s] : 0;
    s_end[t] = h0 >= 0 ? S.first[s + 1] - s_from[t] : 0;
  }
  // kept rows under the filter, in tap order; of images kept pixel by pixel pixel by pixel, so that a stage's rows lie together
  int nrow = 0;
  const int hb = ph * a.g.sh - a.g.pt, wb = pw * a.g.sw - a.g.pl;
  for (int k0 = 0; k0 < a.g.K; k0 += NT) {
    int k = k0 + tid;
    bool keep = k < a.g.K;
    int r = 0, h = 0, w = 0, ci = 0, fh = 0, fw = 0;
    if (keep) {
      if (PIXELS) {
        const int t = k / a.g.Cin;
        ci = k - t * a.g.Cin;
        fw = t / a.g.FH;
        fh = t - fw * a.g.FH;
        k = (ci * a.g.FW + fw) * a.g.FH + fh;
      } else {
        const int t = k / a.g.FH;
        ci = t / a.g.FW;
        fh = k - t * a.g.FH;
        fw = t - ci * a.g.FW;
      }
      h = hb + fh * a.g.dh;
      w = wb + fw * a.g.dw;
      keep = (unsigned)h < (unsigned)a.g.H && (unsigned)w < (unsigned)a.g.W;
      if (keep) {
        r = ci * a.g.HW + w * a.g.H + h;
        if (S.keep_bits != nullptr) keep = (S.keep_bits[r >> 5] >> (r & 31)) & 1;
        else if (S.cls != nullptr) keep = S.cls[r] == kKeep;
      }
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
      if (PIXELS) {
        const int position = (fw * a.g.FH + fh) << kPosBits;
        s_row[at] = r | position;
        s_tap[at] = k * a.coutp;
        s_pos[at] = (pix_slot(h, w, S.in_eh, S.in_ew) * a.g.Cin + ci) | position;
      } else {
        s_row[at] = r;
        s_tap[at] = k;
        s_pos[at] = h | (w << 16);
      }
    }
    __syncthreads();
  }
  const int nk = max(2, (nrow + 2 * KT - 1) / (2 * KT) * 2);  // stages: an even number, so that the loop over them has no branch
  if (tid < nk * KT - nrow) {
    s_row[nrow + tid] = PIXELS ? kNoPosition << kPosBits : -1;
    s_tap[nrow + tid] = 0;
    s_pos[nrow + tid] = PIXELS ? kNoPosition << kPosBits : 0;
  }
  int total = 0;
  for (int g = 0; g < runs; ++g) total += s_end[g];
  __syncthreads();
  if (tid == 0) {
    int end = 0;
    for (int g = 0; g < runs; ++g) s_end[g] = end += s_end[g];  // lengths to ends
  }
  __syncthreads();

  const int wr = wave % WR, wc = wave / WR;
  const int lrow = lane & 15, lcol = lane >> 4;
  double bias[FM];
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int co = m0 + wr * (TM / WR) + i * 16 + lrow;
    bias[i] = a.bias != nullptr && co < a.g.Cout ? a.bias[co] : 0.0;
  }
  const int out_slot = S.out_pix != nullptr ? pix_slot(ph, pw, S.out_eh, S.out_ew) * a.g.Cout : 0;
  double x[FM][4];  // xmin1, xmin2, xmax1, xmax2 of the lane's rows over the columns it has held
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) x[i][q] = 0.0;

  const int lo = (int)((int64_t)total * part / S.parts), hi = (int)((int64_t)total * (part + 1) / S.parts);
  // (the first part's first stretch starts with the centre, which covers every position)
  for (int i0 = lo; i0 < hi || (part == 0 && i0 == lo); i0 += kConvWinCols - 1) {
    // the columns of this stretch whose window covers the position
    int n = 0;
    const int i1 = min(hi, i0 + kConvWinCols - 1);
    if (part == 0 && i0 == lo) {
      n = 1;
      if (tid == 0) {
        s_col[0] = 0;
        s_pl[0] = s_pu[0] = 0.0;
      }
      __syncthreads();
    }
    for (int e0 = i0; e0 < i1; e0 += NT) {
      const int e = e0 + tid;
      bool hit = e < i1;
      int col = 0;
      if (hit) {
        int g = 0;
        for (int hi2 = runs - 1; g < hi2;) {  // the run that holds e: the first that ends behind it
          const int mid = (g + hi2) >> 1;
          if (e < s_end[mid]) hi2 = mid;
          else g = mid + 1;
        }
        col = S.order[s_from[g] + e - (g > 0 ? s_end[g - 1] : 0)];
        const ColBox b = S.out_box[col];
        hit = ph >= b.h0 && ph <= b.h1 && pw >= b.w0 && pw <= b.w1;
      }
      const unsigned long long m = __ballot(hit);
      if (lane == 0) s_cnt[wave] = __popcll(m);
      __syncthreads();
      int before = n;
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        const int c = s_cnt[v];
        before += v < wave ? c : 0;
        n += c;
      }
      if (hit) {
        const int at = before + __popcll(m & ((1ull << lane) - 1ull));
        s_col[at] = col;
        s_pl[at] = S.plb[col - 1];
        s_pu[at] = S.pub[col - 1];
      }
      __syncthreads();
    }
    for (int c0 = 0; c0 < n; c0 += TN) {
      // the images this thread stages: rows 2 * (tid % 8) and the next of every stage
      const int bk = 2 * (tid % (KT / 2));
      const double* img[B_PASS];
      ColBox bb[B_PASS];
      const int* at[B_PASS];       // PIXELS: the list of where the rows lie in it ...
      unsigned inside[B_PASS];     // ... and the filter's positions inside its window
#pragma unroll
      for (int u = 0; u < B_PASS; ++u) {
        const int j = c0 + (tid + u * NT) / (KT / 2);
        bb[u] = ColBox{1, 0, 1, 0};
        img[u] = S.V;
        at[u] = s_pos;
        inside[u] = 0;
        if (j < n) {
          const int col = s_col[j];
          bb[u] = col == 0 ? ColBox{0, (int16_t)(a.g.H - 1), 0, (int16_t)(a.g.W - 1)} : S.in_box[col];
          img[u] = PIXELS && col > 0 ? S.in_pix + (int64_t)col * S.in_pix_ld : S.V + (int64_t)col * S.ld;
          if (PIXELS) {
            if (col == 0) at[u] = s_row;
            for (int fw = 0; fw < a.g.FW; ++fw) {
              const int w = wb + fw * a.g.dw;
              if (w < bb[u].w0 || w > bb[u].w1) continue;
              for (int fh = 0; fh < a.g.FH; ++fh) {
                const int h = hb + fh * a.g.dh;
                inside[u] |= (h >= bb[u].h0 && h <= bb[u].h1 ? 1u : 0u) << (fw * a.g.FH + fh);
              }
            }
          }
        }
      }
      // A stage's operands travel through registers while the two stages before it are multiplied.  Every load is issued
      // whatever its row and column are (what is not wanted is read from the centre and dropped on its way to LDS): behind a
      // branch the compiler could not tell the loads in flight apart and would wait for all of them.
      struct Regs {
        double2 a[A_PASS], b[B_PASS];
        unsigned use;  // bit u: a[u] is wanted; bits 16 + 2 u, 17 + 2 u: b[u].x, b[u].y are
      };
      auto load_tiles = [&](int k0, Regs& g) {
        g.use = 0;
#pragma unroll
        for (int u = 0; u < A_PASS; ++u) {
          const int idx = tid + u * NT;
          const int row = m0 + 2 * (idx % (TM / 2)), k = k0 + idx / (TM / 2);
          g.a[u] = *reinterpret_cast<const double2*>(a.Wk + row + (PIXELS ? s_tap[k] : (int64_t)s_tap[k] * a.coutp));
          if (!PIXELS) g.use |= s_row[k] >= 0 ? 1u << u : 0u;
        }
#pragma unroll
        for (int u = 0; u < B_PASS; ++u) {
          if (PIXELS) {
            const int2 word = *reinterpret_cast<const int2*>(at[u] + k0 + bk);
            auto element = [&](int x) { return in_global(inside[u] >> (x >> kPosBits) & 1u ? img[u] + (x & ((1 << kPosBits) - 1)) : g_zero)[0]; };
            g.b[u].x = element(word.x);
            g.b[u].y = element(word.y);
          } else {
            auto pixel = [&](int k, unsigned bit) {
              const int r = s_row[k], pos = s_pos[k];
              const int h = pos & 0xffff, w = pos >> 16;
              const bool in = r >= 0 && h >= bb[u].h0 && h <= bb[u].h1 && w >= bb[u].w0 && w <= bb[u].w1;
              g.use |= in ? bit : 0u;
              return in_global(in ? img[u] + r : S.V)[0];
            };
            g.b[u].x = pixel(k0 + bk, 1u << (16 + 2 * u));
            g.b[u].y = pixel(k0 + bk + 1, 1u << (17 + 2 * u));
          }
        }
      };
      auto store_tiles = [&](int buf, const Regs& g) {
#pragma unroll
        for (int u = 0; u < A_PASS; ++u) {
          const int idx = tid + u * NT;
          const bool on = PIXELS || (g.use >> u & 1);
          *reinterpret_cast<double2*>(&Ws[buf][(idx / (TM / 2)) * LDA_S + 2 * (idx % (TM / 2))]) =
              make_double2(on ? g.a[u].x : 0.0, on ? g.a[u].y : 0.0);
        }
#pragma unroll
        for (int u = 0; u < B_PASS; ++u) {
          const int j = (tid + u * NT) / (KT / 2);
          Vs[buf][j * LDB_S + bk] = PIXELS || (g.use >> (16 + 2 * u) & 1) ? g.b[u].x : 0.0;  // odd column stride: two 64-bit stores
          Vs[buf][j * LDB_S + bk + 1] = PIXELS || (g.use >> (17 + 2 * u) & 1) ? g.b[u].y : 0.0;
        }
      };
      double4_t acc[FM][FN];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
      // A wave without columns, and a stage of padding, leave the matrix cores to the other blocks: a part has 30 to 60 columns, and
      // half of its second tile is often empty.  64 channels: 74.6 -> 70.5 and 80.8 -> 75.3 us; with 32 a stage's four
      // instructions do not pay for the branch (22.0 -> 22.7).
      const bool some_col = c0 + wc * (TN / WC) < n;
      Regs g0, g1;
      load_tiles(0, g0);
      load_tiles(KT, g1);
      store_tiles(0, g0);
      __syncthreads();
      // stage t from LDS half t & 1; `next` holds stage t + 1, `far` receives stage t + 2 (past the end: the last again)
      auto step = [&](int t, Regs& next, Regs& far) {
        const int cur = t & 1;
        load_tiles(KT * min(t + 2, nk - 1), far);
        if (TM < 64 || (some_col && KT * t < nrow))
          mfma_tile_k16<FM, FN, KT>(&Ws[cur][wr * (TM / WR)], LDA_S, &Vs[cur][(wc * (TN / WC)) * LDB_S], LDB_S, lane, acc);
        store_tiles(cur ^ 1, next);
        __syncthreads();
      };
      for (int t = 0; t < nk; t += 2) {
        step(t, g1, g0);
        step(t + 1, g0, g1);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int co = m0 + wr * (TM / WR) + i * 16 + lrow;
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int c = c0 + wc * (TN / WC) + j * 16 + lcol + 4 * r;
            if (c >= n) continue;
            const int col = s_col[c];
            const double v = acc[i][j][r], pl = s_pl[c], pu = s_pu[c];
            // (the centre takes no part in the sums: an infinite one would leave 0 * Inf there)
            const double vp = col > 0 ? fmax(v, 0.0) : 0.0, vn = col > 0 ? fmin(v, 0.0) : 0.0;
            x[i][0] = fma(vp, pl, x[i][0]);
            x[i][1] = fma(vn, pu, x[i][1]);
            x[i][2] = fma(vp, pu, x[i][2]);
            x[i][3] = fma(vn, pl, x[i][3]);
            if (co < a.g.Cout) {
              if (col > 0 && S.out_pix != nullptr)
                S.out_pix[(int64_t)col * S.out_pix_ld + out_slot + co] = v;
              else
                S.out[(int64_t)col * a.ldo + (int64_t)co * a.g.P + p] = col == 0 && a.bias != nullptr ? v + bias[i] : v;
            }
          }
      }
    }
  }
  // the position's sums: lane groups, then the waves along the columns in order
  double* red = &Ws[0][0];
  static_assert(WC * TM * 4 <= 2 * KT * LDA_S, "the sums of the column waves fit the weight stages");
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      x[i][q] += __shfl_xor(x[i][q], 16);
      x[i][q] += __shfl_xor(x[i][q], 32);
      if (lcol == 0) red[((wc * TM) + wr * (TM / WR) + i * 16 + lrow) * 4 + q] = x[i][q];
    }
  }
  __syncthreads();
  double* dst = S.part + (int64_t)part * 4 * a.ldo;
  for (int t = tid; t < TM * 4; t += NT) {
    const int row = t >> 2, q = t & 3;
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < WC; ++w) s += red[(w * TM + row) * 4 + q];
    if (m0 + row < a.g.Cout) dst[q * a.ldo + (int64_t)(m0 + row) * a.g.P + p] = s;
  }
  // the padding rows behind the image
  if (p == 0 && m0 == 0) {
    const int pad = (int)(a.ldo - (int64_t)a.g.P * a.g.Cout);
    if (tid < 4 * pad) dst[(tid / pad) * a.ldo + (int64_t)a.g.P * a.g.Cout + tid % pad] = 0.0;
  }
}

// By position from about 2000 taps x channels on: below that a block's lists cost more than its product (72 taps into 16
// channels of 16 x 16, 3072 images: 42 us here, 36 us for the implicit GEMM over the windows with the scan behind it; 144 into
// 32, 25 sets of 784 images: 138 us here, 270 there).  The other limits are the tables': one thread of the sort per window start
// (1024 output positions, 32 x 32), the row list (1024 taps), the starts of a window (256 positions), 16-bit column numbers.
bool conv_window_takes(const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo, int64_t dense, int eh, int ew) {
  // (and finite weights: an infinite one times the zero of a reset row is NaN, and the rows left out count then)
  return cv->finite && cv->Wk != nullptr && cv->K * cv->Cout >= 2048 && Ho * Wo <= kSortBuckets && H * W * cv->Cin < (int64_t(1) << 31) && H < 32768 && W < 32768 &&
         cv->K <= kConvWinTaps && dense > 1 && dense - 1 <= kSortColumns && (int64_t)eh * ew <= kConvWinStarts;
}

static int conv_window_tile(const nnvhip_conv2d* cv) { return cv->Cout <= 16 ? 16 : cv->Cout <= 32 ? 32 : 64; }

int conv_window_parts(const nnvhip_conv2d* cv, int64_t Ho, int64_t Wo, int64_t dense, int eh, int ew) {
  // A set by itself: blocks that fill the 1024 places of four to a CU once, or, where positions are too many for that to come
  // out nearly even, twice; about one more a position writes stamps.  No part with less than a tile of columns, which is what
  // decides where a set has no more than some 1000 columns.  (15 x 15 positions, 288 taps into 64 channels: 4 parts 77.9 us, 5 -
  // 1360 blocks - 79.4, 8 - 2032 - 74.6, 12 85.0; 7 x 7 positions, 576 taps: 14 parts 90.0, 19 - 980 blocks - 81.6, 21 - 1088 -
  // 92.4, 32 92.8.)  Where "nearly even" lies: those 980 blocks are 0.96 of the places, and one round; three parts of the 15 x 15
  // would be 900, 0.88, and neither 4 nor 5 is as fast as two rounds.  All layers by position of other networks of four
  // convolutions, us, with 1024 blocks whatever they come out to -> with this -> with 768 places: 32 x 32 x 3 into 16, 16 channels
  // 67.6 -> 65.1 -> 71.8; 16, 32 84.5 -> 80.1 -> 83.1; 32, 48 150.5 -> 149.2 -> 164.0; 5 x 5 taps into 16, 48 133.8 -> 136.8 -> 136.2;
  // 28 x 28 x 3 into 24, 24 81.0 -> 75.3 -> 78.3; 24 x 24 x 3 into 16, 32 41.9 -> 39.4 -> 42.0; smaller ones within 2 % of one another
  // (16-channel tiles too do best with four blocks to a CU).  Arrays take the same parts set by set: 3 sets of 24 x 24 and 8 of
  // 28 x 28 are within 2 % in all three.
  const int64_t a_part = Ho * Wo * ceil_div(cv->Cout, conv_window_tile(cv)), places = 1024;
  int64_t want = (places - Ho * Wo) / a_part;
  if (want < 1 || (double)(want * a_part + Ho * Wo) < 0.93 * (double)places) want = std::max<int64_t>(want, (2 * places - Ho * Wo) / a_part);
  const double cols = (double)(dense - 1) * eh * ew / (double)(Ho * Wo);
  return (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(want, 32), (int64_t)(cols / 32.0)));
}

bool conv_window_takes_pixels(const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t eh, int64_t ew) {
  return cv->FH * cv->FW <= kNoPosition && H * W * cv->Cin < (int64_t(1) << kPosBits) && eh * ew * cv->Cin < (int64_t(1) << kPosBits) &&
         cv->K * cv->coutp < (int64_t(1) << 31);
}

template <bool PIXELS>
static int launch_windows(nnvhip_ctx* ctx, const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo, int64_t ldout, int64_t count,
                          const ConvWindowSet* sets) {
  if (count < 1) return NNVHIP_OK;
  if (count > 65535) NNV_FAIL(NNVHIP_ERR_SHAPE, "at most 65535 sets per call");
  ConvWinArgs a{};
  a.Wk = cv->Wk->as<double>();
  a.bias = cv->bias ? cv->bias->as<double>() : nullptr;
  a.ldo = ldout;
  a.Wt = cv->W->as<double>();
  a.coutp = (int32_t)cv->coutp;
  fill_geom(a.g, cv, H, W, Ho, Wo);
  a.list = (int32_t)round_up(cv->K, 32) + 32;
  int64_t max_parts = 1;
  std::vector<ConvWinSet> tab((size_t)count);
  double flop = 0.0;
  for (int64_t i = 0; i < count; ++i) {
    const ConvWindowSet& s = sets[i];
    tab[(size_t)i] = ConvWinSet{s.in->V, s.in->ld, s.in->box, s.out->box, s.in->rows_pending ? s.in->keep_bits : nullptr,
                                s.in->rows_pending ? s.in->cls : nullptr, s.order, s.first, s.out->V, s.out->plb, s.out->pub, s.part,
                                (int32_t)s.parts, s.eh, s.ew, nullptr, nullptr, 0, 0, 1, 1, 1, 1, StampSet{}};
    ConvWinSet& t = tab[(size_t)i];
    if (PIXELS) {
      t.in_pix = s.in->cs.pix;
      t.in_pix_ld = s.in->cs.pix_ld;
      t.in_eh = s.in->cs.pix_eh;
      t.in_ew = s.in->cs.pix_ew;
    }
    if (s.out->cs.in_pixels()) {
      t.out_pix = const_cast<double*>(s.out->cs.pix);
      t.out_pix_ld = s.out->cs.pix_ld;
      t.out_eh = s.out->cs.pix_eh;
      t.out_ew = s.out->cs.pix_ew;
    }
    if (s.stamp != nullptr) {
      static_assert(sizeof(ConvStampSet) == sizeof(StampSet), "same layout");
      memcpy(&tab[(size_t)i].stamps, s.stamp, sizeof(StampSet));
    }
    max_parts = std::max<int64_t>(max_parts, s.parts);
    ++ctx->routes[NNVHIP_ROUTE_CONV_WINDOW];
    if (s.parts > 1) ++ctx->routes[NNVHIP_ROUTE_CONV_WINDOW_PARTS];
    // (rows a ReLU step has reset are not multiplied; their share under a filter is taken to be that of the image)
    const double kept = s.in->rows_pending && s.in->n_kept >= 0 ? (double)s.in->n_kept / (double)s.in->N : 1.0;
    flop += 2.0 * ((double)(s.dense - 1) * s.eh * s.ew + (double)a.g.P) * (double)cv->Cout * (double)cv->K * kept;
  }
  const ConvWinSet* table = nullptr;
  BufRef dev;
  if (count > 1) {
    NNV_TRY(ctx->upload_table(tab.data(), sizeof(ConvWinSet) * tab.size(), &dev));
    table = dev->as<ConvWinSet>();
  }
  a.per = (int32_t)ceil_div(a.g.P * max_parts, 8);
  const int tm = conv_window_tile(cv);
  const int nt = tm == 16 ? 128 : 256;
  const bool wide_stamps = a.g.K > 32;  // lanes per output row as in the launch that shares the implicit GEMM's
  int64_t stamp_blocks = 0;
  for (int64_t i = 0; i < count; ++i)
    if (sets[i].stamp != nullptr)
      stamp_blocks = std::max<int64_t>(stamp_blocks, sets[i].stamp->pix != nullptr ? conv_stamp_pixel_blocks(a.g.P, a.g.K, nt)
                                                                                     : ceil_div(ldout * (wide_stamps ? 8 : 1), nt));
  a.stamp_blocks = (int32_t)round_up(stamp_blocks, 8);
  const dim3 grid((unsigned)(a.stamp_blocks + 8 * a.per), (unsigned)count, (unsigned)ceil_div(cv->Cout, tm));
  // (also holds the stamps' tap table, 8 bytes a tap, or a wave's 64 columns each)
  const size_t dyn = std::max(3 * sizeof(int32_t) * (size_t)a.list, sizeof(int2) * (size_t)nt);
  NNV_TRY(ctx->kernel_timer_begin(ctx->kernel_timing));
#define NNV_CONV_WINDOW(TM, WR, WC)                                                                                                    \
  do {                                                                                                                                \
    if (wide_stamps)                                                                                                                  \
      NNV_LAUNCH(ctx, ctx->kernel_timing, (conv_window_kernel<TM, 32, WR, WC, 8, PIXELS>), grid, dim3(64 * WR * WC), dyn, table, tab[0], a);  \
    else                                                                                                                              \
      NNV_LAUNCH(ctx, ctx->kernel_timing, (conv_window_kernel<TM, 32, WR, WC, 1, PIXELS>), grid, dim3(64 * WR * WC), dyn, table, tab[0], a);  \
  } while (0)
  if (tm == 16)
    NNV_CONV_WINDOW(16, 1, 2);
  else if (tm == 32)
    NNV_CONV_WINDOW(32, 2, 2);
  else
    NNV_CONV_WINDOW(64, 2, 2);
#undef NNV_CONV_WINDOW
  NNV_TRY(ctx->kernel_timer_end(ctx->kernel_timing, 12, flop));
  NNV_HIP_TRY(hipGetLastError());
  return NNVHIP_OK;
}

int launch_conv_window(nnvhip_ctx* ctx, const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo, int64_t ldout, int64_t count,
                       const ConvWindowSet* sets) {
  std::vector<ConvWindowSet> columns, pixels;
  for (int64_t i = 0; i < count; ++i) (sets[i].in->cs.in_pixels() ? pixels : columns).push_back(sets[i]);
  NNV_TRY(launch_windows<false>(ctx, cv, H, W, Ho, Wo, ldout, (int64_t)columns.size(), columns.data()));
  return launch_windows<true>(ctx, cv, H, W, Ho, Wo, ldout, (int64_t)pixels.size(), pixels.data());
}

}  // namespace nnvhip
