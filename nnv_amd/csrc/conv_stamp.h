// The stamps of a convolution's unit-vector columns, by output row: a block function that the kernels of conv.hip and
// conv_window.hip share, each next to its own tiles.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.h"

namespace nnvhip {

struct ConvGeom {
  int H, W, Cin, Ho, Wo, Cout;
  int FH, FW, sh, sw, dh, dw, pt, pl;
  int K, Kp;
  int P;   // Ho * Wo
  int HW;  // H * W
};

constexpr int kMaxTaps = 4096;  // tap table held in LDS: 8 bytes per (padded) tap

struct StampSet {
  const int32_t* idx;   // input row of every one-hot column
  const double* scale;  // by input row, or null (= 1)
  double* out;          // first of these columns in the output set
  const double* plb;    // predicate bounds of these columns
  const double* pub;
  double* part;         // [chunks][4][ldout] range sums of these columns (as the estimateRanges pass leaves them)
  int32_t m;
  int32_t win_only;     // 1: only the rows inside a column's window (the positions whose taps span its pixel) are written
  const int32_t* pixel_col;  // (by-row pass) input row -> its column here, -1: none
  double* pix;          // (by-row pass) not null: the elements go here, pixel by pixel (ColSource::pix) ...
  int64_t pix_ld;
  int32_t pix_eh, pix_ew;
};

// ---- the stamps by output row (undilated filters) ---------------------------------------------------
// Row r = (ho, wo, co) of the output meets the stamps of the pixels under its filter window, one per tap: for
// tap k = (fh, fw, ci) the pixel (ho*sh - pt + fh, wo*sw - pl + fw, ci), whose unit-vector column t (pixel_col,
// -1: none) gets out(r, t) = 0 + W(k, co) * scale.  One thread per row writes those elements - exactly the
// non-zero candidates, i.e. the rows inside every column's window - and adds up the row's four range sums tap
// by tap.  Everything else in the columns is zero and is written by the caller (or left for later).
// S lanes share a row, lane s taking the taps k = s, s + S, ...; their sums are combined by a butterfly (a fixed
// order).  S is the caller's choice: 1 for at most 32 taps; for more, 8 beside the products of another kernel's blocks and
// 16 in the launch that does nothing else.
// A block first decodes the taps once into LDS (filter position and the tap's offset from the pixel under the
// filter's corner), so that the walk has no division in it, and looks up four taps' pixels before it handles them.
constexpr int kStampTapTable = kMaxTaps;  // taps per output (FH * FW * Cin): no layer has more
// Block `blk` of NT threads; taps: LDS for g.K entries.
template <int S, int NT>
__device__ __forceinline__ void conv_stamp_rows_block(int64_t blk, int2* taps, const StampSet& d, const ConvGeom& g,
                                                      const double* __restrict__ Wt, const int32_t* __restrict__ pixel_col,
                                                      int64_t ldout) {
  for (int k = threadIdx.x; k < g.K; k += NT) {
    const int fh = k % g.FH;
    const int q = k / g.FH;
    const int fw = q % g.FW;
    const int ci = q / g.FW;
    taps[k] = make_int2(fh | (fw << 16), fh + g.H * (fw + g.W * ci));  // x: fh | fw << 16, y: fh + H * (fw + W * ci)
  }
  __syncthreads();
  const int64_t gt = blk * (int64_t)NT + threadIdx.x;
  const int64_t r = gt / S;
  const int s = (int)(gt % S);
  const bool row = r < ldout;
  const int64_t Nout = (int64_t)g.P * g.Cout;
  double x1 = 0.0, x2 = 0.0, y1 = 0.0, y2 = 0.0;
  if (row && r < Nout) {
    const int co = (int)(r / g.P);
    const int p = (int)(r - (int64_t)co * g.P);
    const int wo = p / g.Ho, ho = p - wo * g.Ho;
    const int hb = ho * g.sh - g.pt, wb = wo * g.sw - g.pl;
    const int pbase = hb + g.H * wb;  // the pixel under the filter's corner (may lie outside the image)
    const double* wcol = Wt + (int64_t)co * g.Kp;
    for (int k0 = s; k0 < g.K; k0 += 4 * S) {
      int t[4], pix[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k0 + u * S;
        t[u] = -1;
        pix[u] = 0;
        if (k < g.K) {
          const int2 tp = taps[k];
          const int h = hb + (tp.x & 0xffff), w = wb + (tp.x >> 16);
          if ((unsigned)h < (unsigned)g.H && (unsigned)w < (unsigned)g.W) {
            pix[u] = pbase + tp.y;
            t[u] = pixel_col[pix[u]];
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (t[u] < 0) continue;
        const int k = k0 + u * S;
        const double sc = d.scale != nullptr ? d.scale[pix[u]] : 1.0;
        const double v = __dadd_rn(0.0, __dmul_rn(wcol[k], sc));
        d.out[r + (int64_t)t[u] * ldout] = v;
        const double pl = d.plb[t[u]], pu = d.pub[t[u]];
        const double vp = fmax(v, 0.0), vn = fmin(v, 0.0);
        x1 = fma(vp, pl, x1);  // xmin1
        x2 = fma(vn, pu, x2);  // xmin2
        y1 = fma(vp, pu, y1);  // xmax1
        y2 = fma(vn, pl, y2);  // xmax2
      }
    }
  }
#pragma unroll
  for (int off = 1; off < S; off <<= 1) {
    x1 += __shfl_xor(x1, off);
    x2 += __shfl_xor(x2, off);
    y1 += __shfl_xor(y1, off);
    y2 += __shfl_xor(y2, off);
  }
  if (row && s == 0) {
    d.part[r] = x1;
    d.part[ldout + r] = x2;
    d.part[2 * ldout + r] = y1;
    d.part[3 * ldout + r] = y2;
  }
}

// The same into columns that are kept pixel by pixel, by output position: the columns whose pixel lies under the filter are
// listed once for all channels (by rows every channel looks all taps up again), then the position's threads share out channels
// and listed columns, a column's channels side by side as they lie there.  Weights tap by tap with their channels side by side
// (Wk).  Filters of up to 64 taps: a wave to a position; others: the block.  Row sums: a thread's columns in tap order, then
// lanes, then waves, in a fixed order.  Launches with their products, by rows -> by position: 32 x 32 x 3 network 23, 22, 85, 91
// -> 14, 22, 78, 83 us; 28 x 28, first layer 11 -> 7, 25 of them 25 -> 30, second layer of those 108 -> 86.
constexpr int kStampPixelTaps = 1024;  // taps per output at most
inline int64_t conv_stamp_pixel_blocks(int64_t positions, int64_t taps, int threads) {
  return taps <= 64 ? (positions + threads / 64 - 1) / (threads / 64) : positions;
}
// LDS: red: NT / 64 * 256 doubles, cnt: NT / 64 numbers, list: max(g.K, NT) entries.
template <int NT>
__device__ __forceinline__ void conv_stamp_pixels_block(int64_t blk, double* red, int* cnt, int2* list, const StampSet& d, const ConvGeom& g,
                                                        const double* __restrict__ Wk, int coutp, const int32_t* __restrict__ pixel_col,
                                                        int64_t ldout) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int per = g.K <= 64 ? 1 : NW;  // waves of a position
  const int team = wave / per, member = wave - team * per;
  const int64_t p = blk * (NW / per) + team;
  if (blk * (NW / per) >= g.P) return;  // (the whole block)
  const bool real = p < g.P;
  const int wo = real ? (int)(p / g.Ho) : 0, ho = real ? (int)(p - (int64_t)wo * g.Ho) : 0;
  const int hb = ho * g.sh - g.pt, wb = wo * g.sw - g.pl;
  int2* const mine = list + team * 64;  // (a block with one position: team 0)
  int n = 0;
  for (int k0 = 0; k0 < g.K; k0 += per * 64) {
    const int k = k0 + member * 64 + lane;
    int t = -1;
    if (real && k < g.K) {
      const int q = k / g.FH, ci = q / g.FW;
      const int h = hb + k - q * g.FH, w = wb + q - ci * g.FW;
      if ((unsigned)h < (unsigned)g.H && (unsigned)w < (unsigned)g.W) t = pixel_col[h + g.H * (w + g.W * ci)];
    }
    const unsigned long long m = __ballot(t >= 0);
    if (lane == 0) cnt[wave] = __popcll(m);
    __syncthreads();
    int before = n;
    for (int v = 0; v < per; ++v) {
      const int c = cnt[team * per + v];
      before += v < member ? c : 0;
      n += c;
    }
    if (t >= 0) mine[before + __popcll(m & ((1ull << lane) - 1ull))] = make_int2(t, k);
    __syncthreads();
  }
  const int CL = g.Cout <= 16 ? 16 : g.Cout <= 32 ? 32 : 64;  // lanes along the channels
  const int groups = per * (64 / CL), group = member * (64 / CL) + lane / CL;
  double* const at = d.pix + (int64_t)pix_slot(ho, wo, d.pix_eh, d.pix_ew) * g.Cout;
  for (int co0 = 0; co0 < g.Cout; co0 += CL) {
    const int co = co0 + lane % CL;
    const bool on = co < g.Cout;
    double x[4] = {0.0, 0.0, 0.0, 0.0};  // xmin1, xmin2, xmax1, xmax2
    for (int e0 = group; e0 < n; e0 += 4 * groups) {  // four columns' look-ups in flight
      int2 te[4];
      double v[4], pl[4], pu[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) te[u] = mine[min(e0 + u * groups, n - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double sc = d.scale != nullptr ? d.scale[d.idx[te[u].x]] : 1.0;
        v[u] = __dadd_rn(0.0, __dmul_rn(on ? Wk[(int64_t)te[u].y * coutp + co] : 0.0, sc));
        pl[u] = d.plb[te[u].x];
        pu[u] = d.pub[te[u].x];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (e0 + u * groups >= n) break;
        if (on) at[(int64_t)te[u].x * d.pix_ld + co] = v[u];
        const double vp = fmax(v[u], 0.0), vn = fmin(v[u], 0.0);
        x[0] = fma(vp, pl[u], x[0]);
        x[1] = fma(vn, pu[u], x[1]);
        x[2] = fma(vp, pu[u], x[2]);
        x[3] = fma(vn, pl[u], x[3]);
      }
    }
#pragma unroll
    for (int off = 16; off < 64; off <<= 1)
      if (off >= CL) {
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] += __shfl_xor(x[q], off);
      }
    if (per == 1) {
      if (real && on && lane < CL) {
#pragma unroll
        for (int q = 0; q < 4; ++q) d.part[q * ldout + (int64_t)co * g.P + p] = x[q];
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) red[(wave * 4 + q) * 64 + lane] = x[q];
      __syncthreads();
      if (member < 4 && on && lane < CL) {
        for (int q = member; q < 4; q += per) {
          double s = 0.0;
          for (int w = 0; w < per; ++w) s += red[(w * 4 + q) * 64 + lane];
          d.part[q * ldout + (int64_t)co * g.P + p] = s;
        }
      }
      __syncthreads();
    }
  }
  if (blk == 0)  // the padding rows behind the image
    for (int64_t r = (int64_t)g.P * g.Cout + threadIdx.x; r < ldout; r += NT)
      d.part[r] = d.part[ldout + r] = d.part[2 * ldout + r] = d.part[3 * ldout + r] = 0.0;
}

void fill_geom(ConvGeom& g, const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo);

}  // namespace nnvhip
