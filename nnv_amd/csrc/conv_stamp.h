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

// The same into columns that are kept pixel by pixel: neighbouring threads take the channels of one output position, whose
// elements of a column lie side by side there, and a tap's pixel, column and scale are the same for all of them.  Weights tap by
// tap with their channels side by side (Wk).
template <int S, int NT>
__device__ __forceinline__ void conv_stamp_pixels_block(int64_t blk, int2* taps, const StampSet& d, const ConvGeom& g,
                                                        const double* __restrict__ Wk, int coutp, const int32_t* __restrict__ pixel_col,
                                                        int64_t ldout) {
  for (int k = threadIdx.x; k < g.K; k += NT) {
    const int fh = k % g.FH;
    const int q = k / g.FH;
    const int fw = q % g.FW;
    const int ci = q / g.FW;
    taps[k] = make_int2(fh | (fw << 16), fh + g.H * (fw + g.W * ci));
  }
  __syncthreads();
  const int64_t gt = blk * (int64_t)NT + threadIdx.x;
  const int64_t q = gt / S;
  const int s = (int)(gt % S);
  const bool inside = q < (int64_t)g.P * g.Cout;
  const int p = inside ? (int)(q / g.Cout) : 0, co = inside ? (int)(q - (int64_t)p * g.Cout) : 0;
  double x1 = 0.0, x2 = 0.0, y1 = 0.0, y2 = 0.0;
  if (inside) {
    const int wo = p / g.Ho, ho = p - wo * g.Ho;
    const int hb = ho * g.sh - g.pt, wb = wo * g.sw - g.pl;
    const int pbase = hb + g.H * wb;
    double* const at = d.pix + (int64_t)pix_slot(ho, wo, d.pix_eh, d.pix_ew) * g.Cout + co;
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
      double v[4], pl[4], pu[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const bool on = t[u] >= 0;
        const double sc = !on ? 0.0 : d.scale != nullptr ? d.scale[pix[u]] : 1.0;
        v[u] = on ? __dadd_rn(0.0, __dmul_rn(Wk[(int64_t)(k0 + u * S) * coutp + co], sc)) : 0.0;
        pl[u] = on ? d.plb[t[u]] : 0.0;
        pu[u] = on ? d.pub[t[u]] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (t[u] < 0) continue;
        at[(int64_t)t[u] * d.pix_ld] = v[u];
        const double vp = fmax(v[u], 0.0), vn = fmin(v[u], 0.0);
        x1 = fma(vp, pl[u], x1);  // xmin1
        x2 = fma(vn, pu[u], x2);  // xmin2
        y1 = fma(vp, pu[u], y1);  // xmax1
        y2 = fma(vn, pl[u], y2);  // xmax2
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
  if (q < ldout && s == 0) {  // (behind the image: the padding rows)
    const int64_t r = inside ? (int64_t)co * g.P + p : q;
    d.part[r] = x1;
    d.part[ldout + r] = x2;
    d.part[2 * ldout + r] = y1;
    d.part[3 * ldout + r] = y2;
  }
}

void fill_geom(ConvGeom& g, const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo);

}  // namespace nnvhip
