// affineMap of a Conv2DLayer on an ImageStar (nn/layers/Conv2DLayer.m:559-601): the same
// cross-correlation applied to the centre image (plus bias) and to every generator image.
//
// Implicit GEMM on fp64 MFMA.  With P = Ho*Wo output positions per image and G = n+1 images the
// output, in MATLAB's H x W x C x (n+1) layout, is a (P*G) x Cout matrix whose rows are contiguous in
// memory per (channel, image); the reduction runs over the K = FH*FW*Cin filter taps, which is
// exactly the row order of MATLAB's FH x FW x Cin x Cout weight array.  The im2col operand is never
// materialised: each block gathers its 128-position x 16-tap tile straight from the input images
// (zero for padding taps) into LDS; the weight tile is loaded like the generator tile of the dense
// GEMM.  MFMA operand "b" carries positions (the memory-contiguous direction of the output), "a"
// carries output channels.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "conv_stamp.h"
#include "internal.h"
#include "lds_dma.h"
#include "mfma_tile.h"
#include "relu_sort.h"
#include "window_sort.h"

namespace nnvhip {

constexpr size_t kConvLdsLimit = 64 * 1024;  // LDS of one block: operand tiles + tap table + row mask

// Tap k = fh + FH*(fw + FW*ci) -> packed (input offset ci*H*W : 32 | fh*dh : 16 | fw*dw : 16).
__device__ __forceinline__ unsigned long long pack_tap(const ConvGeom& g, int k) {
  if (k >= g.K) return ~0ull;  // padded tap: never valid
  const int fh = k % g.FH;
  const int t = k / g.FH;
  const int fw = t % g.FW;
  const int ci = t / g.FW;
  return ((unsigned long long)(unsigned)(ci * g.HW) << 32) | ((unsigned long long)(fh * g.dh) << 16) |
         (unsigned long long)(fw * g.dw);
}

// How the rows of the implicit GEMM map to (image, output position).  box == null: row R is position R % P of
// image R / P.  Otherwise rows [0, P) are the centre image and every further image owns `area` = eh x ew rows,
// the positions of its window's corner onwards (row t of the slot: ho = h0 + t % eh, wo = w0 + t / eh; slots of
// positions outside the window are idle): a generator image is computed inside its window only.
struct ConvRows {
  const ColBox* box;
  int eh, area;
  const ColBox* in_box;  // windows of the input images, or null: a tap outside its image's window is not read
};

template <bool COMPACT>
__device__ __forceinline__ bool conv_row(const ConvGeom& g, const ConvRows& cr, int64_t R, int64_t total_rows, int64_t* gi,
                                         int* ho, int* wo) {
  if (R >= total_rows) return false;
  if (!COMPACT || R < g.P) {
    const int64_t im = COMPACT ? 0 : R / g.P;
    const int p = (int)(R - im * g.P);
    *gi = im;
    *wo = p / g.Ho;
    *ho = p - *wo * g.Ho;
    return true;
  }
  const int64_t q = R - g.P;
  const int64_t im = q / cr.area;
  const int t = (int)(q - im * cr.area);
  const ColBox bb = cr.box[1 + im];
  *gi = 1 + im;
  const int tw = t / cr.eh;
  *ho = bb.h0 + (t - tw * cr.eh);
  *wo = bb.w0 + tw;
  return *ho <= bb.h1 && *wo <= bb.w1;
}

template <bool COMPACT>
__device__ __forceinline__ int64_t conv_first_image(const ConvGeom& g, const ConvRows& cr, int64_t R0) {
  if (!COMPACT) return R0 / g.P;
  return R0 < g.P ? 0 : 1 + (R0 - g.P) / cr.area;
}

// Stores a block's accumulators: lane l, register r of acc[i][j] holds out[row R0 + ... + l%16][channel c0 +
// ... + l/16 + 4r]; the bias goes onto the centre image only.
template <int TP, int TC, int WR, int WC, int FM, int FN, bool COMPACT = false>
__device__ __forceinline__ void conv_store_tile(const double4_t (&acc)[FM][FN], double* __restrict__ out, int64_t ldout,
                                                const double* __restrict__ bias, const ConvGeom& g, int64_t total_rows,
                                                int64_t R0, int c0, int wr, int wc, int lane,
                                                const ConvRows cr = ConvRows{nullptr, 0, 0, nullptr}) {
  const int lrow = lane & 15;
  const int lcol = lane >> 4;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int64_t Rr = R0 + wr * (TP / WR) + i * 16 + lrow;
    int64_t gi;
    int ho, wo;
    if (!conv_row<COMPACT>(g, cr, Rr, total_rows, &gi, &ho, &wo)) continue;
    const int p = ho + wo * g.Ho;
    double* o = out + gi * ldout + p;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int co = c0 + wc * (TC / WC) + j * 16 + lcol + 4 * r;
        if (co < g.Cout) {
          double v = acc[i][j][r];
          if (bias != nullptr && gi == 0) v = v + bias[co];  // centre image only
          o[(int64_t)co * g.P] = v;
        }
      }
    }
  }
}

// MASK: the input is the matrix in front of a ReLU step whose row reset has not been run; `keep` holds one
// bit per input row (1 = the row is kept, 0 = it reads as zero: PosLin.m:700-709, Star.m:1442-1461), copied
// into LDS behind the tap table.  A reset row is never loaded.
template <int TP, int TC, int WR, int WC, bool MASK>
__global__ __launch_bounds__(64 * WR * WC) void conv2d_f64_kernel(const double* __restrict__ in, int64_t ldin,
                                                          double* __restrict__ out, int64_t ldout,
                                                          const double* __restrict__ Wt,
                                                          const double* __restrict__ bias, ConvGeom g,
                                                          int64_t total_rows, int tiles_c,
                                                          const uint32_t* __restrict__ keep, int keep_words) {
  constexpr int NT = 64 * WR * WC;  // threads per block
  static_assert(NT % TP == 0 && (TP * kKt) % NT == 0, "gather mapping needs NT = TP * (taps per pass)");
  constexpr int FM = TP / WR / 16;
  constexpr int FN = TC / WC / 16;
  constexpr int LDP_S = TP + kPadRow;  // Ps[k][position]
  constexpr int LDW_S = kKt + kPadK;   // Wts[cout][k]
  __shared__ double Ps[2][kKt * LDP_S];
  __shared__ double Wts[2][TC * LDW_S];
  extern __shared__ unsigned long long taps[];  // Kp entries

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wr = wave % WR;
  const int wc = wave / WR;
  const int64_t bid = blockIdx.x;
  const int c0 = (int)(bid % tiles_c) * TC;
  const int64_t R0 = (bid / tiles_c) * TP;

  for (int k = tid; k < g.Kp; k += NT) taps[k] = pack_tap(g, k);
  uint32_t* keep_s = reinterpret_cast<uint32_t*>(taps + g.Kp);
  if (MASK)
    for (int k = tid; k < keep_words; k += NT) keep_s[k] = keep[k];

  // this thread's gather position (fixed for the whole K loop)
  constexpr int P_PASS = TP * kKt / NT;  // gathered elements per thread per K-tile
  constexpr int K_STEP = NT / TP;        // taps covered by one pass
  const int p_local = tid % TP;
  const int k_first = tid / TP;
  const int64_t R = R0 + p_local;
  const bool rvalid = R < total_rows;
  int h0 = 0, w0 = 0;
  const double* img = in;
  if (rvalid) {
    const int64_t gi = R / g.P;
    const int p = (int)(R - gi * g.P);
    const int wo = p / g.Ho;
    const int ho = p - wo * g.Ho;
    h0 = ho * g.sh - g.pt;
    w0 = wo * g.sw - g.pl;
    img = in + gi * ldin;
  }

  constexpr int W_VEC = TC * kKt / 2;
  constexpr int W_PASS = (W_VEC + NT - 1) / NT;
  double rp[P_PASS];
  double2 rw[W_PASS];

  auto load_tiles = [&](int k0) {
#pragma unroll
    for (int q = 0; q < P_PASS; ++q) {
      const unsigned long long t = taps[k0 + k_first + q * K_STEP];
      const int h = h0 + (int)((t >> 16) & 0xffffu);
      const int w = w0 + (int)(t & 0xffffu);
      bool ok = rvalid && t != ~0ull && (unsigned)h < (unsigned)g.H && (unsigned)w < (unsigned)g.W;
      const int row = ok ? (int)(unsigned)(t >> 32) + h + w * g.H : 0;  // row of the input set (< 2^31)
      if (MASK) ok = ok && ((keep_s[row >> 5] >> (row & 31)) & 1u) != 0;
      rp[q] = ok ? img[row] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < W_PASS; ++q) {
      const int idx = tid + q * NT;
      const int k2 = idx % (kKt / 2);
      const int j = idx / (kKt / 2);
      double2 v = make_double2(0.0, 0.0);
      if (idx < W_VEC && c0 + j < g.Cout) v = *reinterpret_cast<const double2*>(Wt + (k0 + 2 * k2) + (int64_t)(c0 + j) * g.Kp);
      rw[q] = v;
    }
  };
  auto store_tiles = [&](int buf) {
#pragma unroll
    for (int q = 0; q < P_PASS; ++q) Ps[buf][(k_first + q * K_STEP) * LDP_S + p_local] = rp[q];
#pragma unroll
    for (int q = 0; q < W_PASS; ++q) {
      const int idx = tid + q * NT;
      const int k2 = idx % (kKt / 2);
      const int j = idx / (kKt / 2);
      if (idx < W_VEC) {  // odd column stride: two 64-bit stores
        Wts[buf][j * LDW_S + 2 * k2] = rw[q].x;
        Wts[buf][j * LDW_S + 2 * k2 + 1] = rw[q].y;
      }
    }
  };

  double4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};

  __syncthreads();  // tap table ready
  const int nk = g.Kp / kKt;
  load_tiles(0);
  store_tiles(0);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) load_tiles((kt + 1) * kKt);
    mfma_tile_k16<FM, FN>(&Ps[cur][wr * (TP / WR)], LDP_S, &Wts[cur][(wc * (TC / WC)) * LDW_S], LDW_S, lane, acc);
    if (kt + 1 < nk) store_tiles(cur ^ 1);
    __syncthreads();
  }

  conv_store_tile<TP, TC, WR, WC, FM, FN>(acc, out, ldout, bias, g, total_rows, R0, c0, wr, wc, lane);
}

// ---- the same convolution with little vector-ALU work per MFMA ------------------------------------
// On this chip the vector ALU does not issue in the shadow of an fp64 MFMA (measured: every extra VALU
// instruction of a wave costs about as many matrix-pipe cycles as it takes to issue), so the gather of the
// kernel above - tap decode, bounds checks, a 32-bit multiply and 64-bit address arithmetic per element -
// costs a third of the MFMA time.  Here a tap is a wave-uniform (row offset, spatial bit) pair read through
// the scalar unit from a table in global memory, a thread's padding pattern is one 32-bit mask computed once
// (bit fh + FH*fw: that tap falls inside the image), the element's row is one addition, and its address a
// 32-bit offset from a block-uniform base.  The weight tile comes k-major from a second copy of the weights
// straight into LDS (global_load_lds_dwordx4), with no registers or address arithmetic in between.
// Needs FH*FW <= 32 and a tile's images within 2 GiB of its first one; the host checks both.
struct FastTap {
  int32_t off;   // ci*H*W + fh*dh + fw*dw*H: row of the tap relative to the row of tap (0, 0, 0)
  uint32_t bit;  // 1 << (fh + FH*fw); 0 for a padding entry
};

__global__ void conv_fast_taps_kernel(FastTap* __restrict__ tab, ConvGeom g) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= g.Kp) return;
  FastTap t{0, 0u};
  if (k < g.K) {
    const int fh = k % g.FH;
    const int r = k / g.FH;
    const int fw = r % g.FW;
    const int ci = r / g.FW;
    t.off = ci * g.HW + fh * g.dh + fw * g.dw * g.H;
    t.bit = 1u << (fh + g.FH * fw);
  }
  tab[k] = t;
}

// Wk(k, co) = W(k, co) for co < Cout, zero up to coutp: the weights k-major (row k contiguous over channels)
__global__ void conv_weights_kmajor_kernel(const double* __restrict__ W, double* __restrict__ Wk, int Kp, int Cout, int coutp) {
  const int64_t idx = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (idx >= (int64_t)Kp * coutp) return;
  const int k = (int)(idx / coutp), co = (int)(idx % coutp);
  Wk[idx] = co < Cout ? W[k + (int64_t)co * Kp] : 0.0;
}

struct ConvFastArgs {  // the layer
  int64_t ldout;
  const double* Wk;
  int coutp;
  const double* bias;
  ConvGeom g;
  int tiles_c;
  const FastTap* taps;
  int keep_words;
  int stamp_blocks;  // blocks for a set's unit-vector columns, dealt in between its tile blocks (0: none)
};

// One set of a call.  All sets of an array go into one launch (blockIdx.y = set): a convolution of one image's generators
// has a few dozen to a few hundred blocks, and a launch per image left the chip three quarters idle and the host behind
// (25 images of 28x28x1 through 3x3 filters to 16 and to 32 channels: 150 launches, 25 x 18 + 25 x 20 us of kernels plus
// the gaps; now six launches, 68 + 125 us).
struct ConvSet {
  const double* in;
  double* out;
  int64_t ldin;
  int64_t total_rows;
  const uint32_t* keep;
  ConvRows cr;
  int32_t blocks;  // tile blocks
  int32_t stride;  // grid position p is stamp block (p + 1) / stride - 1 where (p + 1) % stride == 0 (and that is < stamp_blocks)
  StampSet d;      // unit-vector columns whose stamps go into the same launch
};

// LDS of a block of the kernel below: the weight tiles [2][k][channel] first (their transfers want 1 KiB alignment),
// then the position tiles [2][k][position]; the row mask (MASK only) sits in the dynamic part behind them.
constexpr size_t conv_fast_lds_bytes(int tc) { return sizeof(double) * 2 * kKt * (128 + (size_t)tc); }

// This block's set.  Field by field: a copy of the whole record is made through a generic pointer, which leaves the fields in
// vector registers.
__device__ __forceinline__ ConvSet conv_set_of_block(const ConvSet* __restrict__ table, const ConvSet& one) {
  if (table == nullptr) return one;
  const ConvSet* __restrict__ t = table + blockIdx.y;
  ConvSet s;
  s.in = t->in;
  s.out = t->out;
  s.ldin = t->ldin;
  s.total_rows = t->total_rows;
  s.keep = t->keep;
  s.cr.box = t->cr.box;
  s.cr.eh = t->cr.eh;
  s.cr.area = t->cr.area;
  s.cr.in_box = t->cr.in_box;
  s.blocks = t->blocks;
  s.stride = t->stride;
  s.d.idx = t->d.idx;
  s.d.scale = t->d.scale;
  s.d.out = t->d.out;
  s.d.plb = t->d.plb;
  s.d.pub = t->d.pub;
  s.d.part = t->d.part;
  s.d.m = t->d.m;
  s.d.win_only = t->d.win_only;
  s.d.pixel_col = t->d.pixel_col;
  s.d.pix = t->d.pix;
  s.d.pix_ld = t->d.pix_ld;
  s.d.pix_eh = t->d.pix_eh;
  s.d.pix_ew = t->d.pix_ew;
  return s;
}

template <int TC, int WR, int WC, bool MASK, bool COMPACT>
__device__ __forceinline__ void conv2d_fast_block(const ConvFastArgs& a, const ConvSet& set, int64_t bid, double* __restrict__ lds,
                                                  uint32_t* keep_s) {
  constexpr int TP = 128, NT = 512;
  static_assert(WR * WC == 8, "eight waves");
  constexpr int FM = TP / WR / 16;
  constexpr int FN = TC / WC / 16;
  constexpr int kWLoads = kKt * TC / 128;  // 1 KiB wave transfers per K-tile of weights
  constexpr int kRowsPerLoad = 128 / TC;   // rows of Wk per transfer
  double(*Wts)[kKt * TC] = reinterpret_cast<double(*)[kKt * TC]>(lds);                // [k][channel]
  double(*Ps)[kKt * TP] = reinterpret_cast<double(*)[kKt * TP]>(lds + 2 * kKt * TC);  // [k][position]
  const double* __restrict__ in = set.in;
  const int64_t ldin = set.ldin;
  double* __restrict__ out = set.out;
  const int64_t ldout = a.ldout;
  const double* __restrict__ Wk = a.Wk;
  const int coutp = a.coutp;
  const double* __restrict__ bias = a.bias;
  const ConvGeom& g = a.g;
  const int64_t total_rows = set.total_rows;
  const int tiles_c = a.tiles_c;
  const FastTap* __restrict__ taps = a.taps;
  const uint32_t* __restrict__ keep = set.keep;
  const int keep_words = a.keep_words;
  const ConvRows& cr = set.cr;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave % WR;
  const int wc = wave / WR;
  const int c0 = (int)(bid % tiles_c) * TC;
  const int64_t R0 = (bid / tiles_c) * TP;

  if (MASK)
    for (int k = tid; k < keep_words; k += NT) keep_s[k] = keep[k];

  // this thread's position (fixed for the whole K loop) and the four consecutive taps of a K-tile it gathers
  const int p_local = tid & (TP - 1);
  const int kq = __builtin_amdgcn_readfirstlane(tid >> 7);
  const int64_t R = R0 + p_local;
  const int64_t gi0 = conv_first_image<COMPACT>(g, cr, R0);
  const char* const base = reinterpret_cast<const char*>(in + gi0 * ldin);  // block-uniform
  uint32_t toff = 0;
  int base_row = 0;
  uint32_t vmask = 0;
  int64_t gi = 0;
  int ho = 0, wo = 0;
  if (conv_row<COMPACT>(g, cr, R, total_rows, &gi, &ho, &wo)) {
    const int h0 = ho * g.sh - g.pt;
    const int w0 = wo * g.sw - g.pl;
    toff = (uint32_t)((gi - gi0) * ldin * 8);
    base_row = h0 + w0 * g.H;
    // taps inside the image - and, where the input images come with windows, inside this image's window (the
    // rows outside it are zero and may not be in memory)
    int ha = 0, hb = g.H - 1, wa = 0, wb = g.W - 1;
    if (COMPACT && cr.in_box != nullptr) {
      const ColBox b = cr.in_box[gi];
      ha = max(ha, (int)b.h0), hb = min(hb, (int)b.h1), wa = max(wa, (int)b.w0), wb = min(wb, (int)b.w1);
    }
    for (int fw = 0; fw < g.FW; ++fw)
      for (int fh = 0; fh < g.FH; ++fh) {
        const int h = h0 + fh * g.dh, w = w0 + fw * g.dw;
        if (h >= ha && h <= hb && w >= wa && w <= wb) vmask |= 1u << (fh + g.FH * fw);
      }
  }

  double rp[4];
  struct alignas(32) Tap4 {
    FastTap t[4];
  };
  auto gather = [&](int k0) {
    const Tap4 t4 = *reinterpret_cast<const Tap4*>(taps + k0 + kq * 4);  // wave-uniform: one scalar load
    int row[4];
    bool ok[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      row[q] = base_row + t4.t[q].off;
      ok[q] = (vmask & t4.t[q].bit) != 0;
    }
    if (MASK) {
      // (the row of a tap outside the image may lie outside the mask, even outside the block's LDS, where a
      // read returns zero: the word read for it is not used)
      uint32_t b[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) b[q] = keep_s[row[q] >> 5];
#pragma unroll
      for (int q = 0; q < 4; ++q) ok[q] = ok[q] && __builtin_amdgcn_ubfe(b[q], (uint32_t)row[q] & 31u, 1u) != 0;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      double v = 0.0;
      if (ok[q]) v = *reinterpret_cast<const double*>(base + (toff + ((uint32_t)row[q] << 3)));
      rp[q] = v;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 4; ++q) Ps[buf][(kq * 4 + q) * TP + p_local] = rp[q];
  };
  // weights: transfer w of a K-tile brings rows w*kRowsPerLoad ... of the tile; lane l its 16 bytes
  const unsigned w_lds = lds_addr_of(&Wts[0][0]) + (unsigned)wave * 1024u;
  const unsigned w_voff = (unsigned)(((lane / (TC / 2)) * coutp + 2 * (lane % (TC / 2))) * 8);
  const double* const w_base = Wk + (int64_t)(wave * kRowsPerLoad) * coutp + c0;
  auto dma = [&](int k0, int buf) {
    if (wave < kWLoads) lds_dma16(w_base + (int64_t)k0 * coutp, w_voff, w_lds + (unsigned)(buf * kKt * TC * 8));
  };

  double4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};

  __syncthreads();  // row mask in place
  const int nk = g.Kp / kKt;
  gather(0);
  dma(0, 0);
  store(0);
  wait_vm<0>();
  block_barrier();
  const int l16 = lane & 15, lq = lane >> 4;
  const double* const ps0 = &Ps[0][wr * (TP / WR) + l16 + lq * TP];
  const double* const ws0 = &Wts[0][wc * (TC / WC) + l16 + lq * TC];
  // one K-tile out of buffer `cur` (a constant, so that every LDS address is a base register plus an immediate)
  auto step = [&](int kt, auto cur_c) {
    constexpr int cur = decltype(cur_c)::value;
    if (kt + 1 < nk) {
      gather((kt + 1) * kKt);
      dma((kt + 1) * kKt, cur ^ 1);
    }
    const double* ps = ps0 + cur * (kKt * TP);
    const double* ws = ws0 + cur * (kKt * TC);
#pragma unroll
    for (int kk = 0; kk < kKt / 4; ++kk) {
      double b[FM], a[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) b[i] = ps[kk * 4 * TP + i * 16];
#pragma unroll
      for (int j = 0; j < FN; ++j) a[j] = ws[kk * 4 * TC + j * 16];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[j], b[i], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < nk) store(cur ^ 1);
    wait_vm<0>();     // this wave's weight transfer has landed ...
    block_barrier();  // ... and everybody's; everybody is done with the tiles of this step
  };
  for (int kt = 0; kt < nk; kt += 2) {
    step(kt, std::integral_constant<int, 0>());
    if (kt + 1 < nk) step(kt + 1, std::integral_constant<int, 1>());
  }
  conv_store_tile<TP, TC, WR, WC, FM, FN, COMPACT>(acc, out, ldout, bias, g, total_rows, R0, c0, wr, wc, lane, cr);
}

template <int TC, int WR, int WC, bool MASK, bool COMPACT>
__global__ __launch_bounds__(512) void conv2d_fast_kernel(ConvFastArgs a, const ConvSet* __restrict__ table, ConvSet one) {
  __shared__ __attribute__((aligned(1024))) double lds[2 * kKt * (128 + TC)];
  extern __shared__ uint32_t keep_s[];  // row mask (MASK only)
  const ConvSet set = conv_set_of_block(table, one);
  if ((int)blockIdx.x >= set.blocks) return;
  conv2d_fast_block<TC, WR, WC, MASK, COMPACT>(a, set, blockIdx.x, lds, keep_s);
}

// Window of column j of the output: from the window of the input's column (in_box null: whole image) or the pixel of its
// unit vector.
__device__ __forceinline__ ColBox conv_out_box(const ConvSetup& d, const ConvGeom& g, int64_t j) {
  int h0 = 0, h1 = g.H - 1, w0 = 0, w1 = g.W - 1;  // window of the input column
  if (j >= d.dense) {
    const int src = d.idx[j - d.dense] % g.HW;
    w0 = w1 = src / g.H;
    h0 = h1 = src - w0 * g.H;
  } else if (j > 0 && d.in_box != nullptr) {
    const ColBox b = d.in_box[j];
    h0 = b.h0, h1 = b.h1, w0 = b.w0, w1 = b.w1;
  }
  // the centre image is not sparse: where every tap falls into the padding it still holds the bias
  if (j == 0) return ColBox{0, (int16_t)(g.Ho - 1), 0, (int16_t)(g.Wo - 1)};
  if (h0 > h1 || w0 > w1) return ColBox{1, 0, 1, 0};
  // output rows whose taps ho*sh - pt + fh*dh (0 <= fh < FH) reach [h0, h1]
  // (strides are the layer's: the branch is uniform, and a division takes some thirty instructions)
  auto floordiv = [](int a, int s) { return (s & (s - 1)) == 0 ? a >> (31 - __builtin_clz(s)) : a >= 0 ? a / s : -((-a + s - 1) / s); };
  const int a0 = h0 + g.pt - (g.FH - 1) * g.dh, a1 = h1 + g.pt;
  const int b0 = w0 + g.pl - (g.FW - 1) * g.dw, b1 = w1 + g.pl;
  const int ho0 = max(0, -floordiv(-a0, g.sh)), ho1 = min(g.Ho - 1, floordiv(a1, g.sh));
  const int wo0 = max(0, -floordiv(-b0, g.sw)), wo1 = min(g.Wo - 1, floordiv(b1, g.sw));
  return (ho0 > ho1 || wo0 > wo1) ? ColBox{1, 0, 1, 0} : ColBox{(int16_t)ho0, (int16_t)ho1, (int16_t)wo0, (int16_t)wo1};
}

// What the kernels above and below look up, for every set of a call (blockIdx.y) in one launch: the windows of the output's
// columns (ConvSetup::out_box), by input row the unit-vector column that sits there (ConvSetup::inv; -1: none), and the
// order of the columns by the start of their windows (ConvSetup::order).  The first sort_blocks blocks make the order, a run
// of columns each, the next inv_blocks build kInvRows entries of the second table each: in LDS, because every entry is written whether
// or not a column names it, then out in order.  Latency bound (a few KB).
constexpr int kInvRows = 4096;
__global__ __launch_bounds__(kSortThreads) void conv_setup_kernel(const ConvSetup* __restrict__ table, ConvSetup one, int sort_blocks,
                                                                  int sort_run, int inv_blocks, ConvGeom g) {
  const ConvSetup d = table ? table[blockIdx.y] : one;
  const int blk = (int)blockIdx.x - sort_blocks;
  if (blk < 0) {
    if (d.order == nullptr) return;
    sort_windows(d.dense - 1, g.P, d.order, d.first, sort_run, blockIdx.x, [&](int j) {
      const ColBox b = conv_out_box(d, g, j);
      return b.h0 > b.h1 ? 0 : b.w0 * g.Ho + b.h0;
    });
    return;
  }
  if (blk < inv_blocks) {
    __shared__ int32_t rows[kInvRows];
    const int r0 = blk * kInvRows, nr = min(kInvRows, d.n_inv - r0);
    if (d.inv == nullptr || nr <= 0) return;
    for (int r = threadIdx.x; r < nr; r += kSortThreads) rows[r] = -1;
    __syncthreads();
    for (int t0 = threadIdx.x; t0 < d.m; t0 += 4 * kSortThreads) {
      int at[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) at[u] = t0 + u * kSortThreads < d.m ? d.idx[t0 + u * kSortThreads] - r0 : -1;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (at[u] >= 0 && at[u] < nr) rows[at[u]] = t0 + u * kSortThreads;
    }
    __syncthreads();
    for (int r = threadIdx.x; r < nr; r += kSortThreads) d.inv[r0 + r] = rows[r];
    return;
  }
  const int64_t j = (blk - inv_blocks) * (int64_t)kSortThreads + threadIdx.x;
  if (d.out_box == nullptr || j >= (int64_t)d.dense + d.m) return;
  d.out_box[j] = conv_out_box(d, g, j);
}

__global__ void zero_pad_rows_kernel(double* __restrict__ V, int64_t ld, int64_t N, int64_t ncols) {
  const int64_t pad = ld - N;
  const int64_t total = pad * ncols;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x)
    V[N + t % pad + (t / pad) * ld] = 0.0;
}


// ---- convolution of one-hot generator images -----------------------------------------------------
// A generator that is s * e_r (r = pixel (h, w, ci)) maps to the filter "stamped" around that pixel:
// out(ho, wo, co) = s * W(fh, fw, ci, co) for the one tap with ho*sh - pt + fh*dh = h and
// wo*sw - pl + fw*dw = w, and zero elsewhere.  The dense accumulation would add exact zeros to that
// one product, so 0 + w*s is the same value.  One pass that writes the output columns (HBM bound);
// lane = two adjacent output rows, the waves of a block interleave columns.
__global__ __launch_bounds__(512) void conv_stamp_kernel(const StampSet* __restrict__ table, StampSet one, ConvGeom g,
                                                         const double* __restrict__ Wt, int64_t ldout, int cols_per_chunk) {
  const StampSet d = table ? table[blockIdx.z] : one;
  const int j0 = min(d.m, (int)blockIdx.y * cols_per_chunk);  // an empty chunk still writes its (zero) sums
  const int j1 = min(d.m, j0 + cols_per_chunk);
  if (d.m == 0) return;
  double2 xmin1 = {0, 0}, xmin2 = {0, 0}, xmax1 = {0, 0}, xmax2 = {0, 0};
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t r0 = (int64_t)blockIdx.x * 128 + 2 * lane;
  const int64_t Nout = (int64_t)g.P * g.Cout;
  // the two output rows of this lane: (ho, wo, co), fixed for all columns
  int hb[2], wb[2], co[2];
  bool real[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int64_t r = r0 + e;
    real[e] = r < Nout;
    const int p = real[e] ? (int)(r % g.P) : 0;
    co[e] = real[e] ? (int)(r / g.P) : 0;
    const int wo = p / g.Ho;
    const int ho = p - wo * g.Ho;
    hb[e] = ho * g.sh - g.pt;  // input row reached by tap fh = 0
    wb[e] = wo * g.sw - g.pl;
  }
  // the columns of the chunk are decoded once per block (pixel position, channel offset into the
  // weights, scale) in batches of kStampBatch and then read back from LDS by all lanes
  constexpr int kStampBatch = 256;
  __shared__ int s_h[kStampBatch], s_w[kStampBatch], s_k[kStampBatch];
  __shared__ double s_s[kStampBatch];
  const bool unit_dil = g.dh == 1 && g.dw == 1;
  for (int jb = j0; jb < j1; jb += kStampBatch) {
    const int nb = min(kStampBatch, j1 - jb);
    __syncthreads();
    for (int t = threadIdx.x; t < nb; t += 512) {
      const int src = d.idx[jb + t];
      const int ci = src / g.HW;
      const int q = src - ci * g.HW;
      const int w = q / g.H;
      s_h[t] = q - w * g.H;
      s_w[t] = w;
      s_k[t] = g.FH * g.FW * ci;
      s_s[t] = d.scale != nullptr ? d.scale[src] : 1.0;
    }
    __syncthreads();
    for (int t = wave; t < nb; t += 8) {
      const int h = s_h[t], w = s_w[t], kc = s_k[t];
      const double s = s_s[t];
      double v[2];
      bool inwin[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        v[e] = 0.0;
        const int th = h - hb[e], tw = w - wb[e];
        inwin[e] = real[e] && th >= 0 && tw >= 0 && th <= (g.FH - 1) * g.dh && tw <= (g.FW - 1) * g.dw;
        if (real[e] && th >= 0 && tw >= 0) {
          int fh = th, fw = tw;
          bool hit = true;
          if (!unit_dil) {
            fh = th / g.dh;
            fw = tw / g.dw;
            hit = fh * g.dh == th && fw * g.dw == tw;
          }
          if (hit && fh < g.FH && fw < g.FW) {
            const double wv = Wt[fh + g.FH * fw + kc + (int64_t)co[e] * g.Kp];
            v[e] = __dadd_rn(0.0, __dmul_rn(wv, s));
          }
        }
      }
      if (d.win_only) {
        double* o = d.out + r0 + (int64_t)(jb + t) * ldout;
        if (inwin[0]) o[0] = v[0];
        if (inwin[1]) o[1] = v[1];
      } else if (r0 < ldout) {
        *reinterpret_cast<double2*>(d.out + r0 + (int64_t)(jb + t) * ldout) = make_double2(v[0], v[1]);
      }
      const double pl = d.plb[jb + t], pu = d.pub[jb + t];
      const double px = fmax(v[0], 0.0), nx = fmin(v[0], 0.0);
      const double py = fmax(v[1], 0.0), ny = fmin(v[1], 0.0);
      xmin1.x = fma(px, pl, xmin1.x);
      xmin1.y = fma(py, pl, xmin1.y);
      xmax1.x = fma(px, pu, xmax1.x);
      xmax1.y = fma(py, pu, xmax1.y);
      xmin2.x = fma(nx, pu, xmin2.x);
      xmin2.y = fma(ny, pu, xmin2.y);
      xmax2.x = fma(nx, pl, xmax2.x);
      xmax2.y = fma(ny, pl, xmax2.y);
    }
  }
  // range sums of this chunk: the eight waves hold different columns of the same rows
  __shared__ double2 red[8][4][64];
  __syncthreads();
  if (wave > 0) {
    red[wave][0][lane] = xmin1;
    red[wave][1][lane] = xmin2;
    red[wave][2][lane] = xmax1;
    red[wave][3][lane] = xmax2;
  }
  __syncthreads();
  if (wave == 0 && r0 < ldout) {
    for (int w = 1; w < 8; ++w) {
      xmin1.x += red[w][0][lane].x;
      xmin1.y += red[w][0][lane].y;
      xmin2.x += red[w][1][lane].x;
      xmin2.y += red[w][1][lane].y;
      xmax1.x += red[w][2][lane].x;
      xmax1.y += red[w][2][lane].y;
      xmax2.x += red[w][3][lane].x;
      xmax2.y += red[w][3][lane].y;
    }
    double* p = d.part + ((int64_t)blockIdx.y * 4) * ldout + r0;
    *reinterpret_cast<double2*>(p) = xmin1;
    *reinterpret_cast<double2*>(p + ldout) = xmin2;
    *reinterpret_cast<double2*>(p + 2 * ldout) = xmax1;
    *reinterpret_cast<double2*>(p + 3 * ldout) = xmax2;
  }
}

// One bit per row of a set with a pending row reset: 1 where the row is kept.  Word w covers rows 32w..32w+31.
struct KeepBits {
  const int32_t* cls;
  uint32_t* bits;
};
__global__ __launch_bounds__(256) void keep_bits_kernel(const KeepBits* __restrict__ table, KeepBits one, int64_t N, int words) {
  const KeepBits set = table ? table[blockIdx.y] : one;
  const int32_t* __restrict__ cls = set.cls;
  uint32_t* __restrict__ bits = set.bits;
  const int64_t r = blockIdx.x * (int64_t)256 + threadIdx.x;
  const unsigned long long b = __ballot(r < N && cls[r] == kKeep);
  const int lane = threadIdx.x & 63;
  const int64_t w = r >> 5;
  if ((lane & 31) == 0 && w < words) bits[w] = (uint32_t)(b >> lane);
}

template <int S>
__global__ __launch_bounds__(256) void conv_stamp_rows_kernel(StampSet d, ConvGeom g, const double* __restrict__ Wt, const double* __restrict__ Wk,
                                                              int coutp, const int32_t* __restrict__ pixel_col, int64_t ldout) {
  __shared__ __attribute__((aligned(16))) int2 taps[kStampTapTable];
  __shared__ int cnt[4];
  static_assert(sizeof(int2) * kStampTapTable >= 8192 + sizeof(int2) * kStampPixelTaps, "sums and list of the pass by position");
  if (d.pix != nullptr)
    conv_stamp_pixels_block<256>(blockIdx.x, reinterpret_cast<double*>(taps), cnt, taps + 1024, d, g, Wk, coutp, pixel_col, ldout);
  else
    conv_stamp_rows_block<S, 256>(blockIdx.x, taps, d, g, Wt, pixel_col, ldout);
}

// The dense images' convolution and the stamps of the unit-vector columns of the same layer in one launch: the two
// write different columns of the output and read nothing of each other, the first is bound by the matrix pipe and the
// second by scattered stores, so their blocks are dealt to the chip in turn (every stride-th block of the grid is a
// stamp block, until there are no more) and run side by side on a compute unit.
template <int TC, int WR, int WC, bool MASK, bool COMPACT, int S>
__global__ __launch_bounds__(512) void conv2d_fast_stamps_kernel(ConvFastArgs a, const double* __restrict__ Wt,
                                                                 const ConvSet* __restrict__ table, ConvSet one) {
  static_assert(sizeof(int2) * kStampTapTable <= conv_fast_lds_bytes(TC), "the stamp blocks' tap table fits the tiles' LDS");
  static_assert(8 * 2064 + sizeof(int2) * kStampPixelTaps <= conv_fast_lds_bytes(TC), "... and so do sums and list by position");
  __shared__ __attribute__((aligned(1024))) double lds[2 * kKt * (128 + TC)];
  extern __shared__ uint32_t keep_s[];  // row mask (MASK only)
  const ConvSet set = conv_set_of_block(table, one);
  const int p = blockIdx.x;
  const int k = (p + 1) / set.stride;
  if ((p + 1) % set.stride == 0 && k <= a.stamp_blocks) {
    if (set.d.pix != nullptr)
      conv_stamp_pixels_block<512>(k - 1, lds, reinterpret_cast<int*>(lds + 2048), reinterpret_cast<int2*>(lds + 2064), set.d, a.g, a.Wk, a.coutp,
                                   set.d.pixel_col, a.ldout);
    else
      conv_stamp_rows_block<S, 512>(k - 1, reinterpret_cast<int2*>(lds), set.d, a.g, Wt, set.d.pixel_col, a.ldout);
    return;
  }
  const int bid = p - min(a.stamp_blocks, p / set.stride);
  if (bid >= set.blocks) return;
  conv2d_fast_block<TC, WR, WC, MASK, COMPACT>(a, set, bid, lds, keep_s);
}

// LDS of the convolution kernel beside its tap table and row mask: the two double-buffered operand tiles
template <int TP, int TC>
constexpr size_t conv_static_lds() {
  return sizeof(double) * 2 * (kKt * (TP + kPadRow) + TC * (kKt + kPadK));
}

template <int TP, int TC, int WR, int WC>
static int launch_conv_cfg(nnvhip_ctx* ctx, const nnvhip_conv2d* cv, const ConvGeom& g, const double* in, int64_t ldin,
                           double* out, int64_t ldout, int64_t ncols, const uint32_t* keep, int keep_words) {
  const int64_t total_rows = (int64_t)g.P * ncols;
  const int64_t tiles_c = ceil_div(g.Cout, TC);
  const int64_t blocks = ceil_div(total_rows, TP) * tiles_c;
  if (blocks >= (int64_t(1) << 31)) NNV_FAIL(NNVHIP_ERR_SHAPE, "convolution too large for one launch");
  const size_t dyn = sizeof(unsigned long long) * g.Kp + (keep ? sizeof(uint32_t) * (size_t)keep_words : 0);
  if (conv_static_lds<TP, TC>() + dyn > kConvLdsLimit)
    NNV_FAIL(NNVHIP_ERR_SHAPE, "filters with %d taps (FH*FW*Cin) and %d output channels are not supported: at most %d taps", g.K, g.Cout,
             (int)((kConvLdsLimit - conv_static_lds<TP, TC>()) / sizeof(unsigned long long) / kKt * kKt));
  NNV_TRY(ctx->kernel_timer_begin(ctx->kernel_timing));
  if (keep)
    NNV_LAUNCH(ctx, ctx->kernel_timing, (conv2d_f64_kernel<TP, TC, WR, WC, true>), dim3((unsigned)blocks), dim3(64 * WR * WC), dyn, in,
               ldin, out, ldout, cv->W->as<double>(), cv->bias ? cv->bias->as<double>() : nullptr, g, total_rows, (int)tiles_c, keep,
               keep_words);
  else
    NNV_LAUNCH(ctx, ctx->kernel_timing, (conv2d_f64_kernel<TP, TC, WR, WC, false>), dim3((unsigned)blocks), dim3(64 * WR * WC), dyn, in,
               ldin, out, ldout, cv->W->as<double>(), cv->bias ? cv->bias->as<double>() : nullptr, g, total_rows, (int)tiles_c, keep,
               keep_words);
  NNV_TRY(ctx->kernel_timer_end(ctx->kernel_timing, 1, 2.0 * (double)total_rows * g.Cout * g.K));
  NNV_HIP_TRY(hipGetLastError());
  return NNVHIP_OK;
}

// ---- which kernel, and whether it can mask rows on load --------------------------------------------
constexpr size_t conv_fast_static_lds(int tc) { return sizeof(double) * 2 * kKt * (128 + (size_t)tc); }
static int conv_tile_channels(const nnvhip_conv2d* cv) { return cv->Cout <= 16 ? 16 : cv->Cout <= 32 ? 32 : 64; }

// The kernel with scalar tap decoding: at most 32 spatial taps (one mask bit each), every byte offset it forms
// (a row of the image plus the images a 128-position tile can span) below 2^31.
static bool conv_fast_ok(const nnvhip_conv2d* cv, const ConvGeom& g, int64_t ldin, int64_t rows_per_image = 0) {
  if (tune_knobs().conv_general != 0 || cv->Wk == nullptr) return false;
  if (cv->FH * cv->FW > 32) return false;
  const int64_t n_in = (int64_t)g.HW * g.Cin;
  const int64_t images_per_tile = 127 / (rows_per_image > 0 ? rows_per_image : g.P) + 2;
  return (n_in + images_per_tile * ldin) * 8 < (int64_t(1) << 31);
}

bool conv2d_can_mask(const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo, int64_t ldin) {
  ConvGeom g;
  fill_geom(g, cv, H, W, Ho, Wo);
  const int64_t n_in = H * W * cv->Cin;
  if (n_in >= (int64_t(1) << 31) || cv->Kp > kMaxTaps) return false;
  const size_t mask = sizeof(uint32_t) * (size_t)ceil_div(n_in, 32);
  if (conv_fast_ok(cv, g, ldin)) return conv_fast_static_lds(conv_tile_channels(cv)) + mask <= kConvLdsLimit;
  // the general kernel, sized for its widest tile (128 x 64): the mask shares the dynamic LDS with the tap table
  return conv_static_lds<128, 64>() + sizeof(unsigned long long) * (size_t)cv->Kp + mask <= kConvLdsLimit;
}

int conv2d_prepare_weights(nnvhip_ctx* ctx, nnvhip_conv2d* cv) {
  cv->coutp = round_up(cv->Cout, 64);
  if (cv->Kp * cv->coutp >= (int64_t(1) << 28)) return NNVHIP_OK;  // stays on the general kernel
  NNV_TRY(ctx->alloc(sizeof(double) * cv->Kp * cv->coutp, &cv->Wk));
  hipLaunchKernelGGL(conv_weights_kmajor_kernel, dim3((unsigned)ceil_div(cv->Kp * cv->coutp, 256)), dim3(256), 0, ctx->stream,
                     cv->W->as<double>(), cv->Wk->as<double>(), (int)cv->Kp, (int)cv->Cout, (int)cv->coutp);
  NNV_HIP_TRY(hipGetLastError());
  return NNVHIP_OK;
}

static int conv_fast_taps(nnvhip_ctx* ctx, const nnvhip_conv2d* cv, const ConvGeom& g, const FastTap** tab) {
  for (const auto& t : cv->tap_tables)
    if (t.H == g.H && t.W == g.W) {
      *tab = t.tab->as<FastTap>();
      return NNVHIP_OK;
    }
  nnvhip_conv2d::TapTable t;
  t.H = g.H;
  t.W = g.W;
  NNV_TRY(ctx->alloc(sizeof(FastTap) * (size_t)g.Kp, &t.tab));
  hipLaunchKernelGGL(conv_fast_taps_kernel, dim3((unsigned)ceil_div(g.Kp, 256)), dim3(256), 0, ctx->stream, t.tab->as<FastTap>(), g);
  NNV_HIP_TRY(hipGetLastError());
  if (cv->tap_tables.size() >= 8) cv->tap_tables.erase(cv->tap_tables.begin());
  cv->tap_tables.push_back(t);
  *tab = t.tab->as<FastTap>();
  return NNVHIP_OK;
}

// The sets of `jobs` have a row mask (keep), windows (compact) and stamps that go into the launch (stamps) all or none.
template <int TC, int WR, int WC>
static int launch_conv_fast(nnvhip_ctx* ctx, const nnvhip_conv2d* cv, const ConvGeom& g, int64_t ldout, const std::vector<ConvSet>& jobs,
                            const std::vector<int64_t>& ncols, bool keep, int keep_words, bool compact, bool stamps) {
  const int64_t tiles_c = ceil_div(g.Cout, TC);
  const size_t dyn = keep ? sizeof(uint32_t) * (size_t)keep_words : 0;
  if (conv_fast_static_lds(TC) + dyn > kConvLdsLimit) NNV_FAIL(NNVHIP_ERR_SHAPE, "internal: row mask too large for the convolution kernel");
  ConvFastArgs a{};
  NNV_TRY(conv_fast_taps(ctx, cv, g, &a.taps));
  a.ldout = ldout;
  a.Wk = cv->Wk->as<double>();
  a.coutp = (int)cv->coutp;
  a.bias = cv->bias ? cv->bias->as<double>() : nullptr;
  a.g = g;
  a.tiles_c = (int)tiles_c;
  a.keep_words = keep_words;
  // lanes per output row of the stamp blocks: 8 for filters with many taps (beside the tile blocks that measured best:
  // CNN 32x32x3 0.747 ms against 0.752 with 16 lanes, 0.756 with 4, 0.782 with 32) and where one lane to a row would leave half
  // of the chip without a block (32 x 32 x 3 into 8 channels, 16 blocks of stamps: 23.8 us, with 8 lanes 128 blocks and 8.0 us),
  // else 1
  const bool wide_stamps = g.K > 32 || ceil_div(ldout, 512) * (int64_t)jobs.size() < 128;
  int64_t stamp_blocks = stamps ? ceil_div(ldout * (wide_stamps ? 8 : 1), 512) : 0;
  for (const ConvSet& s : jobs)
    if (stamps && s.d.pix != nullptr) stamp_blocks = std::max<int64_t>(stamp_blocks, conv_stamp_pixel_blocks(g.P, g.K, 512));
  a.stamp_blocks = (int)stamp_blocks;
  std::vector<ConvSet> sets = jobs;
  double rows = 0.0;
  for (size_t i = 0; i < sets.size(); ++i) {
    ConvSet& s = sets[i];
    s.total_rows = compact ? (int64_t)g.P + (ncols[i] - 1) * s.cr.area : (int64_t)g.P * ncols[i];
    const int64_t blocks = ceil_div(s.total_rows, 128) * tiles_c;
    if (blocks + stamp_blocks >= (int64_t(1) << 31)) NNV_FAIL(NNVHIP_ERR_SHAPE, "convolution too large for one launch");
    s.blocks = (int32_t)blocks;
    s.stride = stamps ? (int32_t)std::max<int64_t>(1, (blocks + stamp_blocks) / stamp_blocks) : 1;
    rows += (double)s.total_rows;
  }
  for (size_t i0 = 0; i0 < sets.size(); i0 += 65535) {
    const size_t cnt = std::min<size_t>(65535, sets.size() - i0);
    int64_t grid_x = 0;
    for (size_t i = i0; i < i0 + cnt; ++i) grid_x = std::max<int64_t>(grid_x, sets[i].blocks + stamp_blocks);
    const ConvSet* table = nullptr;
    BufRef tab;
    if (cnt > 1) {  // (a device copy, as good as the staging ring here: see upload_table)
      NNV_TRY(ctx->upload(sets.data() + i0, sizeof(ConvSet) * cnt, &tab));
      table = tab->as<ConvSet>();
    }
    const ConvSet& one = sets[i0];
    const dim3 grid((unsigned)grid_x, (unsigned)cnt);
    NNV_TRY(ctx->kernel_timer_begin(ctx->kernel_timing));
#define NNV_CONV_FAST(MASK, COMPACT)                                                                                                     \
  do {                                                                                                                                   \
    if (!stamps)                                                                                                                         \
      NNV_LAUNCH(ctx, ctx->kernel_timing, (conv2d_fast_kernel<TC, WR, WC, MASK, COMPACT>), grid, dim3(512), dyn, a, table, one);         \
    else if (wide_stamps)                                                                                                                \
      NNV_LAUNCH(ctx, ctx->kernel_timing, (conv2d_fast_stamps_kernel<TC, WR, WC, MASK, COMPACT, 8>), grid, dim3(512), dyn, a,            \
                 cv->W->as<double>(), table, one);                                                                                       \
    else                                                                                                                                 \
      NNV_LAUNCH(ctx, ctx->kernel_timing, (conv2d_fast_stamps_kernel<TC, WR, WC, MASK, COMPACT, 1>), grid, dim3(512), dyn, a,            \
                 cv->W->as<double>(), table, one);                                                                                       \
  } while (0)
    if (keep && compact)
      NNV_CONV_FAST(true, true);
    else if (keep)
      NNV_CONV_FAST(true, false);
    else if (compact)
      NNV_CONV_FAST(false, true);
    else
      NNV_CONV_FAST(false, false);
#undef NNV_CONV_FAST
    NNV_TRY(ctx->kernel_timer_end(ctx->kernel_timing, 1, 2.0 * rows * g.Cout * g.K * ((double)cnt / (double)sets.size())));
    NNV_HIP_TRY(hipGetLastError());
  }
  return NNVHIP_OK;
}

int launch_zero_pad_rows(nnvhip_ctx* ctx, double* V, int64_t ld, int64_t N, int64_t ncols) {
  if (ld == N || ncols <= 0) return NNVHIP_OK;
  hipLaunchKernelGGL(zero_pad_rows_kernel, dim3(256), dim3(256), 0, ctx->stream, V, ld, N, ncols);
  NNV_HIP_TRY(hipGetLastError());
  return NNVHIP_OK;
}

int64_t conv_box_extent(const nnvhip_conv2d* cv, int dim, int64_t e, int64_t out_size) {
  // output positions whose taps reach a run of e input positions: floor((e - 1 + (F - 1) * dil) / stride) + 1
  const int64_t F = dim == 0 ? cv->FH : cv->FW;
  return std::min<int64_t>(out_size, (e - 1 + (F - 1) * cv->dil[dim]) / cv->stride[dim] + 1);
}

static int launch_setup(nnvhip_ctx* ctx, const ConvGeom& g, int64_t count, const ConvSetup* sets) {
  for (int64_t i0 = 0; i0 < count; i0 += 65535) {
    const int64_t cnt = std::min<int64_t>(65535, count - i0);
    int64_t inv_rows = 0, cols = 0;
    int64_t sorted = 0, sort_sets = 0;  // columns of a set at most, sets
    for (int64_t i = i0; i < i0 + cnt; ++i) {
      if (sets[i].order != nullptr) {
        sorted = std::max<int64_t>(sorted, sets[i].dense - 1);
        ++sort_sets;
      }
      if (sets[i].inv != nullptr) inv_rows = std::max<int64_t>(inv_rows, sets[i].n_inv);
      if (sets[i].out_box != nullptr) cols = std::max<int64_t>(cols, (int64_t)sets[i].dense + sets[i].m);
    }
    const int sort_run = sort_window_run(sorted, sort_sets), sort_blocks = sort_sets > 0 ? sort_window_blocks(sorted, sort_run) : 0;
    const int64_t inv_blocks = ceil_div(inv_rows, kInvRows), blocks = sort_blocks + inv_blocks + ceil_div(cols, kSortThreads);
    if (blocks == 0) continue;
    const ConvSetup* table = nullptr;
    BufRef tab;
    if (cnt > 1) {
      NNV_TRY(ctx->upload_table(sets + i0, sizeof(ConvSetup) * (size_t)cnt, &tab));
      table = tab->as<ConvSetup>();
    }
    hipLaunchKernelGGL(conv_setup_kernel, dim3((unsigned)blocks, (unsigned)cnt), dim3(kSortThreads), 0, ctx->stream, table, sets[i0],
                       sort_blocks, sort_run, (int)inv_blocks, g);
    NNV_HIP_TRY(hipGetLastError());
  }
  return NNVHIP_OK;
}

int launch_conv_setup(nnvhip_ctx* ctx, const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo, int64_t count,
                      const ConvSetup* sets) {
  ConvGeom g;
  fill_geom(g, cv, H, W, Ho, Wo);
  return launch_setup(ctx, g, count, sets);
}

int launch_pool_setup(nnvhip_ctx* ctx, int64_t H, int64_t W, int64_t Ho, int64_t Wo, const int64_t pool[2], const int64_t stride[2],
                      int64_t pad_top, int64_t pad_left, int64_t count, const ConvSetup* sets) {
  ConvGeom g{};
  g.H = (int)H;
  g.W = (int)W;
  g.Ho = (int)Ho;
  g.Wo = (int)Wo;
  g.FH = (int)pool[0];
  g.FW = (int)pool[1];
  g.sh = (int)stride[0];
  g.sw = (int)stride[1];
  g.dh = g.dw = 1;
  g.pt = (int)pad_top;
  g.pl = (int)pad_left;
  g.HW = (int)(H * W);
  return launch_setup(ctx, g, count, sets);
}

bool conv2d_in_windows(const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo, int64_t ldin, int64_t ncols,
                       const ColBox* out_box, int eh, int ew) {
  ConvGeom g;
  fill_geom(g, cv, H, W, Ho, Wo);
  return out_box != nullptr && ncols > 1 && eh > 0 && ew > 0 && 2 * (int64_t)eh * ew <= g.P &&
         conv_fast_ok(cv, g, ldin, (int64_t)eh * ew);
}

int launch_conv2d(nnvhip_ctx* ctx, const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo, int64_t ldout,
                  std::vector<ConvJob>& jobs) {
  if (cv->Kp > kMaxTaps) NNV_FAIL(NNVHIP_ERR_SHAPE, "filters with more than %d taps (FH*FW*Cin) are not supported", kMaxTaps);
  if ((cv->FH - 1) * cv->dil[0] > 0xffff || (cv->FW - 1) * cv->dil[1] > 0xffff)
    NNV_FAIL(NNVHIP_ERR_SHAPE, "dilated filter extent too large");
  ConvGeom g;
  fill_geom(g, cv, H, W, Ho, Wo);
  // a pending row reset of an input is applied on load, from one bit per input row
  const int64_t n_in = H * W * cv->Cin;
  const int keep_words = (int)ceil_div(n_in, 32);
  std::vector<const uint32_t*> keep(jobs.size(), nullptr);
  BufRef bits, bits_tab;
  {
    std::vector<KeepBits> kb;
    for (size_t i = 0; i < jobs.size(); ++i) {
      if (jobs[i].pending_cls == nullptr) continue;
      if (!conv2d_can_mask(cv, H, W, Ho, Wo, jobs[i].ldin)) NNV_FAIL(NNVHIP_ERR_SHAPE, "internal: row mask too large for the convolution kernel");
      keep[i] = jobs[i].pending_bits;
      if (keep[i] == nullptr) kb.push_back(KeepBits{jobs[i].pending_cls, nullptr});
    }
    if (!kb.empty()) {
      const int64_t words = round_up((int64_t)keep_words, 16);
      NNV_TRY(ctx->alloc(sizeof(uint32_t) * (size_t)words * kb.size(), &bits));
      size_t k = 0;
      for (size_t i = 0; i < jobs.size(); ++i)
        if (jobs[i].pending_cls != nullptr && keep[i] == nullptr) {
          kb[k].bits = bits->as<uint32_t>() + words * (int64_t)k;
          keep[i] = kb[k++].bits;
        }
      // whole waves only, so that every word is written by a lane that exists
      for (size_t i0 = 0; i0 < kb.size(); i0 += 65535) {
        const size_t cnt = std::min<size_t>(65535, kb.size() - i0);
        const KeepBits* table = nullptr;
        if (cnt > 1) {
          NNV_TRY(ctx->upload_table(kb.data() + i0, sizeof(KeepBits) * cnt, &bits_tab));
          table = bits_tab->as<KeepBits>();
        }
        hipLaunchKernelGGL(keep_bits_kernel, dim3((unsigned)ceil_div(n_in, 256), (unsigned)cnt), dim3(256), 0, ctx->stream, table, kb[i0],
                           n_in, keep_words);
        NNV_HIP_TRY(hipGetLastError());
      }
    }
  }
  // 128 positions x Cout tile, eight waves per block (two per SIMD keep the MFMA pipe fed while
  // the other wave gathers).  Sets that take the same instantiation share a launch.
  std::vector<ConvSet> group[8];
  std::vector<int64_t> group_cols[8];
  for (size_t i = 0; i < jobs.size(); ++i) {
    ConvJob& jb = jobs[i];
    // Generator images with known windows are computed inside them only (the caller has zeroed the rest) when that
    // at least halves the rows; it takes the kernel with scalar tap decoding.
    ConvSet set{};
    if (conv2d_in_windows(cv, H, W, Ho, Wo, jb.ldin, jb.ncols, jb.out_box, jb.eh, jb.ew))
      set.cr = ConvRows{jb.out_box, jb.eh, jb.eh * jb.ew, jb.in_box};
    const bool compact = set.cr.box != nullptr;
    if (!compact && (jb.in_box != nullptr || jb.leave_outside))
      NNV_FAIL(NNVHIP_ERR_ARG, "internal: the convolution was to stay inside the images' windows");
    if (compact && !jb.leave_outside)  // everything outside the windows
      NNV_HIP_TRY(hipMemsetAsync(jb.out + ldout, 0, sizeof(double) * (size_t)ldout * (size_t)(jb.ncols - 1), ctx->stream));
    if (!compact && !conv_fast_ok(cv, g, jb.ldin)) {
      int st;
      if (cv->Cout <= 16)
        st = launch_conv_cfg<128, 16, 8, 1>(ctx, cv, g, jb.in, jb.ldin, jb.out, ldout, jb.ncols, keep[i], keep_words);
      else if (cv->Cout <= 32)
        st = launch_conv_cfg<128, 32, 4, 2>(ctx, cv, g, jb.in, jb.ldin, jb.out, ldout, jb.ncols, keep[i], keep_words);
      else
        st = launch_conv_cfg<128, 64, 4, 2>(ctx, cv, g, jb.in, jb.ldin, jb.out, ldout, jb.ncols, keep[i], keep_words);
      NNV_TRY(st);
      continue;
    }
    // the stamps of the set's unit-vector columns ride along where they are made row by row and come with their
    // pixel table and a place for their range sums
    static_assert(sizeof(ConvStampSet) == sizeof(StampSet), "same layout");
    const ConvStampSet* stamp = jb.stamp;
    jb.stamped = stamp != nullptr && stamp->m > 0 && stamp->pixel_col != nullptr && stamp->part != nullptr && cv->dil[0] == 1 &&
                 cv->dil[1] == 1 && g.K <= kStampTapTable;
    if (jb.stamped) {
      memcpy(&set.d, stamp, sizeof set.d);
      if (!set.d.win_only)  // whole columns: the zeros first
        NNV_HIP_TRY(hipMemsetAsync(set.d.out, 0, sizeof(double) * (size_t)ldout * (size_t)set.d.m, ctx->stream));
    }
    set.in = jb.in;
    set.ldin = jb.ldin;
    set.out = jb.out;
    set.keep = keep[i];
    const int key = (keep[i] != nullptr ? 1 : 0) | (compact ? 2 : 0) | (jb.stamped ? 4 : 0);
    group[key].push_back(set);
    group_cols[key].push_back(jb.ncols);
  }
  for (int key = 0; key < 8; ++key) {
    if (group[key].empty()) continue;
    const bool masked = key & 1, compact = key & 2, stamps = key & 4;
    if (cv->Cout <= 16)
      NNV_TRY((launch_conv_fast<16, 8, 1>(ctx, cv, g, ldout, group[key], group_cols[key], masked, keep_words, compact, stamps)));
    else if (cv->Cout <= 32)
      NNV_TRY((launch_conv_fast<32, 4, 2>(ctx, cv, g, ldout, group[key], group_cols[key], masked, keep_words, compact, stamps)));
    else
      NNV_TRY((launch_conv_fast<64, 4, 2>(ctx, cv, g, ldout, group[key], group_cols[key], masked, keep_words, compact, stamps)));
  }
  return NNVHIP_OK;
}

void fill_geom(ConvGeom& g, const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo) {
  g.H = (int)H;
  g.W = (int)W;
  g.Cin = (int)cv->Cin;
  g.Ho = (int)Ho;
  g.Wo = (int)Wo;
  g.Cout = (int)cv->Cout;
  g.FH = (int)cv->FH;
  g.FW = (int)cv->FW;
  g.sh = (int)cv->stride[0];
  g.sw = (int)cv->stride[1];
  g.dh = (int)cv->dil[0];
  g.dw = (int)cv->dil[1];
  g.pt = (int)cv->pad[0];
  g.pl = (int)cv->pad[2];
  g.K = (int)cv->K;
  g.Kp = (int)cv->Kp;
  g.P = (int)(Ho * Wo);
  g.HW = (int)(H * W);
}

static bool conv_stamps_by_row(const nnvhip_conv2d* cv) { return cv->dil[0] == 1 && cv->dil[1] == 1; }
bool conv_stamps_by_pixel(const nnvhip_conv2d* cv) { return conv_stamps_by_row(cv); }

int64_t conv_stamp_chunks(const nnvhip_conv2d* cv, int64_t ldout, int64_t count, int64_t max_m) {
  if (conv_stamps_by_row(cv)) return 1;
  const int64_t row_blocks = ceil_div(ldout, 128);
  int64_t chunks = std::max<int64_t>(1, std::min<int64_t>(ceil_div(8192, row_blocks * count), ceil_div(std::max<int64_t>(max_m, 1), 32)));
  const int64_t cpc = ceil_div(std::max<int64_t>(max_m, 1), chunks);
  return ceil_div(std::max<int64_t>(max_m, 1), cpc);
}

int launch_conv_stamps(nnvhip_ctx* ctx, const nnvhip_conv2d* cv, int64_t H, int64_t W, int64_t Ho, int64_t Wo,
                       int64_t ldout, int64_t count, const ConvStampSet* sets, int64_t chunks) {
  static_assert(sizeof(ConvStampSet) == sizeof(StampSet), "same layout");
  if (count <= 0) return NNVHIP_OK;
  if (count > 65535) NNV_FAIL(NNVHIP_ERR_SHAPE, "at most 65535 sets per call");
  int64_t max_m = 0;
  double bytes = 0.0;
  for (int64_t i = 0; i < count; ++i) {
    max_m = std::max<int64_t>(max_m, sets[i].m);
    // algorithmic: the output columns -- whole ones, or, when only the rows inside each column's window are written,
    // the filter stamp itself (at most FH * FW positions of every output channel)
    const double rows_written = sets[i].win_only ? (double)std::min<int64_t>(Ho * Wo, cv->FH * cv->FW) * (double)cv->Cout
                                                 : (double)(Ho * Wo * cv->Cout);
    bytes += 8.0 * rows_written * (double)sets[i].m;
  }
  if (max_m == 0) return NNVHIP_OK;
  ConvGeom g;
  fill_geom(g, cv, H, W, Ho, Wo);
  if (conv_stamps_by_row(cv)) {
    if (chunks != 1) NNV_FAIL(NNVHIP_ERR_ARG, "internal: one chunk of range sums per set");
    if (g.K > kStampTapTable) NNV_FAIL(NNVHIP_ERR_SHAPE, "internal: more taps than the stamp kernel's table holds");
    NNV_TRY(ctx->kernel_timer_begin(ctx->kernel_timing));
    for (int64_t i = 0; i < count; ++i) {
      if (sets[i].m == 0) continue;
      StampSet one;
      memcpy(&one, &sets[i], sizeof one);
      const int32_t* pc = one.pixel_col;
      if (pc == nullptr) NNV_FAIL(NNVHIP_ERR_ARG, "internal: stamps without their pixel table");
      if (!one.win_only)  // whole columns: the zeros first
        NNV_HIP_TRY(hipMemsetAsync(one.out, 0, sizeof(double) * (size_t)ldout * (size_t)one.m, ctx->stream));
      const int64_t blocks = one.pix != nullptr ? conv_stamp_pixel_blocks(g.P, g.K, 256) : ceil_div(ldout * (g.K <= 32 ? 1 : 16), 256);
      if (g.K <= 32)
        NNV_LAUNCH(ctx, ctx->kernel_timing && i == 0, conv_stamp_rows_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, one, g,
                   cv->W->as<double>(), cv->Wk ? cv->Wk->as<double>() : nullptr, (int)cv->coutp, pc, ldout);
      else
        NNV_LAUNCH(ctx, ctx->kernel_timing && i == 0, conv_stamp_rows_kernel<16>, dim3((unsigned)blocks), dim3(256), 0,
                   one, g, cv->W->as<double>(), cv->Wk ? cv->Wk->as<double>() : nullptr, (int)cv->coutp, pc, ldout);
    }
    NNV_TRY(ctx->kernel_timer_end(ctx->kernel_timing, 5, bytes));
    NNV_HIP_TRY(hipGetLastError());
    return NNVHIP_OK;
  }
  const int64_t row_blocks = ceil_div(ldout, 128);
  const int64_t cpc = ceil_div(max_m, chunks);
  const StampSet* table = nullptr;
  BufRef tab;
  if (count > 1) {
    NNV_TRY(ctx->upload_table(sets, sizeof(StampSet) * count, &tab));
    table = tab->as<StampSet>();
  }
  StampSet one;
  memcpy(&one, &sets[0], sizeof one);
  NNV_TRY(ctx->kernel_timer_begin(ctx->kernel_timing));
  NNV_LAUNCH(ctx, ctx->kernel_timing, conv_stamp_kernel, dim3((unsigned)row_blocks, (unsigned)chunks, (unsigned)count), dim3(512), 0,
             table, one, g, cv->W->as<double>(), ldout, (int)cpc);
  NNV_TRY(ctx->kernel_timer_end(ctx->kernel_timing, 5, bytes));
  NNV_HIP_TRY(hipGetLastError());
  return NNVHIP_OK;
}

}  // namespace nnvhip
