// affineMap of a fully connected layer: C = W * [c V] on fp64 MFMA (v_mfma_f64_16x16x4_f64).
//
// Both operands are staged through LDS.  The MFMA operand roles are chosen for
// column-major stores: the instruction's "b" operand carries 16 consecutive ROWS of W (the
// memory-contiguous direction of C), its "a" operand 16 columns of V, so lane l, register r of
// an accumulator holds C[row0 + l%16][col0 + l/16 + 4r] and lanes 0..15 store one 128-byte line.
#include <algorithm>
#include <cstdlib>
#include <string>

#include "internal.h"
#include "lds_dma.h"
#include "mfma_tile.h"

namespace nnvhip {

// Where a block's tile lies and what it reads (both kernels below).
struct GemmTile {
  int m0;
  int64_t nt, n0;
  const int32_t* kmap;  // rows of B (= columns of A) the product goes over, -1 padded to whole stages; null: all
  const double* Bk;     // those rows of B packed (row t = row kmap[t]), or null
  int64_t ldbk, bk_col0;
  int64_t col_base;     // column of B and C behind the tile's first column
  int64_t col_end;      // first column past the valid ones, in the same numbering
  int64_t b_col_base;   // column of B behind the tile's first column
  // fused range sums: the tile's first column and the end of the valid ones in the numbering of plb / pub (the set's own
  // columns), and the chunk of partial sums the tile fills
  const double *plb, *pub;
  double* rpart;
  int64_t rcol0, rcol_end, rchunk;
  int Kp;
};
struct GemmArgs {
  const double* A;
  const double* B;
  double* C;
  const double* bias;
  double* part;  // split-K workspace
  const double *plb, *pub;
  double* rpart;
  const int32_t* kmap;
  const GemmSeg* segs;
  const int32_t* colmap;
  const int32_t* bmap;
  const double* Bk;
  int64_t lda, ldb, ldc, ldbk, ncols;
  int32_t Mp, Kp, tiles_m, tiles_n, xr, local_m, ksplit;
};

// XCD-aware tile mapping.  Workgroups are dealt round-robin to the 8 XCDs (each with its own 4 MiB L2) by linear id, so
// blockIdx.x % 8 names the XCD.  The XCDs form an xr x (8/xr) grid over the tile matrix: XCD (i, j) owns the row tiles
// congruent to i mod xr and the column tiles congruent to j mod 8/xr, i.e. it touches 1/xr of W and xr/8 of V instead of
// all of V.  Inside an XCD consecutive blocks walk down the row tiles of one column tile, keeping its V tile hot.
template <int TM, int TN, bool MAPPED>
__device__ __forceinline__ bool gemm_tile_of(const GemmArgs& g, GemmTile* t) {
  const int xcd = blockIdx.x & 7;
  const int slot = blockIdx.x >> 3;
  const int xc = 8 / g.xr;
  const int mt = (slot % g.local_m) * g.xr + (xcd % g.xr);
  const int64_t nt = (int64_t)(slot / g.local_m) * xc + (xcd / g.xr);
  if (mt >= g.tiles_m || nt >= g.tiles_n) return false;
  t->m0 = mt * TM;
  t->nt = nt;
  t->n0 = nt * TN;
  t->kmap = g.kmap;
  t->Bk = g.Bk;
  t->ldbk = g.ldbk;
  t->bk_col0 = t->n0;
  t->col_base = t->n0;
  t->col_end = g.ncols;
  t->b_col_base = t->n0;
  t->plb = g.plb;
  t->pub = g.pub;
  t->rpart = g.rpart;
  t->rcol0 = t->n0;
  t->rcol_end = g.ncols;
  t->rchunk = nt;
  t->Kp = g.Kp;
  if (MAPPED && g.segs != nullptr) {
    const GemmSeg sg = g.segs[nt];
    t->rpart = sg.rpart;
    t->plb = sg.plb;
    t->pub = sg.pub;
    t->rcol0 = sg.col_local0;
    t->rcol_end = sg.col_local0 + sg.valid;
    t->rchunk = 0;
    t->kmap = sg.kmap;
    t->Kp = sg.kp;
    t->col_base = sg.col_base;
    t->col_end = sg.col_base + sg.valid;
    t->b_col_base = sg.b_col_base;
    t->Bk = sg.Bk;
    t->ldbk = sg.ldbk;
    t->bk_col0 = sg.col_local0;
  }
  return true;
}

// What both kernels do with a finished tile: the fused range sums, then the bias on column 0 and the stores.
// pbs: LDS, the predicate bounds of the tile's columns ([2][TN], zero where there is none); red: WC * TM * 4 doubles of LDS
// that nobody reads any more.
template <int TM, int TN, int WR, int WC, bool MAPPED>
__device__ __forceinline__ void gemm_finish(const GemmArgs& g, const GemmTile& t, double* red, const double (*pbs)[TN],
                                            double4_t (&acc)[TM / WR / 16][TN / WC / 16]) {
  constexpr int NT = 64 * WR * WC, FM = TM / WR / 16, FN = TN / WC / 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave % WR, wc = wave / WR;
  const int lrow = lane & 15, lcol = lane >> 4;
  double* C = g.C;
  int64_t ldc = g.ldc;
  const double* bias = g.bias;
  if (g.ksplit > 1) {  // partial sums go to the workspace (ld = Mp); bias is added by the reduction
    C = g.part + (int64_t)blockIdx.y * g.Mp * g.ncols;
    ldc = g.Mp;
    bias = nullptr;
  }
  // ---- fused estimateRanges: partial sums of this column tile ----------------------------------
  // xmin1 = sum max(v,0)*plb, xmin2 = sum min(v,0)*pub, xmax1 = sum max(v,0)*pub, xmax2 = sum min(v,0)*plb
  // over the tile's generator columns (column 0, the centre, is skipped), per output row.
  if (t.rpart != nullptr) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int ct = wc * (TN / WC) + j * 16 + lcol + 4 * r;
          const int64_t col = t.rcol0 + ct;
          if (col >= 1 && col < t.rcol_end) {
            const double v = acc[i][j][r];
            const double pl = pbs[0][ct], pu = pbs[1][ct];
            const double p = fmax(v, 0.0), q = fmin(v, 0.0);
            s0 = fma(p, pl, s0);
            s1 = fma(q, pu, s1);
            s2 = fma(p, pu, s2);
            s3 = fma(q, pl, s3);
          }
        }
      }
      // the four lane groups (lcol) hold different columns of the same rows
      s0 += __shfl_xor(s0, 16);
      s1 += __shfl_xor(s1, 16);
      s2 += __shfl_xor(s2, 16);
      s3 += __shfl_xor(s3, 16);
      s0 += __shfl_xor(s0, 32);
      s1 += __shfl_xor(s1, 32);
      s2 += __shfl_xor(s2, 32);
      s3 += __shfl_xor(s3, 32);
      if (lcol == 0) {
        double* dst = red + ((wc * TM) + wr * (TM / WR) + i * 16 + lrow) * 4;
        dst[0] = s0;
        dst[1] = s1;
        dst[2] = s2;
        dst[3] = s3;
      }
    }
    __syncthreads();
    for (int e = tid; e < TM * 4; e += NT) {  // waves along the columns are combined in order
      const int row = e >> 2, q = e & 3;
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < WC; ++w) s += red[(w * TM + row) * 4 + q];
      if (t.m0 + row < g.Mp) t.rpart[(t.rchunk * 4 + q) * ldc + t.m0 + row] = s;
    }
  }
  // ---- epilogue: bias on column 0, 128-byte line stores --------------------------------------
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int row = t.m0 + wr * (TM / WR) + i * 16 + lrow;
    if (row >= g.Mp) continue;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t ccol = t.col_base + wc * (TN / WC) + j * 16 + lcol + 4 * r;
        if (ccol < t.col_end) {
          double v = acc[i][j][r];
          if (bias != nullptr && ccol == 0) v = v + bias[row];
          // (partial products of a split go to the workspace column by column; the reduction maps them)
          C[row + ((MAPPED && g.colmap != nullptr && g.ksplit == 1) ? (int64_t)g.colmap[ccol] : ccol) * ldc] = v;
        }
      }
    }
  }
}

// This thread's entry of the predicate bounds of the tile's columns (the lower ones of all columns, then the upper ones).
template <int TN>
__device__ __forceinline__ double gemm_pred_bound(const GemmTile& t, int tid) {
  double v = 0.0;
  if (t.rpart != nullptr && tid < 2 * TN) {
    const int64_t col = t.rcol0 + tid % TN;
    if (col >= 1 && col < t.rcol_end) v = (tid < TN ? t.plb : t.pub)[col - 1];
  }
  return v;
}

constexpr int kMapLds = 2048;  // entries of a row list in LDS at a time
__device__ double g_zero_rows[128];  // what a padding entry of a row list reads in place of a column of A (never written)

// TM x TN output tile per block of WR x WC waves, each wave owning (TM/WR) x (TN/WC) = (16*FM) x (16*FN).
//
// What bounds it: fp64 MFMA, and where a CU has one tile or two the gaps between the products - every wave of a block
// waits for the same stage, and what a wave does between its last product of one stage and its first of the next (the wait,
// the barrier, the next transfers, address arithmetic, the first LDS reads) leaves the matrix cores idle.  So:
//  - Both operands travel global -> LDS directly (global_load_lds_dwordx4, no staging registers), KT rows of B a stage, S
//    stages in a ring; S - 1 of them are in flight while one is multiplied.
//  - Every wave brings the same number of transfers of each operand (UA, UB), so the loop has no branch on who brings what,
//    and a transfer's address is a scalar that advances plus a lane offset that does not.
//  - The loop is unrolled over the ring: LDS addresses are lane constants plus immediate offsets.
//  - Operands are read from LDS four rows ahead of the product they are for, over the end of a stage as well.
// 1024 x 784 over 480 and 1920 rows: 30 and 91 us with the operands staged through registers one stage ahead, 18 and 59 us
// now (32 x 64 tiles); 704 x 1501 over 1008 rows 74 -> 47 us; 2048 x 1024 over 1024 rows (64 x 64 tiles) 104 -> 77 us inside a reach;
// 70 TFLOP/s over 1920 rows, which is what the largest library product reaches here.
//
// A transfer (1 KB, a wave's 64 lanes x 16 bytes) of A holds whole rows k of the stage, lanes along the rows of W.  One of B
// holds the KT rows of 128 / KT columns; LDS takes its pieces in lane order, so lanes fetch the 16-byte pieces of a column in
// an order turned by the column's number, and the 16 lanes that read one row of 16 columns meet two to a bank pair instead
// of 16 to one.  The ring stays inside the first 64 KB of LDS.
//
// MAPPED = false: the plain product.  MAPPED = true additionally honours a row list (kmap) with packed rows of B (Bk), a
// per-tile segment table (segs) and a column map for C; kept apart so that the plain kernel pays nothing.
constexpr int kMaxLdaDma = 1 << 24, kMaxLdbDma = 1 << 22;  // leading dimensions whose lane offsets fit 32 bits
template <int TM, int TN, int WR, int WC, int KT, bool MAPPED>
__global__ __launch_bounds__(64 * WR * WC) void gemm_f64_kernel(GemmArgs g) {
  constexpr int NT = 64 * WR * WC, NW = WR * WC;
  constexpr int FM = TM / WR / 16, FN = TN / WC / 16;
  constexpr int kStage = KT * (TM + TN);
  constexpr int S = 65536 / (8 * kStage) > 4 ? 4 : 65536 / (8 * kStage);
  constexpr int UA = TM * KT / 128 / NW, UB = TN * KT / 128 / NW, U = UA + UB;
  static_assert(KT == 32, "stages of two groups of 16 rows");
  static_assert(S >= 2 && UA >= 1 && UB >= 1 && UA * NW * 128 == TM * KT && UB * NW * 128 == TN * KT, "every wave brings the same share of a stage");
  static_assert(WC * TM * 4 <= S * kStage && 2 * TN <= NT, "sums and bounds of the epilogue");
  // (rows 0 .. KT - 1 of A, less than lda entries into one; columns 0 .. TN - 1 of B, less than KT entries into one; packed rows of B
  // have no larger leading dimension than B)
  static_assert((uint64_t)KT * (kMaxLdaDma - 1) * 8 < (uint64_t(1) << 32) && ((uint64_t)(TN - 1) * (kMaxLdbDma - 1) + KT) * 8 < (uint64_t(1) << 32),
                "lane offsets of a stage");
  struct Lds {
    double ring[S * kStage];
    double pbs[2][TN];
    int kmap[MAPPED ? kMapLds : 1];
  };
  static_assert(kMapLds / 2 % NT == 0 && kMapLds / 2 % KT == 0, "halves of whole stages, whole passes of the block");
  __shared__ __attribute__((aligned(1024))) Lds sm;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  GemmTile t;
  if (!gemm_tile_of<TM, TN, MAPPED>(g, &t)) return;
  const double pb_reg = gemm_pred_bound<TN>(t, tid);
  const bool mapped = MAPPED && t.kmap != nullptr;  // uniform over the block
  // split-K: block row blockIdx.y owns the rows [k0, k0 + 16 * n16) and writes a partial product
  const int nk16 = t.Kp / 16;
  const int k16 = (int)((int64_t)nk16 * blockIdx.y / g.ksplit);
  const int n16 = (int)((int64_t)nk16 * (blockIdx.y + 1) / g.ksplit) - k16;
  const int k0 = k16 * 16;
  // The transfers' row numbers come from LDS: a load from the list in memory would have to be waited for, and with it all
  // transfers in flight.  (So would a choice between the two: it becomes one load that may go to either.)  Entry k of the
  // block's rows lies at k % kMapLds; a longer list goes through there half by half, the next half when nobody needs the place of
  // the last but one any more, which is the one such wait in kMapLds / 2 rows.  A lane reads its row numbers of a stage while
  // it issues the one before.  100 x 1900 rows over 1200 columns, 512 x 4275 over 300, 512 x 8550 over 1200: with the choice 53,
  // 135 and 536 us, from LDS alone 42, 89 and 387, read a stage ahead 36, 74 and 339.
  auto copy_list = [&](int from, int to) {  // entries of the block's rows; at most half of kMapLds
    constexpr int E = kMapLds / 2 / NT;
    const int32_t* const list = in_global(t.kmap) + k0;
    int v[E];
#pragma unroll
    for (int u = 0; u < E; ++u) v[u] = from + u * NT + tid < to ? list[from + u * NT + tid] : 0;
#pragma unroll
    for (int u = 0; u < E; ++u)
      if (from + u * NT + tid < to) sm.kmap[(from + u * NT + tid) % kMapLds] = v[u];
  };
  if (mapped) {
    copy_list(0, min(16 * n16, kMapLds / 2));
    copy_list(kMapLds / 2, min(16 * n16, kMapLds));
    __syncthreads();
  }
  auto next_half = [&](int k) {  // in front of the transfers of rows k ..., behind a barrier behind those of the rows before
    if (mapped && k != 0 && k % (kMapLds / 2) == 0) copy_list(k + kMapLds / 2, min(16 * n16, k + kMapLds));
  };
  const bool half = n16 & 1;  // the last stage has 16 rows
  const int nk = (n16 + 1) / 2;

  // This wave's transfers of a stage: rows ka + u * kAStep of A, columns cb + u * kBStep of B.  Rows of W past the last and
  // columns past the tile's end are read from its last rows and first column (such results are neither stored nor summed).
  constexpr int kAStep = NW * 128 / TM, kBStep = NW * 128 / KT;
  const int ka = wave * 128 / TM + lane / (TM / 2);
  const int ra = min(t.m0 + 2 * (lane % (TM / 2)), g.Mp - 2);
  const int cb = wave * 128 / KT + lane / (KT / 2);
  const int piece = (lane & (KT / 2 - 1)) ^ (cb & 7);  // (kBStep is a multiple of 16)
  const bool packed = MAPPED && t.Bk != nullptr;
  const int64_t ldb = packed ? t.ldbk : g.ldb;
  const double* a_base = g.A + (mapped ? 0 : (int64_t)k0 * g.lda);
  const double* b_base = (packed ? t.Bk + t.bk_col0 * ldb : g.B + t.b_col_base * ldb) + k0;
  const unsigned a_off = (unsigned)((ra + (mapped ? 0 : (int64_t)ka * g.lda)) * 8);
  unsigned b_col[UB];
#pragma unroll
  for (int u = 0; u < UB; ++u) b_col[u] = (unsigned)((t.col_base + cb + u * kBStep < t.col_end ? cb + u * kBStep : 0) * ldb * 8);
  const unsigned lds0 = lds_addr_of(sm.ring) + wave * 1024;
  const char* const a_row0 = reinterpret_cast<const char*>(g.A + ra);
  const uint32_t lda8 = (uint32_t)g.lda * 8;
  int a_row[UA];  // the listed rows that this lane's transfers of the stage to be issued next bring
  auto rows_of_stage = [&](int st) {
    const int rows = (half && st == nk - 1) ? 16 : KT;
#pragma unroll
    for (int u = 0; u < UA; ++u) a_row[u] = sm.kmap[(st * KT + min(ka + u * kAStep, rows - 1)) % kMapLds];
  };
  if (mapped) rows_of_stage(0);
  // Stage st into place `slot` of the ring; stages are issued in order.  The rows a half stage does not have are read from
  // its last one and not multiplied.
  auto issue = [&](int st, int slot) {
    const unsigned at = lds0 + slot * (kStage * 8);
    const int rows = (half && st == nk - 1) ? 16 : KT;
    if (mapped) {
#pragma unroll
      for (int u = 0; u < UA; ++u) {
        const char* const row = a_row0 + (uint64_t)(uint32_t)a_row[u] * lda8;
        lds_dma16_at(a_row[u] >= 0 ? reinterpret_cast<const double*>(row) : g_zero_rows + 2 * lane, at + u * (NW * 1024));
      }
      if (st + 1 < nk) rows_of_stage(st + 1);
    } else if (rows == KT) {
#pragma unroll
      for (int u = 0; u < UA; ++u) lds_dma16(a_base + (int64_t)u * kAStep * g.lda, a_off, at + u * (NW * 1024));
      a_base += KT * g.lda;
    } else {
#pragma unroll
      for (int u = 0; u < UA; ++u)
        lds_dma16(a_base, (unsigned)((ra + (int64_t)min(ka + u * kAStep, rows - 1) * g.lda) * 8), at + u * (NW * 1024));
    }
    const unsigned b_row = (unsigned)(rows == KT ? piece : min(piece, rows / 2 - 1)) * 16;
#pragma unroll
    for (int u = 0; u < UB; ++u) lds_dma16(b_base, b_col[u] + b_row, at + KT * TM * 8 + u * (NW * 1024));
    b_base += KT;
  };
  double4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int st = 0; st < S; ++st)
    if (st < nk) issue(st, st);

  const int wr = wave % WR, wc = wave / WR, l16 = lane & 15, q = lane >> 4;
  const int px = (q >> 1) ^ (l16 & 7);  // turns the piece that holds row q of a column
  // this wave's transfers of a stage have landed (those of `ahead` later ones may be in flight) and its LDS reads are done
  auto arrived = [&](int ahead) {
    if (S > 3 && ahead == 3) wait_vm_lds<3 * U>();
    else if (S > 2 && ahead == 2) wait_vm_lds<2 * U>();
    else if (ahead == 1) wait_vm_lds<U>();
    else wait_vm_lds<0>();
  };
  struct Frag {
    double b[FM], a[FN];
  };
  const double* as = sm.ring + wr * (TM / WR) + l16 + q * TM;
  const double* bs[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) bs[s] = sm.ring + KT * TM + (wc * (TN / WC) + l16) * KT + (q & 1) + 2 * ((2 * s) ^ px);
  auto read = [&](int slot, int s, Frag& f) {  // rows 4 s .. 4 s + 3 of a stage
#pragma unroll
    for (int i = 0; i < FM; ++i) f.b[i] = as[slot * kStage + s * 4 * TM + i * 16];
#pragma unroll
    for (int j = 0; j < FN; ++j) f.a[j] = bs[s & 3][slot * kStage + j * 16 * KT + (s >> 2) * 16];
  };
  auto multiply = [&](const Frag& f) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[j], f.b[i], acc[i][j], 0, 0, 0);
  };
  Frag f0, f1;
  arrived(min(nk, S) - 1);
  block_barrier();
  read(0, 0, f0);
  for (int st0 = 0; st0 < nk; st0 += S) {
#pragma unroll
    for (int slot = 0; slot < S; ++slot) {
      const int st = st0 + slot;
      if (st >= nk) break;
      const bool last = st == nk - 1;
#pragma unroll
      for (int s = 0; s < KT / 4; s += 2) {  // (the reads stay in front of the products they overlap)
        read(slot, s + 1, f1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f0);
        __builtin_amdgcn_sched_barrier(0);
        if (s + 2 == KT / 4 || (s == 2 && half && last)) break;
        read(slot, s + 2, f0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (!last) {
        arrived(min(nk - 2 - st, S - 2));
        block_barrier();  // stage st + 1 is there, and nobody reads stage st any more: its place takes the next transfers
        read((slot + 1) % S, 0, f0);
        if (st + S < nk) {
          next_half((st + S) * KT);
          issue(st + S, slot);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      multiply(f1);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (t.rpart != nullptr) {
    if (tid < 2 * TN) sm.pbs[tid / TN][tid % TN] = pb_reg;
    __syncthreads();  // everybody is done with the last stage; the bounds are in place
  }
  gemm_finish<TM, TN, WR, WC, MAPPED>(g, t, sm.ring, sm.pbs, acc);
}

// The same product where the rows of B are read through the row list (nobody packed them: products bound by their launch,
// and outputs of few rows, where packing would cost more than it saves), where the columns of B are picked by a map, and for
// matrices whose lane offsets do not fit 32 bits: 8-byte pieces and 64-bit addresses, through registers one stage ahead.
// Arrays (segs) may mix such tiles with packed ones.
template <int TM, int TN, int WR, int WC>
__global__ __launch_bounds__(64 * WR * WC) void gemm_gather_kernel(GemmArgs g) {
  constexpr int KT = 16;
  constexpr int NT = 64 * WR * WC;  // threads per block
  constexpr int FM = TM / WR / 16;
  constexpr int FN = TN / WC / 16;
  constexpr int LDA_S = TM + kPadRow;  // Ws[k][row]
  constexpr int LDB_S = KT + kPadK;    // Vs[col][k]
  __shared__ double Ws[2][KT * LDA_S];
  __shared__ double Vs[2][TN * LDB_S];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wr = wave % WR;
  const int wc = wave / WR;
  GemmTile t;
  if (!gemm_tile_of<TM, TN, true>(g, &t)) return;
  const double pb_reg = gemm_pred_bound<TN>(t, tid);
  const bool b_packed = t.Bk != nullptr;
  // The row list of this tile is copied into LDS first: the staging loads then take their row numbers
  // from there instead of through a dependent global load ahead of every operand load.
  __shared__ int kmap_s[kMapLds];
  __shared__ double pbs[2][TN];
  const bool map_lds = t.kmap != nullptr && t.Kp <= kMapLds;  // uniform over the block
  if (map_lds) {
    for (int k = tid; k < t.Kp; k += NT) kmap_s[k] = t.kmap[k];
    __syncthreads();
  }

  // ---- global -> register staging ----------------------------------------------------------
  constexpr int A_VEC = TM * KT / 2;           // double2 elements in a W tile
  constexpr int A_PASS = (A_VEC + NT - 1) / NT;
  constexpr int B_VEC = TN * KT / 2;
  constexpr int B_PASS = (B_VEC + NT - 1) / NT;
  double2 ra[A_PASS], rb[B_PASS];
  // column of B behind each staged element (-1: none)
  int64_t bcol[B_PASS];
#pragma unroll
  for (int p = 0; p < B_PASS; ++p) {
    const int64_t jl = (tid + p * NT) / (KT / 2);
    const int64_t col = t.col_base + jl;
    bcol[p] = col < t.col_end ? (g.bmap != nullptr ? (int64_t)g.bmap[col] : t.b_col_base + jl) : -1;
  }

  auto load_tiles = [&](int k0) {
#pragma unroll
    for (int p = 0; p < A_PASS; ++p) {
      int idx = tid + p * NT;
      int i2 = idx % (TM / 2);
      int k = idx / (TM / 2);
      int row = t.m0 + 2 * i2;
      double2 v = make_double2(0.0, 0.0);
      if (idx < A_VEC && row < g.Mp) {
        const int kk = t.kmap != nullptr ? (map_lds ? kmap_s[k0 + k] : t.kmap[k0 + k]) : k0 + k;
        if (kk >= 0) v = *reinterpret_cast<const double2*>(g.A + row + (int64_t)kk * g.lda);
      }
      ra[p] = v;
    }
#pragma unroll
    for (int p = 0; p < B_PASS; ++p) {
      int idx = tid + p * NT;
      int k2 = idx % (KT / 2);
      int j = idx / (KT / 2);
      double2 v = make_double2(0.0, 0.0);
      if (idx < B_VEC && bcol[p] >= 0) {
        if (b_packed) {
          v = *reinterpret_cast<const double2*>(t.Bk + (k0 + 2 * k2) + (t.bk_col0 + j) * t.ldbk);
        } else if (t.kmap != nullptr) {
          const int ka = map_lds ? kmap_s[k0 + 2 * k2] : t.kmap[k0 + 2 * k2];
          const int kb = map_lds ? kmap_s[k0 + 2 * k2 + 1] : t.kmap[k0 + 2 * k2 + 1];
          if (ka >= 0) v.x = g.B[ka + bcol[p] * g.ldb];
          if (kb >= 0) v.y = g.B[kb + bcol[p] * g.ldb];
        } else {
          v = *reinterpret_cast<const double2*>(g.B + (k0 + 2 * k2) + bcol[p] * g.ldb);
        }
      }
      rb[p] = v;
    }
  };
  auto store_tiles = [&](int buf) {
#pragma unroll
    for (int p = 0; p < A_PASS; ++p) {
      int idx = tid + p * NT;
      int i2 = idx % (TM / 2);
      int k = idx / (TM / 2);
      if (idx < A_VEC) *reinterpret_cast<double2*>(&Ws[buf][k * LDA_S + 2 * i2]) = ra[p];
    }
#pragma unroll
    for (int p = 0; p < B_PASS; ++p) {
      int idx = tid + p * NT;
      int k2 = idx % (KT / 2);
      int j = idx / (KT / 2);
      if (idx < B_VEC) {  // odd column stride: two 64-bit stores
        Vs[buf][j * LDB_S + 2 * k2] = rb[p].x;
        Vs[buf][j * LDB_S + 2 * k2 + 1] = rb[p].y;
      }
    }
  };

  double4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};

  // split-K: block row blockIdx.y owns the K-tiles [kt0, kt1) and writes a partial product
  const int nk_all = t.Kp / KT;
  const int kt0 = (int)((int64_t)nk_all * blockIdx.y / g.ksplit);
  const int kt1 = (int)((int64_t)nk_all * (blockIdx.y + 1) / g.ksplit);
  // two LDS stages: tile t+1 travels global -> registers while tile t is multiplied, then goes to the
  // other stage; one barrier per K-tile
  const int nk = kt1 - kt0;
  load_tiles(kt0 * KT);
  store_tiles(0);
  __syncthreads();
  for (int st = 0; st < nk; ++st) {
    const int cur = st & 1;
    if (st + 1 < nk) load_tiles((kt0 + st + 1) * KT);
    mfma_tile_k16<FM, FN, KT>(&Ws[cur][wr * (TM / WR)], LDA_S, &Vs[cur][(wc * (TN / WC)) * LDB_S], LDB_S, lane, acc);
    if (st + 1 < nk) store_tiles(cur ^ 1);
    __syncthreads();
  }
  if (t.rpart != nullptr) {
    if (tid < 2 * TN) pbs[tid / TN][tid % TN] = pb_reg;
    __syncthreads();
  }
  gemm_finish<TM, TN, WR, WC, true>(g, t, &Ws[0][0], pbs, acc);
}

// colmap (or null): column t of the partial products belongs at column colmap[t] of C.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const double* __restrict__ part, int ksplit, int Mp,
                                                             int64_t ncols, double* __restrict__ C, int64_t ldc,
                                                             const double* __restrict__ bias,
                                                             const int32_t* __restrict__ colmap) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t total = (int64_t)Mp * ncols;
  if (t >= total) return;
  double s = 0.0;
  for (int k0 = 0; k0 < ksplit; k0 += 16) {  // sixteen loads in flight, added in split order
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = k0 + u < ksplit ? part[(int64_t)(k0 + u) * total + t] : 0.0;
#pragma unroll
    for (int u = 0; u < 16; ++u)
      if (k0 + u < ksplit) s += v[u];
  }
  const int64_t col = t / Mp;
  const int row = (int)(t - col * Mp);
  if (bias != nullptr && col == 0) s = s + bias[row];
  C[row + (colmap != nullptr ? (int64_t)colmap[col] : col) * ldc] = s;
}

template <int TM, int TN, int WR, int WC, int KT, bool GATHER = false>
static int launch_cfg(nnvhip_ctx* ctx, const double* A, int64_t lda, const double* B, int64_t ldb, double* C,
                      int64_t ldc, int64_t Mp, int64_t ncols, int64_t Kp, const double* bias, RangeFuse* fuse,
                      const GemmRows* rows, SplitKDefer* defer) {
  int64_t tiles_m = ceil_div(Mp, TM);
  int64_t tiles_n = ceil_div(ncols, TN);
  int64_t blocks = tiles_m * tiles_n;
  if (blocks >= (int64_t(1) << 28)) NNV_FAIL(NNVHIP_ERR_SHAPE, "matrix too large for one launch");
  // XCD grid xr x (8/xr): least HBM/fabric traffic (8/xr)*|W| + xr*|V| among the shapes whose
  // busiest XCD has (almost) the fewest tiles
  int64_t best_xr = 8, best_slots = 0;
  double best_cost = 0.0;
  for (int64_t xr = 1; xr <= 8; xr *= 2) {
    const int64_t slots = ceil_div(tiles_m, xr) * ceil_div(tiles_n, 8 / xr);
    const double traffic = (8.0 / xr) * (double)Mp * Kp + (double)xr * Kp * (double)ncols;
    // an XCD has 32 CUs: up to 32 tiles per XCD still run in one round, so small imbalances are free
    const int64_t eff_slots = slots < 128 ? ceil_div(slots, 32) * 32 : slots;
    const double cost = (double)eff_slots * (1.0 + 0.03 * traffic / ((double)Mp * Kp + (double)Kp * ncols) / 8.0);
    if (best_slots == 0 || cost < best_cost) {
      best_cost = cost;
      best_xr = xr;
      best_slots = slots;
    }
  }
  if (const int v = tune_knobs().gemm_xr) {
    best_xr = std::max(1, std::min(8, v));
    best_slots = ceil_div(tiles_m, best_xr) * ceil_div(tiles_n, 8 / best_xr);
  }
  const int64_t local_m = ceil_div(tiles_m, best_xr);
  const int64_t grid_x = 8 * best_slots;
  // Split-K when the output has too few tiles to occupy the chip: partial products into a workspace,
  // summed in split order by a second kernel (deterministic, no floating-point atomics).
  const int64_t nk = Kp / 16;
  int64_t ksplit = 1;
  // From 128 tiles on, one to a CU, that is worth its second kernel and the range sums that are no longer formed along the way only
  // where the rows are listed (a stage then takes half as long again) and many for a tile's size.  Product and ReLU step behind it,
  // in one part and in three: 100 x 950 rows over 1200 columns 56 us, 56; 100 x 1615 67, 60; 512 x 1900 over 300 68, 61; 512 x 4275
  // 109, 82; 512 x 8550 180, 118; 1024 x 1900 over 300 (32 x 64 tiles) 81, 85; 1024 x 4275 136, 132; all rows of 200 x 2100 over 700
  // 56, 61.
  if (blocks < 128 && nk >= 8)
    ksplit = std::min<int64_t>(std::min<int64_t>(16, nk / 4), ceil_div(512, blocks));
  else if (rows != nullptr && rows->kmap != nullptr && blocks < 256 && 2 * Kp >= 3 * TM * TN)
    ksplit = 512 / blocks;
  if (const int v = tune_knobs().gemm_ksplit) ksplit = std::max<int64_t>(1, std::min<int64_t>(v, nk));
  // the split-K workspace is laid out for one plain column range: no segment tables (a column map is
  // applied by the reduction)
  if (rows != nullptr && rows->segs != nullptr) ksplit = 1;
  if (rows != nullptr && rows->colmap != nullptr && defer != nullptr) ksplit = 1;
  if (rows != nullptr && rows->segs != nullptr && rows->seg_cols != TN)
    NNV_FAIL(NNVHIP_ERR_ARG, "internal: segment table built for another tile width");
  BufRef ws;
  if (ksplit > 1) NNV_TRY(ctx->alloc(sizeof(double) * ksplit * Mp * ncols, &ws));
  double* rpart = nullptr;
  if (fuse != nullptr && ksplit == 1) {  // the epilogue sees final values: fuse the range sums
    NNV_TRY(ctx->alloc(sizeof(double) * 4 * ldc * (tiles_n + fuse->extra_chunks), &fuse->part));
    fuse->chunks = tiles_n;
    rpart = fuse->part->as<double>();
  }
  const bool timed = ctx->kernel_timing && Mp > 32;
  NNV_TRY(ctx->kernel_timer_begin(timed));
  GemmArgs g{};
  g.A = A;
  g.B = B;
  g.C = C;
  g.bias = bias;
  g.part = ws ? ws->as<double>() : nullptr;
  g.plb = fuse ? fuse->plb : nullptr;
  g.pub = fuse ? fuse->pub : nullptr;
  g.rpart = rpart;
  g.lda = lda;
  g.ldb = ldb;
  g.ldc = ldc;
  g.ncols = ncols;
  g.Mp = (int32_t)Mp;
  g.Kp = (int32_t)Kp;
  g.tiles_m = (int32_t)tiles_m;
  g.tiles_n = (int32_t)tiles_n;
  g.xr = (int32_t)best_xr;
  g.local_m = (int32_t)local_m;
  g.ksplit = (int32_t)ksplit;
  const dim3 grid((unsigned)grid_x, (unsigned)ksplit), block(64 * WR * WC);
  if (rows != nullptr) {
    g.kmap = rows->kmap;
    g.segs = rows->segs;
    g.colmap = rows->colmap;
    g.bmap = rows->b_plain ? nullptr : rows->colmap;
    g.Bk = rows->Bk;
    g.ldbk = rows->ldbk;
  }
  if constexpr (GATHER)
    NNV_LAUNCH(ctx, timed, (gemm_gather_kernel<TM, TN, WR, WC>), grid, block, 0, g);
  else if (rows != nullptr)
    NNV_LAUNCH(ctx, timed, (gemm_f64_kernel<TM, TN, WR, WC, KT, true>), grid, block, 0, g);
  else
    NNV_LAUNCH(ctx, timed, (gemm_f64_kernel<TM, TN, WR, WC, KT, false>), grid, block, 0, g);
  NNV_TRY(ctx->kernel_timer_end(timed, 0, rows && rows->flop > 0.0 ? rows->flop : 2.0 * (double)Mp * (double)Kp * (double)ncols));
  if (defer != nullptr) {
    defer->ws = ws;
    defer->ksplit = ksplit;
  } else if (ksplit > 1) {
    const int64_t total = Mp * ncols;
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, ctx->stream,
                       ws->as<double>(), (int)ksplit, (int)Mp, ncols, C, ldc, bias, rows ? rows->colmap : nullptr);
  }
  NNV_HIP_TRY(hipGetLastError());
  return NNVHIP_OK;
}

// Tile width of an array's launch by the kernels that take wide tiles (gemm_seg.hip, and products whose rows are read through a list):
// 128 columns when there are enough tiles to cover the chip, 64 for small arrays and outputs of few rows.
int gemm_seg_cols(int64_t Mp, int64_t count, const int64_t* cols) {
  if (Mp <= 32) return 64;
  int64_t tiles = 0;
  for (int64_t i = 0; i < count; ++i) tiles += ceil_div(cols[i], 128);
  return tiles * ceil_div(Mp, 128) < 256 ? 64 : 128;
}

int launch_gemm(nnvhip_ctx* ctx, const double* A, int64_t lda, const double* B, int64_t ldb, double* C, int64_t ldc,
                int64_t Mp, int64_t ncols, int64_t Kp, const double* bias, RangeFuse* fuse, const GemmRows* rows,
                SplitKDefer* defer) {
  if (Mp % 16 || Kp % 16 || lda % 2 || ldb % 2 || Mp > lda || Kp > ldb || Mp > ldc)
    NNV_FAIL(NNVHIP_ERR_SHAPE, "internal: GEMM operands violate the padding contract");
  if (Mp >= (int64_t(1) << 31) || Kp >= (int64_t(1) << 31)) NNV_FAIL(NNVHIP_ERR_SHAPE, "matrix too large");
  if (ncols == 0) return NNVHIP_OK;
#define NNV_GEMM(TM, TN, WR, WC, KT) launch_cfg<TM, TN, WR, WC, KT>(ctx, A, lda, B, ldb, C, ldc, Mp, ncols, Kp, bias, fuse, rows, defer)
#define NNV_GEMM_GATHER(TM, TN, WR, WC) \
  launch_cfg<TM, TN, WR, WC, 16, true>(ctx, A, lda, B, ldb, C, ldc, Mp, ncols, Kp, bias, fuse, rows, defer)
  const int64_t kCUs = 256;
  const bool wide_seg = rows != nullptr && rows->segs != nullptr && rows->seg_cols != 64;
  bool gather = lda >= kMaxLdaDma || ldb >= kMaxLdbDma;
  if (rows != nullptr)
    gather = gather || rows->gathered || (rows->segs == nullptr && rows->kmap != nullptr && rows->Bk == nullptr) ||
             (rows->colmap != nullptr && !rows->b_plain);
  if (gather) {
    if (Mp <= 16) return NNV_GEMM_GATHER(16, 64, 1, 4);
    if (wide_seg) return NNV_GEMM_GATHER(128, 128, 2, 4);
    // (2^24 rows of W, 16 and 64 columns of it, over 130 columns: 8.9 and 15.2 ms; on 128 x 128 tiles 13.0 and 22.9)
    return NNV_GEMM_GATHER(64, 64, 2, 4);
  }
  if (Mp <= 16) return NNV_GEMM(16, 64, 1, 4, 32);
  if (wide_seg) NNV_FAIL(NNVHIP_ERR_ARG, "internal: segment table built for another kernel");
  // (an array's tiles: 20 sets of 601 columns, 300 x 2627 rows each, 397 us; with 64 x 128 tiles 500, 128 x 128 from registers 915)
  if (rows != nullptr && rows->segs != nullptr) return Mp <= 32 ? NNV_GEMM(32, 64, 2, 4, 32) : NNV_GEMM(64, 64, 4, 2, 32);
  // The tiles of a launch are dealt evenly to the CUs and those of a CU share its matrix cores, so the time goes with
  // ceil(tiles / CUs) * tile area / rate.  The rates are those of a 2048 x 1024 x 1920 product; a CU with a single 64 x 64
  // tile has nothing to fill the gaps between its stages with.  Measured (1920 rows, in this order): 1024 x 784 63.6, 59.1,
  // 69.0 us; 704 x 1501 113, 85.5, 84.6; 512 x 500 60, 32.5, 21.9; 1024 x 3000 169.5, 168.3, 197.9.  (With operands that are
  // not in the caches yet the smallest tile, which reads them most often, falls behind: its rate is set for that.)
  struct Shape {
    int tm, tn;
    double rate, rate_alone;  // TFLOP/s
  };
  static const Shape shapes[] = {{64, 64, 70.0, 64.0}, {32, 64, 67.0, 64.0}, {32, 32, 52.0, 45.0}};
  int best = 0;
  double best_cost = 0.0;
  for (int i = 0; i < (int)(sizeof(shapes) / sizeof(shapes[0])); ++i) {
    const int64_t tiles = ceil_div(Mp, shapes[i].tm) * ceil_div(ncols, shapes[i].tn);
    const double cost = (double)ceil_div(tiles, kCUs) * shapes[i].tm * shapes[i].tn / (tiles <= kCUs ? shapes[i].rate_alone : shapes[i].rate);
    if (i == 0 || cost < best_cost * 0.999) {
      best = i;
      best_cost = cost;
    }
  }
  if (!tune_knobs().gemm_tile.empty()) {  // tuning knob: "TMxTN" of one of the shapes above
    for (int i = 0; i < (int)(sizeof(shapes) / sizeof(shapes[0])); ++i)
      if (std::to_string(shapes[i].tm) + "x" + std::to_string(shapes[i].tn) == tune_knobs().gemm_tile) best = i;
  }
  switch (best) {
    case 0: return NNV_GEMM(64, 64, 4, 2, 32);
    case 1: return NNV_GEMM(32, 64, 2, 4, 32);
    default: return NNV_GEMM(32, 32, 2, 2, 32);
  }
#undef NNV_GEMM_GATHER
#undef NNV_GEMM
}

// Packs the listed rows of every set's leading columns: Vk(t, j) = V(kept[t], j), zero where kept[t] < 0.
// Lane = two packed rows, the waves of a block interleave columns.  Grid: (row blocks of 128, column
// chunks, sets).
__global__ __launch_bounds__(512) void pack_rows_kernel(const PackSet* __restrict__ table, PackSet one, int cols_per_chunk) {
  const PackSet d = table ? table[blockIdx.z] : one;
  const int j0 = blockIdx.y * cols_per_chunk;
  if (j0 >= d.ncols) return;
  const int j1 = min(d.ncols, j0 + cols_per_chunk);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t0 = blockIdx.x * 128 + 2 * lane;
  if (t0 >= d.kp) return;
  const int ra = d.kept[t0], rb = d.kept[t0 + 1];
  // image positions of the two rows, for columns that are only defined inside their windows
  int ha = 0, wa = 0, hb = 0, wb = 0;
  if (d.box != nullptr) {
    const int P = d.bH * d.bW;
    const int pa = max(ra, 0) % P, pb = max(rb, 0) % P;
    wa = pa / d.bH, ha = pa - wa * d.bH;
    wb = pb / d.bH, hb = pb - wb * d.bH;
  }
  for (int jb = j0 + 4 * wave; jb < j1; jb += 32) {
    double2 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      v[u] = make_double2(0.0, 0.0);
      const int j = jb + u;
      if (j < j1 && !(j >= 1 && j < d.zero_to)) {
        if (d.W != nullptr && j >= d.wfrom && j < d.wend) {  // the value the gather pass wrote, recomputed
          const int src = d.widx[j - d.wfrom];
          const double sc = d.wscale ? d.wscale[src] : 1.0;
          const double* col = d.W + (int64_t)src * d.ldw;
          if (ra >= 0) v[u].x = __dadd_rn(0.0, __dmul_rn(col[ra], sc));
          if (rb >= 0) v[u].y = __dadd_rn(0.0, __dmul_rn(col[rb], sc));
        } else {
          const double* col = d.V + (int64_t)j * d.ld;
          bool ina = ra >= 0, inb = rb >= 0;
          if (d.box != nullptr && j >= d.box_from && j < d.box_to) {
            const ColBox b = d.box[j];
            ina = ina && ha >= b.h0 && ha <= b.h1 && wa >= b.w0 && wa <= b.w1;
            inb = inb && hb >= b.h0 && hb <= b.h1 && wb >= b.w0 && wb <= b.w1;
          }
          if (ina) v[u].x = col[ra];
          if (inb) v[u].y = col[rb];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (jb + u < j1) *reinterpret_cast<double2*>(d.Vk + t0 + (int64_t)(jb + u) * d.kp) = v[u];
  }
}

PackSet pack_of(const nnvhip_star* s, const int32_t* kept, double* dst, int64_t kp, int64_t ncols) {
  PackSet p{s->V, kept, dst, s->ld, (int32_t)kp, (int32_t)ncols};
  const ColSource& cs = s->cs;
  if (cs.W != nullptr && cs.from < ncols) {
    p.W = cs.W;
    p.ldw = cs.ldw;
    p.Wt = cs.Wt;
    p.ldwt = cs.ldwt;
    p.wrows = cs.rows;
    p.widx = cs.idx;
    p.wscale = cs.scale;
    p.wfrom = (int32_t)cs.from;
    p.wend = (int32_t)std::min<int64_t>(ncols, cs.from + cs.cols);
  }
  p.zero_to = (int32_t)std::min<int64_t>(ncols, cs.zero_to);
  if (cs.win_pending() && cs.win_from < ncols) {
    p.box = cs.win_box;
    p.box_from = (int32_t)cs.win_from;
    p.box_to = (int32_t)std::min<int64_t>(ncols, cs.win_to);
    p.bH = cs.win_H;
    p.bW = cs.win_W;
  }
  return p;
}

int launch_pack_rows(nnvhip_ctx* ctx, int64_t count, const PackSet* sets) {
  if (count <= 0) return NNVHIP_OK;
  if (count > 65535) NNV_FAIL(NNVHIP_ERR_SHAPE, "at most 65535 sets per call");
  int64_t max_kp = 0, max_cols = 0;
  for (int64_t i = 0; i < count; ++i) {
    max_kp = std::max<int64_t>(max_kp, sets[i].kp);
    max_cols = std::max<int64_t>(max_cols, sets[i].ncols);
  }
  if (max_kp == 0 || max_cols == 0) return NNVHIP_OK;
  const int64_t row_blocks = ceil_div(max_kp, 128);
  int64_t chunks = std::max<int64_t>(1, std::min<int64_t>(ceil_div(8192, row_blocks * count), ceil_div(max_cols, 32)));
  const int64_t cpc = ceil_div(max_cols, chunks);
  chunks = ceil_div(max_cols, cpc);
  const PackSet* table = nullptr;
  BufRef tab;
  if (count > 1) {
    NNV_TRY(ctx->upload_table(sets, sizeof(PackSet) * count, &tab));
    table = tab->as<PackSet>();
  }
  hipLaunchKernelGGL(pack_rows_kernel, dim3((unsigned)row_blocks, (unsigned)chunks, (unsigned)count), dim3(512), 0, ctx->stream,
                     table, sets[0], (int)cpc);
  NNV_HIP_TRY(hipGetLastError());
  return NNVHIP_OK;
}

__global__ void bias_columns_kernel(double* const* __restrict__ cols, const double* __restrict__ bias, int Mp) {
  double* col = cols[blockIdx.y];
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < Mp) col[r] = col[r] + bias[r];
}

int launch_bias_columns(nnvhip_ctx* ctx, double* const* centre_cols_dev, int64_t count, const double* bias,
                        int64_t Mp) {
  if (count <= 0) return NNVHIP_OK;
  for (int64_t off = 0; off < count; off += 65535) {
    int64_t n = std::min<int64_t>(65535, count - off);
    hipLaunchKernelGGL(bias_columns_kernel, dim3((unsigned)ceil_div(Mp, 256), (unsigned)n), dim3(256), 0, ctx->stream,
                       centre_cols_dev + off, bias, (int)Mp);
  }
  NNV_HIP_TRY(hipGetLastError());
  return NNVHIP_OK;
}

}  // namespace nnvhip
