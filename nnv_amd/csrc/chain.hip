// A whole reach of a small fully connected network in ONE launch: one 1024-thread block per input set
// walks the layer list of NN.reach_noConns (nn/NN.m:1529-1551) -- Star.affineMap (set/Star.m:313-343),
// Star.estimateRanges (set/Star.m:1078-1106) and the relax-star ReLU step at relaxFactor = 1
// (nn/funcs/PosLin.m:863-1650, 685-742; set/Star.m:1442-1461) -- and writes every layer's output set
// into buffers sized for the worst case (every neuron of every ReLU layer crossing).
//
// Networks of this size (tens of neurons per layer; an ACAS-Xu-shaped network is the type) are bound by
// the latency of a launch per layer step and of a host wait per ReLU on the layer-by-layer path; here the
// crossing counts never leave the block, the host reads them once at the end and only to fill in the
// handles.  Arrays of input sets (a branch-and-bound front over such a network) take one block each.
//
// The arithmetic is the layer kernels' (products accumulated in ascending row order from +0, the bias added
// last, lb = (c + xmin1) + xmin2), but sums are cut differently from the tiled kernels, so values agree with
// the layer-by-layer path to rounding, not bit for bit.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>

#include "internal.h"
#include "lds_dma.h"
#include "mfma_tile.h"
#include "relu_sort.h"

namespace nnvhip {

constexpr int kChainMaxLayers = 32;
constexpr int kChainThreads = 1024;
constexpr int kChainMaxN = 512;  // widest layer (the block's LDS holds a few vectors of that length)

struct ChainLayer {
  const double* W;     // fc: M rows (padded to ldw) x K, column-major
  const double* bias;  // fc: or null
  int32_t kind;        // NNVHIP_LAYER_FC / NNVHIP_LAYER_RELU
  int32_t M;           // dimension of the layer's output
  int32_t K;           // fc: columns of W
  int32_t ldw;
  int32_t ld;          // leading dimension of the output matrix
  int32_t npad;        // relu: padded worst-case number of predicates of the output
  // offsets (in doubles) into the set's slice of the arena
  int64_t v_off;       // the output matrix
  int64_t rng_off;     // lb[ld], ub[ld]: estimated ranges of the output (fc) / of the input when the layer before left none (relu)
  int64_t pred_off;    // relu: plb[npad], pub[npad]
  int64_t lbub_off;    // relu: lb[ld], ub[ld] of the crossing neurons in new-predicate order
  int64_t idx_off;     // relu, in ints, into the set's slice of the index arena: cross[ld], keep[ld + 16]
};

struct ChainSet {
  const double* V;    // the input set, fully in memory - or, with idx, a box of which only the centre is (the first layer
  const double* plb;  // is an FC layer then): column 1 + t is scale[idx[t]] at row idx[t]
  const double* pub;
  const int32_t* idx;
  const double* scale;
  int64_t ld;
  int32_t N, n;
};

struct ChainArgs {
  ChainLayer layers[kChainMaxLayers];
  int32_t n_layers;
  int32_t order;
  double* arena;
  int64_t set_stride;
  int32_t* iarena;
  int64_t iset_stride;
  int32_t* counts;     // [set][layer][2]: crossing, inactive (zero for fc layers)
  int32_t* mailbox;    // host-pinned words, [relu ordinal * sets + set], or null
  int32_t mailbox_seq;
  int32_t n_sets;
};

// lb / ub of the N x (n+1) matrix V over the predicate box, 16 lanes per row (each lane takes every
// sixteenth generator in ascending order, then a fixed tree over the 16), into LDS and global memory.
// Only for a ReLU layer whose input did not come out of an FC layer of the same launch.
__device__ __forceinline__ void chain_ranges(const double* __restrict__ V, int ld, int N, int n, const double* __restrict__ plb,
                                             const double* __restrict__ pub, double* s_lb, double* s_ub, double* g_rng, int tid) {
  const int q = tid & 15;
  for (int r0 = 0; r0 < N; r0 += kChainThreads / 16) {
    const int i = r0 + (tid >> 4);
    double x1 = 0.0, x2 = 0.0, y1 = 0.0, y2 = 0.0;
    if (i < N) {
      for (int j = 1 + q; j <= n; j += 16) {
        const double v = V[i + (int64_t)j * ld];
        const double pl = plb[j - 1], pu = pub[j - 1];
        const double vp = fmax(v, 0.0), vn = fmin(v, 0.0);
        x1 = fma(vp, pl, x1);  // xmin1
        x2 = fma(vn, pu, x2);  // xmin2
        y1 = fma(vp, pu, y1);  // xmax1
        y2 = fma(vn, pl, y2);  // xmax2
      }
    }
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) {
      x1 += __shfl_xor(x1, off);
      x2 += __shfl_xor(x2, off);
      y1 += __shfl_xor(y1, off);
      y2 += __shfl_xor(y2, off);
    }
    if (q == 0 && i < N) {
      const double c = V[i];
      const double lb = (c + x1) + x2;  // set/Star.m:1098-1104, left to right
      const double ub = (c + y1) + y2;
      s_lb[i] = lb;
      s_ub[i] = ub;
      g_rng[i] = lb;
      g_rng[ld + i] = ub;
    }
  }
  __syncthreads();
}

// Barrier for data exchanged through LDS only: waits for the wave's LDS operations, not for its global stores
// (__syncthreads would also sit out the round trip of every store still in flight).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Scratch in LDS that the phases of a layer share: the sort stages its keys here, the FC phase its range sums.
struct ChainScratch {
  union {
    struct {
      double key[kChainMaxN];
      int idx[kChainMaxN];
      int rank[kChainMaxN];
    } sort;
    struct {
      double part[4][kChainMaxN];  // [sum][column group * ld + row]: range sums of the contracted columns per column group of waves
      double gat[2][kChainMaxN];   // S+ / S- of the gathered columns, by row
      double cen[kChainMaxN];      // the centre column
    } fc;
  };
};

__global__ __launch_bounds__(kChainThreads) void reach_chain_kernel(const ChainSet* __restrict__ sets, ChainSet one, ChainArgs a) {
  __shared__ double s_lb[kChainMaxN], s_ub[kChainMaxN];
  __shared__ ChainScratch sc;
  __shared__ int s_keep[kChainMaxN];
  __shared__ int s_cross[kChainMaxN];
  __shared__ int s_cls[kChainMaxN];
  __shared__ int4 wcnt[4];  // per wave: crossing | inactive << 10 | kept << 20 (each at most 64)
  __shared__ int s_counts[2 * kChainMaxLayers];
  const ChainSet S = sets ? sets[blockIdx.x] : one;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double* A = a.arena + (int64_t)blockIdx.x * a.set_stride;
  int32_t* IA = a.iarena + (int64_t)blockIdx.x * a.iset_stride;
  int32_t* counts = a.counts + (int64_t)blockIdx.x * a.n_layers * 2;

  const double* V = S.V;        // the current set's matrix ...
  const double* Vsrc = S.V;     // ... and where an FC layer reads its kept rows from (a ReLU output: the ReLU's input,
  int ld = (int)S.ld, N = S.N, n = S.n;  // whose kept rows are the same values and were written a layer earlier)
  const double* plb = S.plb;
  const double* pub = S.pub;
  const double* plb_s = S.plb;  // likewise the bounds of the predicates in front of the ones a ReLU layer appended: the
  const double* pub_s = S.pub;  // ReLU's input holds the same values, written a layer earlier
  bool have_rng = false;        // s_lb / s_ub hold the ranges of V
  int n_keep = -1;              // >= 0: V is a ReLU output; its rows s_keep[0..n_keep) are the ones not reset,
  int oh_from = 0;              //       and its columns from oh_from on are the unit vectors of s_cross
  int relu_ord = 0;

  // every layer's weights are asked for once up front (one 128-byte line per thread and step), so that the
  // layers find them in the cache instead of each paying a trip to memory
  for (int l = 1; l < a.n_layers; ++l) {
    const ChainLayer& L = a.layers[l];
    if (L.kind != NNVHIP_LAYER_FC) continue;
    const int lines = (L.ldw * L.K) / 16;
    for (int t = tid; t < lines; t += kChainThreads) {
      const double w = L.W[(int64_t)t * 16];
      asm volatile("" ::"v"(w));
    }
  }

  for (int l = 0; l < a.n_layers; ++l) {
    const ChainLayer& L = a.layers[l];
    if (L.kind == NNVHIP_LAYER_FC) {
      // ---- Star.affineMap on the matrix cores, 16 x 16 output tiles, one wave each.  Operand layout of
      // v_mfma_f64_16x16x4_f64: lane l supplies a[i = l%16][k = l/16] (a column of V) and b[k = l/16][j = l%16]
      // (16 consecutive rows of W); result register r of lane l is out[row = l%16][column = l/16 + 4r].
      // The contraction runs over the kept rows only (reset rows hold +0) and over the columns in front of the
      // appended unit vectors; every wave keeps the four range sums of its rows over its columns.
      double* O = A + L.v_off;
      const int ldo = L.ld, ldw = L.ldw;
      const int R = ldo / 16;
      const int nd = n_keep >= 0 ? oh_from : n + 1;
      const int CT = (nd + 15) / 16;
      const int Kk = n_keep >= 0 ? n_keep : L.K;
      int RW = 1;
      while (RW * 2 <= min(R, 16)) RW *= 2;
      const int WC = 16 / RW;  // WC * ldo <= kChainMaxN (RW > R / 2, or WC = 1)
      const int wr = wave % RW, wc = wave / RW;
      const int l16 = lane & 15, kq = lane >> 4;
      for (int tr = wr; tr < R; tr += RW) {
        const int row = tr * 16 + l16;
        const double* wrow = L.W + row;
        double x1 = 0.0, x2 = 0.0, y1 = 0.0, y2 = 0.0;
        for (int tc = wc; tc < CT; tc += WC) {
          const int col_a = tc * 16 + l16;  // the column this lane feeds
          const bool col_ok = col_a < nd;
          const bool box = l == 0 && S.idx != nullptr;  // (uniform)
          const double* vcol = Vsrc + (int64_t)(col_ok && !box ? col_a : 0) * ld;
          int hot = -1;  // a box's generator column: its one row and the value there
          double hot_v = 0.0;
          if (box && col_ok && col_a > 0) {
            hot = S.idx[col_a - 1];
            hot_v = S.scale[hot];
          }
          double pl[4], pu[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {  // predicate bounds of the lane's four result columns
            const int col = tc * 16 + kq + 4 * r;
            pl[r] = pu[r] = 0.0;
            if (col >= 1 && col < nd) {
              pl[r] = plb_s[col - 1];
              pu[r] = pub_s[col - 1];
            }
          }
          const double bias0 = (tc == 0 && kq == 0 && L.bias != nullptr) ? L.bias[row] : 0.0;
          double4_t acc = {0.0, 0.0, 0.0, 0.0};
          for (int k0 = 0; k0 < Kk; k0 += 32) {  // eight MFMA steps per round, their loads issued first
            double av[8], bv[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              const int k = k0 + 4 * u + kq;
              av[u] = 0.0;
              bv[u] = 0.0;
              if (k < Kk) {
                const int kk = n_keep >= 0 ? s_keep[k] : k;
                bv[u] = wrow[(int64_t)kk * ldw];
                if (hot >= 0) av[u] = kk == hot ? hot_v : 0.0;
                else if (col_ok) av[u] = vcol[kk];
              }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bv[u], acc, 0, 0, 0);
          }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int col = tc * 16 + kq + 4 * r;
            if (col >= nd) continue;
            double v = acc[r];
            if (col == 0) {
              v = v + bias0;  // newV(:,1) = newV(:,1) + b
              sc.fc.cen[row] = v;
            } else {
              const double vp = fmax(v, 0.0), vn = fmin(v, 0.0);
              x1 = fma(vp, pl[r], x1);  // xmin1
              x2 = fma(vn, pu[r], x2);  // xmin2
              y1 = fma(vp, pu[r], y1);  // xmax1
              y2 = fma(vn, pl[r], y2);  // xmax2
            }
            O[row + (int64_t)col * ldo] = v;  // rows [M, ld): W's padding rows are zero
          }
        }
        // the four lane groups hold different columns of the same rows
        x1 += __shfl_xor(x1, 16);
        x2 += __shfl_xor(x2, 16);
        y1 += __shfl_xor(y1, 16);
        y2 += __shfl_xor(y2, 16);
        x1 += __shfl_xor(x1, 32);
        x2 += __shfl_xor(x2, 32);
        y1 += __shfl_xor(y1, 32);
        y2 += __shfl_xor(y2, 32);
        if (kq == 0) {
          sc.fc.part[0][wc * ldo + row] = x1;
          sc.fc.part[1][wc * ldo + row] = x2;
          sc.fc.part[2][wc * ldo + row] = y1;
          sc.fc.part[3][wc * ldo + row] = y2;
        }
      }
      // the appended unit vectors: W * e_r = W(:, r), and their range sums (bounds 0 / ub_r):
      // xmin2 += sum min(w, 0) * ub_r, xmax1 += sum max(w, 0) * ub_r
      const int mg = n_keep >= 0 ? n + 1 - oh_from : 0;
      if (mg > 0) {
        const int total = ldo * mg;
        for (int e = tid; e < total; e += kChainThreads) {
          const int i = e % ldo, t = e / ldo;
          O[i + (int64_t)(oh_from + t) * ldo] = 0.0 + L.W[i + (int64_t)s_cross[t] * ldw];
        }
        const int q = tid & 15;
        for (int r0 = 0; r0 < ldo; r0 += kChainThreads / 16) {
          const int i = r0 + (tid >> 4);
          double sp = 0.0, sn = 0.0;
          if (i < ldo) {
            for (int t0 = q; t0 < mg; t0 += 64) {
              double w[4], u[4];
#pragma unroll
              for (int s = 0; s < 4; ++s) {
                const int t = t0 + 16 * s;
                w[s] = u[s] = 0.0;
                if (t < mg) {
                  const int neuron = s_cross[t];
                  w[s] = L.W[i + (int64_t)neuron * ldw];
                  u[s] = s_ub[neuron];
                }
              }
#pragma unroll
              for (int s = 0; s < 4; ++s) {
                sp = fma(fmax(w[s], 0.0), u[s], sp);
                sn = fma(fmin(w[s], 0.0), u[s], sn);
              }
            }
          }
#pragma unroll
          for (int off = 1; off < 16; off <<= 1) {
            sp += __shfl_xor(sp, off);
            sn += __shfl_xor(sn, off);
          }
          if (q == 0 && i < ldo) {
            sc.fc.gat[0][i] = sp;
            sc.fc.gat[1][i] = sn;
          }
        }
      }
      lds_barrier();
      double* g = A + L.rng_off;
      if (tid < L.M) {  // the column groups in order, then the gathered columns; lb = (c + xmin1) + xmin2
        double x1 = 0.0, x2 = 0.0, y1 = 0.0, y2 = 0.0;
        for (int w2 = 0; w2 < WC; ++w2) {
          if (w2 >= CT) break;
          x1 += sc.fc.part[0][w2 * ldo + tid];
          x2 += sc.fc.part[1][w2 * ldo + tid];
          y1 += sc.fc.part[2][w2 * ldo + tid];
          y2 += sc.fc.part[3][w2 * ldo + tid];
        }
        if (mg > 0) {
          y1 += sc.fc.gat[0][tid];
          x2 += sc.fc.gat[1][tid];
        }
        const double c = sc.fc.cen[tid];
        const double lo = (c + x1) + x2, up = (c + y1) + y2;
        g[tid] = lo;
        g[ldo + tid] = up;
        s_lb[tid] = lo;
        s_ub[tid] = up;
      }
      if (tid == 0) {
        s_counts[2 * l] = 0;
        s_counts[2 * l + 1] = 0;
      }
      // A ReLU layer next reads the ranges from LDS and meets a full barrier before anybody loads the matrix; an FC
      // layer next loads the matrix other waves have just stored, so their stores must have completed.
      if (l + 1 < a.n_layers && a.layers[l + 1].kind == NNVHIP_LAYER_FC)
        __syncthreads();
      else
        lds_barrier();
      V = O;
      Vsrc = O;
      plb_s = plb;
      pub_s = pub;
      ld = ldo;
      N = L.M;
      n_keep = -1;
      oh_from = 0;
      have_rng = true;
    } else {
      if (!have_rng) {
        __syncthreads();  // the matrix may have been written a moment ago (a ReLU layer's output)
        chain_ranges(V, ld, N, n, plb, pub, s_lb, s_ub, A + L.rng_off, tid);
      }
      // ---- classification (N <= 1024: thread r owns neuron r), ascending lists by ballot + prefix sum
      int32_t* cross_g = IA + L.idx_off;
      int32_t* keep_g = cross_g + ld;
      const int r = tid;
      const bool valid = r < N;
      const double lo = valid ? s_lb[r] : 0.0;
      const double up = valid ? s_ub[r] : 1.0;
      const bool inactive = valid && (up <= 0.0);               // map1 = find(ub <= 0)
      const bool crossing = valid && (lo < 0.0) && (up > 0.0);  // map2 = find(lb < 0 & ub > 0)
      const bool kept = valid && !inactive && !crossing;
      const unsigned long long bc = __ballot(crossing);
      const unsigned long long bi = __ballot(inactive);
      const unsigned long long bk = __ballot(kept);
      if (lane == 0) reinterpret_cast<int*>(wcnt)[wave] = __popcll(bc) | (__popcll(bi) << 10) | (__popcll(bk) << 20);
      lds_barrier();
      int before = 0, all = 0;  // the three counts stay packed: none of the sums passes 2^10
#pragma unroll
      for (int w4 = 0; w4 < 4; ++w4) {
        const int4 c4 = wcnt[w4];
        const int cw[4] = {c4.x, c4.y, c4.z, c4.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          before += 4 * w4 + u < wave ? cw[u] : 0;
          all += cw[u];
        }
      }
      const int woff = before & 1023, koff = before >> 20;
      const int m = all & 1023, inact = (all >> 10) & 1023, nk = all >> 20;
      if (r < kChainMaxN) s_cls[r] = crossing ? 0 : inactive ? kZero : kKeep;  // rows past N: untouched (zero anyway)
      const int kpos = koff + __popcll(bk & ((1ull << lane) - 1ull));
      if (kept) s_keep[kpos] = r;
      const bool sorted = a.order != NNVHIP_ORDER_INDEX;
      if (crossing) {
        const int p = woff + __popcll(bc & ((1ull << lane) - 1ull));
        if (sorted) {
          // areas = 0.5*(abs(ub).*abs(lb))  |  ub - lb   (nn/funcs/PosLin.m:1049-1052, 934-936)
          sc.sort.key[p] = a.order == NNVHIP_ORDER_AREA ? 0.5 * (fabs(up) * fabs(lo)) : up - lo;
          sc.sort.idx[p] = r;
          sc.sort.rank[p] = 0;
        } else {
          s_cross[p] = r;
        }
      }
      if (tid == 0) {
        s_counts[2 * l] = m;
        s_counts[2 * l + 1] = inact;
      }
      lds_barrier();
      if (sorted && m > 0) {
        // stable descending key sort by counting: rank(i) = #{j : key_j > key_i, or key_j == key_i and j < i} over the
        // ascending list (j < i there is "smaller neuron index", what MATLAB's stable sort keeps).  The block's
        // threads share the m x m comparisons; the partial counts meet in integer adds, whose order does not matter.
        int mp = 64;
        while (mp < m) mp *= 2;
        const int tpi = kChainThreads / mp;  // threads per entry (m <= 512: at least two)
        const int i = tid % mp, c0 = tid / mp;
        if (i < m) {
          const double ki = sc.sort.key[i];
          int cnt = 0;
          for (int j = c0; j < m; j += tpi) {
            const double kj = sc.sort.key[j];
            cnt += (kj > ki || (kj == ki && j < i)) ? 1 : 0;
          }
          if (cnt) atomicAdd(&sc.sort.rank[i], cnt);
        }
        lds_barrier();
        if (tid < m) s_cross[sc.sort.rank[tid]] = sc.sort.idx[tid];
      }
      // (a full barrier: the layer's input matrix, written by other threads a few phases ago, is read below; every
      // store of this phase to global memory comes after it, so that no barrier has a fresh store to wait for)
      __syncthreads();
      if (kept) keep_g[kpos] = r;
      if (tid < 2 * (int)kLdAlign) {  // the kept-row list ends with -1 up to a whole group of 16 (at least one group)
        const int end = max((nk + (int)kLdAlign - 1) / (int)kLdAlign * (int)kLdAlign, (int)kLdAlign);
        if (nk + tid < end) keep_g[nk + tid] = -1;
      }
      if (tid < m) cross_g[tid] = s_cross[tid];
      if (tid == 0 && a.mailbox != nullptr)
        post_counts(a.mailbox + 2 * ((int64_t)relu_ord * a.n_sets + blockIdx.x), m, inact, a.mailbox_seq);
      // ---- the output set: V' = [V with the inactive and crossing rows reset, unit vectors of the crossing
      // neurons], new_pred_lb = [plb; 0], new_pred_ub = [pub; ub(index)]  (nn/funcs/PosLin.m:700-738).  Nothing
      // in this launch waits for these stores: the next FC layer reads the kept rows from V itself.
      double* O = A + L.v_off;
      const int ncols_in = n + 1;
      const int total = ld * (ncols_in + m);
      for (int e0 = tid; e0 < total; e0 += 4 * kChainThreads) {
        double val[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {  // the loads of four steps go out together
          const int e = e0 + u * kChainThreads;
          val[u] = 0.0;
          if (e < total) {
            const int i = e % ld, j = e / ld;
            if (j < ncols_in) val[u] = (i >= N || s_cls[i] == kKeep) ? V[e] : 0.0;
            else val[u] = i == s_cross[j - ncols_in] ? 1.0 : 0.0;
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int e = e0 + u * kChainThreads;
          if (e < total) O[e] = val[u];
        }
      }
      double* P = A + L.pred_off;
      double* LU = A + L.lbub_off;
      for (int j = tid; j < n + m; j += kChainThreads) {
        if (j < n) {
          P[j] = plb[j];
          P[L.npad + j] = pub[j];
        } else {
          const int neuron = s_cross[j - n];
          const double ubn = s_ub[neuron];
          P[j] = 0.0;
          P[L.npad + j] = ubn;
          LU[j - n] = s_lb[neuron];
          LU[ld + (j - n)] = ubn;
        }
      }
      if (n_keep >= 0) {  // ReLU after ReLU: its input has appended columns of its own
        __syncthreads();
        Vsrc = O;
        plb_s = P;
        pub_s = P + L.npad;
      } else {
        Vsrc = V;
        plb_s = plb;
        pub_s = pub;
      }
      V = O;
      oh_from = n + 1;
      n += m;
      n_keep = nk;
      plb = P;
      pub = P + L.npad;
      have_rng = false;
      ++relu_ord;
    }
  }
  lds_barrier();
  if (tid < 2 * a.n_layers) counts[tid] = s_counts[tid];
}

// The same launch for networks no layer of which is wider than 64 neurons, every ReLU layer behind an FC layer: the set stays on the
// compute unit.  What the kernel above spends its time on are trips to the cache: a layer's matrix goes out, is read back for
// the row reset, and its kept rows, the weights and the bounds are read again by the next layer.  Here
//  - eight waves: what every wave does for itself (the classification, addresses) costs the block half of what sixteen make of it;
//  - the next FC layer's weights are on their way (in registers) while this one is multiplied;
//  - the columns of a layer stay in the accumulators until its neurons are classified, and then leave for the output
//    matrices and, only the kept rows and without gaps, for the LDS the next layer multiplies from; nothing that went out is
//    read back, so no barrier waits for a store;
//  - a neuron is a lane: every wave classifies all of them by itself, and they meet for the ranking only.
// One box through 5 - 50 x 6 - 5: 48 us there, 38 here (43 with sixteen waves, 60 with four); 128 boxes 70 -> 51.  A set takes up to
// 160 KB of LDS, so a CU has one block where the kernel above has two, and this one is the quicker all the same, however many sets
// there are (us, by events): 256 boxes 88 -> 58, 512 173 -> 111, 1024 331 -> 210, 2048 640 -> 401; 256, 1024 and 4096 through
// 5 - 20 x 3 - 5 (several blocks to a CU either way) 28 -> 23, 102 -> 84, 383 -> 314.
constexpr int kLdsChainN = 64;     // widest layer
constexpr int kLdsChainThreads = 512;
constexpr int kLdsChainTiles = 8;  // column tiles of a wave
// x summed over the four rows of 16 lanes, in every one of them
__device__ __forceinline__ double sum_of_rows(double x) {
  union {
    double d;
    unsigned w[2];
  } a, b;
  a.d = x;
  {
    const auto lo = __builtin_amdgcn_permlane32_swap(a.w[0], a.w[0], false, false), hi = __builtin_amdgcn_permlane32_swap(a.w[1], a.w[1], false, false);
    a.w[0] = lo[0], b.w[0] = lo[1], a.w[1] = hi[0], b.w[1] = hi[1];
    a.d = a.d + b.d;
  }
  const auto lo = __builtin_amdgcn_permlane16_swap(a.w[0], a.w[0], false, false), hi = __builtin_amdgcn_permlane16_swap(a.w[1], a.w[1], false, false);
  a.w[0] = lo[0], b.w[0] = lo[1], a.w[1] = hi[0], b.w[1] = hi[1];
  return a.d + b.d;
}
constexpr int kLdsChainStatic = 16 * 1024;  // bytes of LDS beside the dynamic part, at most
struct ChainLds {
  int32_t pred;    // doubles: where the predicate bounds lie in the dynamic LDS (the kept rows first), lower, then upper ones ...
  int32_t ncap;    // ... room for so many of either
  int32_t weights; // where the weights lie
};

__global__ __launch_bounds__(kLdsChainThreads) void reach_chain_lds_kernel(const ChainSet* __restrict__ sets, ChainSet one, ChainArgs a, ChainLds p) {
  constexpr int NT = kLdsChainThreads, NW = NT / 64, kParts = NW * 16;
  constexpr int kUnits = kLdsChainN / NW;  // columns of the appended unit vectors, to a wave
  extern __shared__ __attribute__((aligned(16))) double lds[];
  double* const sV = lds;             // kept row k of column j at j * ldv + k
  double* const s_pl = lds + p.pred;
  double* const s_pu = s_pl + p.ncap;
  double* const sW = lds + p.weights;
  __shared__ double part[4][kParts];  // [sum][column group * ld + row]: range sums of the contracted columns
  __shared__ double gat[NW][2][kLdsChainN];  // ... of the columns that are columns of the weights, S+ / S-, by wave
  __shared__ double cen[kLdsChainN], s_lb[kLdsChainN], s_ub[kLdsChainN];
  __shared__ int s_keep[kLdsChainN], s_cross[kLdsChainN], s_rank[kLdsChainN];
  __shared__ int s_counts[2 * kChainMaxLayers];
  const ChainSet S = sets ? sets[blockIdx.x] : one;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kq = lane >> 4;
  double* const A = a.arena + (int64_t)blockIdx.x * a.set_stride;
  int32_t* const IA = a.iarena + (int64_t)blockIdx.x * a.iset_stride;

  // weights of a layer: pieces of 16 bytes (64 x 64 at most)
  constexpr int kPieces = kLdsChainN * kLdsChainN / 2 / NT;
  double2 wreg[kPieces];
  auto load_weights = [&](const ChainLayer& L) {
#pragma unroll
    for (int u = 0; u < kPieces; ++u) {
      const int e = 2 * (tid + u * NT);
      wreg[u] = e < L.ldw * L.K ? *reinterpret_cast<const double2*>(L.W + e) : make_double2(0.0, 0.0);
    }
  };
  auto store_weights = [&]() {  // (the LDS has room for 64 x 64, or for what the layers need)
#pragma unroll
    for (int u = 0; u < kPieces; ++u) {
      const int e = 2 * (tid + u * NT);
      if (e < p.pred - p.weights) *reinterpret_cast<double2*>(sW + e) = wreg[u];
    }
  };
  load_weights(a.layers[0]);
  // the input set: everything of it is asked for at once
  const int N = S.N;
  int n = S.n;                   // predicates of the current set
  int nk = N, ldv = N | 1;       // its rows in the LDS (an odd stride: 16 columns meet 16 bank pairs)
  int nd = n + 1, mg = 0;        // columns there; unit vectors of s_cross behind them
  const int order = a.order, n_layers = a.n_layers;
  const bool box = S.idx != nullptr;  // column 1 + t is scale[idx[t]] at row idx[t], the centre is in memory
  double in[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int j = wave + NW * u;
    in[u] = lane < N && j <= (box ? 0 : n) ? S.V[lane + (int64_t)j * S.ld] : 0.0;
  }
  const double scale = box && tid < N ? S.scale[tid] : 0.0;
  const int hot = box && tid < n ? S.idx[tid] : 0;  // (a box has no more columns than rows)
  const double pl0 = tid < n ? S.plb[tid] : 0.0, pu0 = tid < n ? S.pub[tid] : 0.0;
  // The layer list is read through the scalar cache, a line or two a layer: all of it is brought in now, and so is a line of the
  // later layers' weights per thread and step.
  {
    int touched = 0;
#pragma unroll
    for (int l = 0; l < kChainMaxLayers; ++l) touched ^= a.layers[l].kind ^ (int)a.layers[l].idx_off;
    asm volatile("" ::"s"(touched));
  }
  int first = 0;  // lines in front of a layer's
  for (int l = 1; l < n_layers; ++l) {
    const ChainLayer& L = a.layers[l];
    if (L.kind != NNVHIP_LAYER_FC) continue;
    const int lines = L.ldw * L.K / 16, e = (tid - first) & (NT - 1);  // (at most 256)
    if (e < lines) lds_dma16_at(L.W + (int64_t)e * 16, lds_addr_of(&gat[wave][0][0]));  // (nobody reads it there)
    first += lines;
  }
  if (tid < n) {
    s_pl[tid] = pl0;
    s_pu[tid] = pu0;
  }
  for (int j = tid + NT; j < n; j += NT) {
    s_pl[j] = S.plb[j];
    s_pu[j] = S.pub[j];
  }
  if (tid < kLdsChainN) {
    s_keep[tid] = tid;
    cen[tid] = scale;
  }
  if (tid < 2 * n_layers) s_counts[tid] = 0;
  if (box) {
    for (int j = wave; j <= n; j += NW)
      if (lane < N) sV[j * ldv + lane] = j == 0 ? in[0] : 0.0;
    lds_barrier();
    if (tid < n) sV[(1 + tid) * ldv + hot] = cen[hot];
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (wave + NW * u <= n && lane < N) sV[(wave + NW * u) * ldv + lane] = in[u];
    for (int j = wave + 4 * NW; j <= n; j += NW)
      if (lane < N) sV[j * ldv + lane] = S.V[lane + (int64_t)j * S.ld];
  }
  store_weights();
  wait_vm_lds<0>();  // (the touched weights have landed: their place is about to be used)
  lds_barrier();

  int relu_ord = 0;
  for (int l = 0; l < n_layers;) {
    const ChainLayer& L = a.layers[l];
    const bool relu = l + 1 < n_layers && a.layers[l + 1].kind == NNVHIP_LAYER_RELU;
    const int next = l + (relu ? 2 : 1);
    const int M = L.M, ldo = L.ld, ldw = L.ldw, R = ldo / 16;
    const int RW = R > 2 ? 4 : R, WC = NW / RW;
    const int wr = wave % RW, wc = wave / RW;
    const int row = wr * 16 + l16;  // of the tiles this lane has columns of
    const bool tiles = wr < R;
    const int CT = (nd + 15) / 16;
    if (next < n_layers) load_weights(a.layers[next]);
    const double bias = tiles && wc == 0 && kq == 0 && L.bias != nullptr ? L.bias[row] : 0.0;
    if (tid < kLdsChainN) s_rank[tid] = 0;

    // ---- Star.affineMap of the columns in the LDS (operand layout as above)
    double4_t acc[kLdsChainTiles];
#pragma unroll
    for (int t = 0; t < kLdsChainTiles; ++t) acc[t] = double4_t{0.0, 0.0, 0.0, 0.0};
    if (tiles) {
      for (int k0 = 0; k0 < nk; k0 += 32) {  // eight products a round, their operands asked for together
        int kk[8];
        double bv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) kk[u] = s_keep[min(k0 + 4 * u + kq, kLdsChainN - 1)];  // (past the list: some row's number)
#pragma unroll
        for (int u = 0; u < 8; ++u) bv[u] = sW[(kk[u] & (kLdsChainN - 1)) * ldw + row];
#pragma unroll
        for (int u = 0; u < 8; ++u) bv[u] = k0 + 4 * u + kq < nk ? bv[u] : 0.0;
#pragma unroll
        for (int t = 0; t < kLdsChainTiles; ++t) {
          const int tc = wc + t * WC;
          if (tc >= CT) break;
          const double* col = sV + min(tc * 16 + l16, nd - 1) * ldv;  // (columns past the last one: computed and dropped)
#pragma unroll
          for (int u0 = 0; u0 < 8; u0 += 4) {
            if (k0 + 4 * u0 >= nk) break;
            double av[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) av[u] = col[min(k0 + 4 * (u0 + u) + kq, nk - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u) av[u] = k0 + 4 * (u0 + u) + kq < nk ? av[u] : 0.0;
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bv[u0 + u], acc[t], 0, 0, 0);
          }
        }
      }
      if (wc == 0 && kq == 0) {
        acc[0][0] = acc[0][0] + bias;  // newV(:,1) = newV(:,1) + b
        cen[row] = acc[0][0];
      }
      double x[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int t = 0; t < kLdsChainTiles; ++t) {
        const int tc = wc + t * WC;
        if (tc >= CT) break;
        double pl[4], pu[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {  // (the centre and columns past the last one take no part)
          const int col = tc * 16 + kq + 4 * r, j = min(max(col, 1), max(nd - 1, 1)) - 1;
          pl[r] = s_pl[j];
          pu[r] = s_pu[j];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int col = tc * 16 + kq + 4 * r;
          const bool in = col >= 1 && col < nd;
          const double vp = in ? fmax(acc[t][r], 0.0) : 0.0, vn = in ? fmin(acc[t][r], 0.0) : 0.0;
          const double l0 = in ? pl[r] : 0.0, u0 = in ? pu[r] : 0.0;
          x[0] = fma(vp, l0, x[0]);  // xmin1
          x[1] = fma(vn, u0, x[1]);  // xmin2
          x[2] = fma(vp, u0, x[2]);  // xmax1
          x[3] = fma(vn, l0, x[3]);  // xmax2
        }
      }
      // the four lane groups hold different columns of the same rows
#pragma unroll
      for (int q = 0; q < 4; ++q) x[q] = sum_of_rows(x[q]);
      if (kq == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) part[q][wc * ldo + row] = x[q];
      }
    }
    // the appended unit vectors: W * e_r = W(:, r), and their range sums (bounds 0 / ub_r); a column to a wave, a row to a lane
    double unit[kUnits];
#pragma unroll
    for (int s = 0; s < kUnits; ++s) unit[s] = 0.0;
    if (mg > 0) {
      double sp = 0.0, sn = 0.0;
      int at[kUnits];
      double u[kUnits];
#pragma unroll
      for (int s = 0; s < kUnits; ++s) {
        const int t = min(wave + NW * s, mg - 1);
        at[s] = s_cross[t];
        u[s] = s_pu[nd - 1 + t];
      }
#pragma unroll
      for (int s = 0; s < kUnits; ++s) {
        if (wave + NW * s >= mg) break;
        unit[s] = 0.0 + sW[at[s] * ldw + min(lane, ldo - 1)];
      }
#pragma unroll
      for (int s = 0; s < kUnits; ++s) {
        if (wave + NW * s >= mg) break;
        sp = fma(fmax(unit[s], 0.0), u[s], sp);
        sn = fma(fmin(unit[s], 0.0), u[s], sn);
      }
      gat[wave][0][lane] = sp;
      gat[wave][1][lane] = sn;
    }
    lds_barrier();  // the sums are there; nobody reads this layer's weights, rows or lists any more
    if (tid < 256) {  // the column groups in order, then the gathered columns; lb = (c + xmin1) + xmin2
      const int i = wave * 16 + l16;  // kq: which sum
      const int np = min(WC, CT), ng = kq == 1 || kq == 2 ? min(NW, mg) : 0;
      const double c = cen[i];
      double s = 0.0, t = 0.0;
#pragma unroll
      for (int w0 = 0; w0 < NW; w0 += 4) {  // four reads at a time
        if (w0 >= np) break;
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = part[kq][min(min(w0 + u, np - 1) * ldo + i, kParts - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u) s += w0 + u < np ? v[u] : 0.0;
      }
      if (mg > 0) {
        double g[NW];
#pragma unroll
        for (int u = 0; u < NW; ++u) g[u] = gat[min(u, min(NW, mg) - 1)][kq == 1][i];
#pragma unroll
        for (int u = 0; u < NW; ++u) t += u < ng ? g[u] : 0.0;
      }
      if (ng > 0) s += t;
      const double s1 = __shfl(s, (lane + 16) & 63);
      if (i < M && kq == 0) s_lb[i] = (c + s) + s1;
      if (i < M && kq == 2) s_ub[i] = (c + s) + s1;
    }
    lds_barrier();
    // ---- the ReLU layer: classification, a neuron to a lane, by every wave; the waves share the comparisons of the ranking
    const double lo = lane < M ? s_lb[lane] : 0.0, up = lane < M ? s_ub[lane] : 1.0;
    bool crossing = false, kept = lane < M;
    int m = 0, inact = 0, nk_out = M, kpos = lane, rank = 0;
    if (relu) {
      const bool inactive = lane < M && (up <= 0.0);      // map1 = find(ub <= 0)
      crossing = lane < M && (lo < 0.0) && (up > 0.0);    // map2 = find(lb < 0 & ub > 0)
      kept = lane < M && !inactive && !crossing;
      const unsigned long long bc = __ballot(crossing), bk = __ballot(kept), below = (1ull << lane) - 1ull;
      m = __popcll(bc);
      inact = __popcll(__ballot(inactive));
      nk_out = __popcll(bk);
      kpos = __popcll(bk & below);
      rank = __popcll(bc & below);
      if (order != NNVHIP_ORDER_INDEX && m > 1) {
        // stable descending key sort by counting: areas = 0.5*(abs(ub).*abs(lb))  |  ub - lb  (nn/funcs/PosLin.m:1049-1052, 934-936)
        const double key = order == NNVHIP_ORDER_AREA ? 0.5 * (fabs(up) * fabs(lo)) : up - lo;
        const long long bits = __double_as_longlong(key);
        int cnt = 0;
        for (unsigned mine = (unsigned)(bc >> (kLdsChainN / NW * wave)) & ((1u << (kLdsChainN / NW)) - 1u); mine != 0; mine &= mine - 1) {
          const int j = kLdsChainN / NW * wave + __builtin_ctz(mine);
          const int jl = __builtin_amdgcn_readlane((int)(unsigned)(bits & 0xffffffffll), j), jh = __builtin_amdgcn_readlane((int)(bits >> 32), j);
          const double kj = __longlong_as_double(((long long)jh << 32) | (unsigned)jl);
          cnt += (kj > key || (kj == key && j < lane)) ? 1 : 0;
        }
        if (crossing && cnt) atomicAdd(&s_rank[lane], cnt);
        lds_barrier();
        rank = s_rank[lane];
      }
    }
    // ---- what the next layer reads (everybody is past the last reader of what is overwritten)
    const int ldv_out = nk_out | 1;
    const bool more = next < n_layers;
    if (more) store_weights();
    const int kp = __shfl(kept ? kpos : -1, row & 63);  // place of this lane's tile row among the kept ones
    if (tiles && more && kp >= 0) {
#pragma unroll
      for (int t = 0; t < kLdsChainTiles; ++t) {
        const int tc = wc + t * WC;
        if (tc >= CT) break;
        double* const v = sV + (tc * 16 + kq) * ldv_out + kp;
        const int left = nd - tc * 16 - kq;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * r < left) v[4 * r * ldv_out] = acc[t][r];
      }
    }
    if (more && mg > 0 && kept) {
#pragma unroll
      for (int s = 0; s < kUnits; ++s)
        if (wave + NW * s < mg) sV[(nd + wave + NW * s) * ldv_out + kpos] = unit[s];
    }
    if (wave == 0) {
      if (kept) s_keep[kpos] = lane;
      if (crossing) {
        s_cross[rank] = lane;
        s_pl[n + rank] = 0.0;
        s_pu[n + rank] = up;
      }
    }
    // ---- the output sets, which nothing in this launch reads
    double* const O = A + L.v_off;
    double* const g = A + L.rng_off;
    if (tid < M) {
      g[tid] = lo;
      g[ldo + tid] = up;
    }
    double* const O2 = relu ? A + a.layers[l + 1].v_off : nullptr;  // V' = [V with the inactive and crossing rows reset, unit vectors]
    if (tiles) {
      const bool stays = kp >= 0 || row >= M;  // rows [M, ld): zeros, W's padding rows
#pragma unroll
      for (int t = 0; t < kLdsChainTiles; ++t) {
        const int tc = wc + t * WC;
        if (tc >= CT) break;
        double* const o = O + row + (int64_t)(tc * 16 + kq) * ldo;
        double* const o2 = O2 + row + (int64_t)(tc * 16 + kq) * ldo;
        const int left = nd - tc * 16 - kq;  // columns from this lane's first on
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * r < left) o[4 * r * ldo] = acc[t][r];
        if (relu) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (4 * r < left) o2[4 * r * ldo] = stays ? acc[t][r] : 0.0;
        }
      }
    }
    if (lane < ldo) {
      if (mg > 0) {
#pragma unroll
        for (int s = 0; s < kUnits; ++s) {
          const int t = wave + NW * s;
          if (t >= mg) break;
          O[lane + (int64_t)(nd + t) * ldo] = unit[s];
          if (relu) O2[lane + (int64_t)(nd + t) * ldo] = kept || lane >= M ? unit[s] : 0.0;
        }
      }
      for (int t = wave; t < m; t += NW) O2[lane + (int64_t)(n + 1 + t) * ldo] = crossing && rank == t ? 1.0 : 0.0;
    }
    if (relu) {
      const ChainLayer& Q = a.layers[l + 1];
      double* const P = A + Q.pred_off;    // new_pred_lb = [plb; 0], new_pred_ub = [pub; ub(index)]  (nn/funcs/PosLin.m:737-738)
      double* const LU = A + Q.lbub_off;
      int32_t* const cross_g = IA + Q.idx_off;
      int32_t* const keep_g = cross_g + ldo;
      for (int j = tid; j < n; j += NT) {
        P[j] = s_pl[j];
        P[Q.npad + j] = s_pu[j];
      }
      if (wave == 0) {
        if (crossing) {
          P[n + rank] = 0.0;
          P[Q.npad + n + rank] = up;
          LU[rank] = lo;
          LU[ldo + rank] = up;
          cross_g[rank] = lane;
        }
        if (kept) keep_g[kpos] = lane;
      }
      if (tid < 2 * (int)kLdAlign) {  // the kept-row list ends with -1 up to a whole group of 16 (at least one group)
        const int end = max((nk_out + (int)kLdAlign - 1) / (int)kLdAlign * (int)kLdAlign, (int)kLdAlign);
        if (nk_out + tid < end) keep_g[nk_out + tid] = -1;
      }
      if (tid == 0) {
        s_counts[2 * (l + 1)] = m;
        s_counts[2 * (l + 1) + 1] = inact;
        if (a.mailbox != nullptr)
          post_counts(a.mailbox + 2 * ((int64_t)relu_ord * a.n_sets + blockIdx.x), m, inact, a.mailbox_seq);
      }
      ++relu_ord;
    }
    nd = n + 1;
    n += m;
    mg = m;
    nk = nk_out;
    ldv = ldv_out;
    l = next;
    lds_barrier();
  }
  if (tid < 2 * a.n_layers) a.counts[(int64_t)blockIdx.x * a.n_layers * 2 + tid] = s_counts[tid];
}

// Worst-case layout of one set's slice of the arenas for the given layer list.
struct ChainPlan {
  ChainArgs args{};
  std::vector<int64_t> ncap;  // worst-case predicate count of every layer's output
  int64_t doubles = 0, ints = 0;
  int n_relu = 0;
  bool in_lds = false;  // reach_chain_lds_kernel takes it
  ChainLds lds{};
  int64_t lds_doubles = 0;
};

// Whether a set of at most n0_max predicates stays in the LDS through the planned layers, whatever crosses.  (How many sets there are
// does not matter: see the kernel.)
static void plan_chain_lds(int64_t N0, int64_t n0_max, ChainPlan* plan) {
  const ChainArgs& a = plan->args;
  int64_t rows = 0, weights = 0, before = n0_max, dense = n0_max;  // predicates in front of the layer, and those that are not its ReLU layer's
  if (N0 > kLdsChainN || a.layers[0].kind != NNVHIP_LAYER_FC) return;
  rows = (n0_max + 1) * (N0 | 1);
  for (int l = 0; l < a.n_layers; ++l) {
    const ChainLayer& L = a.layers[l];
    if (L.ld > kLdsChainN) return;
    if (L.kind == NNVHIP_LAYER_FC) {
      const int64_t groups = kLdsChainThreads / 64 / (L.ld > 32 ? 4 : L.ld / 16);  // of waves along the columns
      if (ceil_div(dense + 1, 16) > groups * kLdsChainTiles) return;  // (the columns a ReLU layer appends are columns of the weights)
      weights = std::max(weights, (int64_t)L.ldw * L.K);
    } else if (a.layers[l - 1].kind != NNVHIP_LAYER_FC) {
      return;
    }
    // (the columns a ReLU layer appends do not lie there; the last layer leaves nothing)
    if (l + 1 < a.n_layers) rows = std::max(rows, (before + 1) * (L.M | 1));
    dense = before;
    before = plan->ncap[(size_t)l];
  }
  rows = round_up(rows, 2);
  plan->lds = ChainLds{(int32_t)(rows + weights), (int32_t)std::max<int64_t>(before, 1), (int32_t)rows};
  plan->lds_doubles = rows + weights + 2 * std::max<int64_t>(before, 1);
  plan->in_lds = 8 * plan->lds_doubles + kLdsChainStatic <= 160 * 1024;
}

static bool plan_chain(nnvhip_ctx* c, int64_t n_layers, const int32_t* kind, const void* const* layer, int64_t N0, int64_t n0_max,
                       ChainPlan* plan) {
  if (n_layers < 1 || n_layers > kChainMaxLayers) return false;
  int64_t N = N0, ncap = n0_max;
  int64_t off = 0, ioff = 0;
  double work = 0.0;
  plan->ncap.resize((size_t)n_layers);
  for (int64_t l = 0; l < n_layers; ++l) {
    ChainLayer& L = plan->args.layers[l];
    L = ChainLayer{};
    L.kind = kind[l];
    if (kind[l] == NNVHIP_LAYER_FC) {
      const nnvhip_fc* fc = static_cast<const nnvhip_fc*>(layer[l]);
      if (!fc || fc->ctx != c || fc->K != N || fc->M > kChainMaxN) return false;
      L.W = fc->W->as<double>();
      L.bias = fc->bias ? fc->bias->as<double>() : nullptr;
      L.M = (int32_t)fc->M;
      L.K = (int32_t)fc->K;
      L.ldw = (int32_t)fc->Mp;
      N = fc->M;
      L.ld = (int32_t)round_up(N, kLdAlign);
      work += (double)L.ld * (double)fc->K * (double)(ncap + 1);
    } else if (kind[l] == NNVHIP_LAYER_RELU) {
      if (N > kChainMaxN) return false;
      L.M = (int32_t)N;
      L.ld = (int32_t)round_up(N, kLdAlign);
      ncap += N;
      L.npad = (int32_t)round_up(std::max<int64_t>(ncap, 1), kLdAlign);
      ++plan->n_relu;
    } else {
      return false;
    }
    plan->ncap[l] = ncap;
    L.v_off = off;
    off += (int64_t)L.ld * (ncap + 1);
    L.rng_off = off;
    off += 2 * (int64_t)L.ld;
    if (kind[l] == NNVHIP_LAYER_RELU) {
      L.pred_off = off;
      off += 2 * (int64_t)L.npad;
      L.lbub_off = off;
      off += 2 * (int64_t)L.ld;
      L.idx_off = ioff;
      ioff += 2 * (int64_t)L.ld + kLdAlign;
    }
  }
  // one block does all of it: only networks whose worst case is a few hundred thousand matrix entries
  if (off > (int64_t(1) << 18) || work > 6.4e7) return false;
  plan->doubles = off;
  plan->ints = std::max<int64_t>(ioff, kLdAlign);
  plan->args.n_layers = (int32_t)n_layers;
  plan_chain_lds(N0, n0_max, plan);
  return true;
}

// Whether the layer list runs as one launch for these sets, and the layout of its arenas if so.
static bool chain_takes(nnvhip_ctx* c, int64_t n_layers, const int32_t* kind, const void* const* layer, int order, int64_t count,
                        nnvhip_star* const* in, ChainPlan* plan) {
  if (!c->small_chain || c->dense_affine || count < 1 || count > 65535) return false;
  if (order != NNVHIP_ORDER_INDEX && order != NNVHIP_ORDER_AREA && order != NNVHIP_ORDER_RANGE) return false;
  int64_t n0_max = 0;
  for (int64_t i = 0; i < count; ++i) {
    if (!in[i] || in[i]->ctx != c || in[i]->N != in[0]->N) return false;  // the layer loop reports it
    n0_max = std::max(n0_max, in[i]->n);
  }
  if (!plan_chain(c, n_layers, kind, layer, in[0]->N, n0_max, plan)) return false;
  return (double)plan->doubles * (double)count <= 5.0e8;  // 4 GB of worst-case buffers
}

bool small_chain_takes(nnvhip_ctx* c, int64_t n_layers, const int32_t* kind, const void* const* layer, int order, int64_t count,
                       nnvhip_star* const* in) {
  ChainPlan plan;
  return chain_takes(c, n_layers, kind, layer, order, count, in, &plan);
}

int reach_small_chain(nnvhip_ctx* c, int64_t n_layers, const int32_t* kind, const void* const* layer, int order, int64_t count,
                      nnvhip_star* const* in, nnvhip_star** out, bool* taken) {
  *taken = false;
  ChainPlan plan;
  if (!chain_takes(c, n_layers, kind, layer, order, count, in, &plan)) return NNVHIP_OK;
  *taken = true;

  // boxes go in as they are where the first layer is an FC layer
  auto as_box = [&](const nnvhip_star* s) {
    return kind[0] == NNVHIP_LAYER_FC && is_unwritten_box(s);
  };
  {
    std::vector<nnvhip_star*> full;
    for (int64_t i = 0; i < count; ++i)
      if (!as_box(in[i])) full.push_back(in[i]);
    if (!full.empty()) NNV_TRY(ensure_dense_batch(c, (int64_t)full.size(), full.data(), true, true));
  }
  BufRef arena, iarena, cnt;
  NNV_TRY(c->alloc(sizeof(double) * plan.doubles * count, &arena));
  NNV_TRY(c->alloc(sizeof(int32_t) * plan.ints * count, &iarena));
  NNV_TRY(c->alloc(sizeof(int32_t) * 2 * n_layers * count, &cnt));
  ChainArgs& a = plan.args;
  a.order = order;
  a.arena = arena->as<double>();
  a.set_stride = plan.doubles;
  a.iarena = iarena->as<int32_t>();
  a.iset_stride = plan.ints;
  a.counts = cnt->as<int32_t>();
  a.n_sets = (int32_t)count;
  const int64_t words = (int64_t)plan.n_relu * count;
  const bool use_mailbox = words > 0 && words <= nnvhip_ctx::kMailboxSets && c->mailbox != nullptr;
  if (use_mailbox) {
    ++c->mailbox_seq;
    volatile unsigned long long* box = reinterpret_cast<volatile unsigned long long*>(c->mailbox);
    for (int64_t i = 0; i < words; ++i) box[i] = kMailboxEmpty;
    std::atomic_thread_fence(std::memory_order_seq_cst);
    a.mailbox = const_cast<int32_t*>(c->mailbox);
    a.mailbox_seq = (int32_t)(c->mailbox_seq & 0xffffu);
  }
  std::vector<ChainSet> sets((size_t)count);
  for (int64_t i = 0; i < count; ++i) {
    const bool box = as_box(in[i]);
    sets[i] = ChainSet{in[i]->V, in[i]->plb, in[i]->pub, box ? in[i]->oh_idx : nullptr, box ? in[i]->oh_scale : nullptr, in[i]->ld,
                       (int32_t)in[i]->N, (int32_t)in[i]->n};
  }
  const ChainSet* table = nullptr;
  BufRef tab;
  if (count > 1) {
    NNV_TRY(c->upload(sets.data(), sizeof(ChainSet) * count, &tab));
    table = tab->as<ChainSet>();
  }
  if (plan.in_lds)
    NNV_LAUNCH(c, c->kernel_timing, reach_chain_lds_kernel, dim3((unsigned)count), dim3(kLdsChainThreads), (unsigned)(8 * plan.lds_doubles), table,
               sets[0], a, plan.lds);
  else
    NNV_LAUNCH(c, c->kernel_timing, reach_chain_kernel, dim3((unsigned)count), dim3(kChainThreads), 0, table, sets[0], a);
  NNV_HIP_TRY(hipGetLastError());
  c->routes[plan.in_lds ? NNVHIP_ROUTE_CHAIN_LDS : NNVHIP_ROUTE_CHAIN] += count;
  // Handles of earlier arrays that were released but not let go yet go now, all of them, while the kernel runs: their
  // arenas are what the next call of this size takes (a thousand sets come to a gigabyte, and a queue that grows from
  // call to call would have the pool ask the driver for another one each time).
  c->drain_deferred();

  // the crossing counts: all the host needs to know to fill in the handles
  std::vector<int32_t> counts((size_t)(2 * n_layers * count), 0);
  if (use_mailbox) {
    const auto t0 = std::chrono::steady_clock::now();
    long spins = 0;
    const volatile unsigned long long* box = reinterpret_cast<const volatile unsigned long long*>(c->mailbox);
    int ord = 0;
    for (int64_t l = 0; l < n_layers; ++l) {
      if (kind[l] != NNVHIP_LAYER_RELU) continue;
      for (int64_t i = 0; i < count; ++i) {
        const int64_t w_i = (int64_t)ord * count + i;
        unsigned long long w = box[w_i];
        while (w == kMailboxEmpty) {
          if ((++spins & 0xfff) == 0 && std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count() > 10.0) {
            NNV_HIP_TRY(hipStreamSynchronize(c->stream));
            if (box[w_i] == kMailboxEmpty) NNV_FAIL(NNVHIP_ERR_HIP, "the reach kernel did not report its counts");
          }
          w = box[w_i];
        }
        int m_ = 0, inact_ = 0, seq_ = 0;
        mailbox_unpack(w, &m_, &inact_, &seq_);
        if (seq_ != (int)(c->mailbox_seq & 0xffffu)) NNV_FAIL(NNVHIP_ERR_HIP, "internal: mailbox word of another call");
        counts[(size_t)((i * n_layers + l) * 2)] = m_;
        counts[(size_t)((i * n_layers + l) * 2 + 1)] = inact_;
      }
      ++ord;
    }
  } else if (plan.n_relu > 0) {
    void* hc = nullptr;
    NNV_TRY(c->stage(sizeof(int32_t) * counts.size(), &hc));
    NNV_HIP_TRY(hipMemcpyAsync(hc, cnt->ptr, sizeof(int32_t) * counts.size(), hipMemcpyDeviceToHost, c->stream));
    NNV_HIP_TRY(hipStreamSynchronize(c->stream));
    memcpy(counts.data(), hc, sizeof(int32_t) * counts.size());
  }
  if (c->kernel_timing) {
    // algorithmic bytes: the weights read once per set, every layer's output matrix written once
    double bytes = 0.0;
    for (int64_t i = 0; i < count; ++i) {
      int64_t n = in[i]->n;
      for (int64_t l = 0; l < n_layers; ++l) {
        if (kind[l] == NNVHIP_LAYER_FC) bytes += 8.0 * (double)a.layers[l].M * (double)a.layers[l].K;
        n += counts[(size_t)((i * n_layers + l) * 2)];
        bytes += 8.0 * (double)a.layers[l].M * (double)(n + 1);
      }
    }
    NNV_TRY(c->kernel_timer_end(true, 8, bytes));
  }

  // ---- handles: every layer's output set, described exactly as the layer-by-layer path would leave it
  // once every pending piece had been written
  for (int64_t i = 0; i < count; ++i) {
    double* A = arena->as<double>() + i * plan.doubles;
    int32_t* IA = iarena->as<int32_t>() + i * plan.ints;
    const nnvhip_star* prev = in[i];
    const double* prev_ub = nullptr;  // upper bounds of prev's estimated ranges, when the kernel left them
    for (int64_t l = 0; l < n_layers; ++l) {
      const ChainLayer& L = a.layers[l];
      nnvhip_star* o = new_star(c);
      o->N = L.M;
      o->ld = L.ld;
      o->Vbuf = arena;
      o->V = A + L.v_off;
      if (L.kind == NNVHIP_LAYER_FC) {
        o->n = prev->n;
        o->pbuf = prev->pbuf;
        o->plb = prev->plb;
        o->pub = prev->pub;
        o->ptails = prev->ptails;
        o->pslot = prev->pslot;
        o->pcap = prev->pcap;
        o->cons = prev->cons;
        o->has_zono = prev->has_zono;
        o->rbuf = arena;
        o->lb = A + L.rng_off;
        o->ub = o->lb + L.ld;
        prev_ub = o->ub;
      } else {
        const int64_t m = counts[(size_t)((i * n_layers + l) * 2)];
        const int64_t inact = counts[(size_t)((i * n_layers + l) * 2 + 1)];
        o->n = prev->n + m;
        o->pbuf = arena;
        o->plb = A + L.pred_off;
        o->pub = o->plb + L.npad;
        o->n_inactive = inact;
        o->n_crossing = m;
        o->pre_ub_buf = arena;
        o->pre_ub = prev_ub ? prev_ub : A + L.rng_off + L.ld;
        o->pre_lb = o->pre_ub - L.ld;  // (lb in front of ub, ld apart)
        o->n_kept = L.M - m - inact;
        o->kept_buf = iarena;
        o->kept_idx = IA + L.idx_off + L.ld;
        if (m > 0) {
          o->oh_from = prev->n + 1;
          o->oh_plb_zero = true;
          o->oh_idx_buf = iarena;
          o->oh_idx = IA + L.idx_off;
          auto node = make_cons(c);
          node->prev = prev->cons;
          node->n_before = prev->n;
          node->src = prev->Vbuf;  // C2/C3 rows are rows of the pre-ReLU [c V]
          node->src_V = prev->V;
          node->src_ld = prev->ld;
          node->index = iarena;
          node->index_off = (IA + L.idx_off) - iarena->as<int32_t>();
          node->m = m;
          node->p_total = prev->cons->p_total + 3 * m;
          node->n_total = o->n;
          node->lbub = arena;
          node->lbub_off = (A + L.lbub_off) - arena->as<double>();
          node->ld_lbub = L.ld;
          o->cons = std::move(node);
        } else {
          o->cons = prev->cons;
        }
        prev_ub = nullptr;
      }
      out[l * count + i] = o;
      prev = o;
    }
  }
  return NNVHIP_OK;
}

}  // namespace nnvhip
