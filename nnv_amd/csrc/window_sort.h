// Stable counting sort of the columns of a set by where their windows start, by a few blocks of kSortThreads threads.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace nnvhip {

constexpr int kSortThreads = 1024;
constexpr int kSortBuckets = 1024;   // at most (one thread each)
constexpr int kSortColumns = 65535;  // at most
constexpr int kSortRun = 512;        // columns a block puts in place at most, by one wave

// Columns of a block where `sets` sets of n columns are sorted in one launch, and its blocks per set.  A wave takes 0.4 us for 64
// columns, one after the other, and every block counts all columns: short runs as long as the blocks find a place side by side.
// The set-up launches of a 32 x 32 x 3 network (runs of 512 -> 64): 11.3, 13.2 and 13.2 us -> 6.4, 7.4 and 8.2; of a 28 x 28 x 1
// network 8.7 -> 5.2, 25 of them (runs of 128) 10.6 -> 7.0.
inline int sort_window_run(int64_t n, int64_t sets) {
  int run = 64;
  while (run < kSortRun && sets * ((n + run - 1) / run) > 256) run *= 2;
  return run;
}
inline int sort_window_blocks(int64_t n, int run) { return (int)std::max<int64_t>(1, (n + run - 1) / run); }

// order[0 .. n): the columns 1 .. n, by bucket_of(column) in [0, buckets), a bucket's columns ascending; first (or null):
// buckets + 1 entries, where each bucket's columns begin.  Block blk of sort_window_blocks(n, run); all threads of
// a block call it.  Every block counts all columns (integer atomics in LDS, whose order does not matter), once in total and
// once those in front of its own run, and then knows where the run's columns go: no block waits for another.  (One block
// with a table of counts per wave took 13 us for 4300 columns, this takes 5.)
template <class BucketOf>
__device__ __forceinline__ void sort_windows(int n, int buckets, int32_t* __restrict__ order, int32_t* __restrict__ first, int run, int blk,
                                             const BucketOf& bucket_of) {
  __shared__ int s_all[kSortBuckets], s_before[kSortBuckets], s_wave[kSortThreads / 64], s_key[kSortRun];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j0 = min(n, blk * run), j1 = min(n, j0 + run);
  if (blk > 0 && j0 >= j1) return;  // (block 0 writes `first`)
  s_all[tid] = 0;
  s_before[tid] = 0;
  __syncthreads();
  constexpr int kAhead = 4;  // columns whose windows are asked for together
  for (int jj = tid; jj < n; jj += kAhead * kSortThreads) {
    int key[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) key[u] = jj + u * kSortThreads < n ? bucket_of(1 + jj + u * kSortThreads) : 0;
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int j = jj + u * kSortThreads;
      if (j >= n) break;
      atomicAdd(&s_all[key[u]], 1);
      if (j < j0) atomicAdd(&s_before[key[u]], 1);
      else if (j < j1) s_key[j - j0] = key[u];
    }
  }
  __syncthreads();
  const int total = s_all[tid];  // (0 from `buckets` on)
  int scan = total;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(scan, off);
    if (lane >= off) scan += v;
  }
  if (lane == 63) s_wave[wave] = scan;
  __syncthreads();
  int base = scan - total;
  for (int w = 0; w < wave; ++w) base += s_wave[w];
  if (first != nullptr && blk == 0) {
    if (tid < buckets) first[tid] = base;
    if (tid == 0) first[buckets] = n;
  }
  s_before[tid] += base;
  __syncthreads();
  if (wave != 0) return;
  int bits = 0;
  while ((1 << bits) < buckets) ++bits;
  for (int j = j0; j < j1; j += 64) {  // lanes with the same bucket find each other by one ballot per bit
    const bool valid = j + lane < j1;
    const int key = valid ? s_key[j - j0 + lane] : 0;
    unsigned long long m = __ballot(valid);
    for (int b = 0; b < bits; ++b) {
      const unsigned long long v = __ballot((key >> b) & 1);
      m &= ((key >> b) & 1) ? v : ~v;
    }
    const int rank = __popcll(m & ((1ull << lane) - 1ull));
    const int at = valid ? s_before[key] : 0;
    if (valid) order[at + rank] = 1 + j + lane;
    if (valid && rank == 0) s_before[key] = at + __popcll(m);
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace nnvhip
