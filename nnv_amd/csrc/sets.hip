// Set handles: constructors (Star(V, C, d, lb, ub), Star(lb, ub) for arrays of boxes, the reduceMem box), reference
// counting, property reads and the estimateRanges entry points.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <map>

#include "internal.h"

using namespace nnvhip;

namespace {

// Read-back of lb / ub: the kernel stores them straight into pinned host memory in the caller's layout (lb of all
// sets, then ub of all sets, N entries each) and the host watches one flag per block.  What bounds it is latency, not
// bytes: a device-to-host copy into pageable memory costs the host some 20 us each (two per call: 36-40 us for a
// ten-row set), the kernel plus the host's last look at the flag about 10 us.  A block ends with a system-scope fence
// behind its stores and then its flag, so whoever sees the flag sees the block's values.
struct PostSet {
  const double* lb;
  const double* ub;
};
// A thread looks a set up, loads and stores two values only, both asked for before the first is stored, and places are
// 32-bit numbers (total <= kPostMax).  Blocks of 4096 values had sixteen such look-ups one behind the other in each thread, a
// 64-bit division in each: 2 x 10 values of 100 sets 11.6 us, 6.2 now; 1400 values of one set 5.4 -> 3.8; the bounds of images
// of 6272 and 12 544 neurons, together 23 -> 15.6 us (the larger one's 200 KB then go over at 22 GB/s); ten rows 2.6 as before.
constexpr int kPostEach = 2;
constexpr int kPostBlock = 256 * kPostEach;
__global__ __launch_bounds__(256) void post_ranges_kernel(const PostSet* __restrict__ table, PostSet one, uint32_t N, uint32_t total,
                                                           double* __restrict__ dst, uint32_t* __restrict__ flags) {
  const uint32_t half = total / 2;
  const uint32_t e0 = blockIdx.x * (uint32_t)kPostBlock + threadIdx.x;
  double v[kPostEach];
#pragma unroll
  for (int u = 0; u < kPostEach; ++u) {
    const uint32_t e = e0 + 256 * u;
    v[u] = 0.0;
    if (e < total) {
      const uint32_t q = e < half ? e : e - half;
      const uint32_t i = table ? q / N : 0;
      const PostSet s = table ? table[i] : one;
      v[u] = (e < half ? s.lb : s.ub)[q - i * N];
    }
  }
#pragma unroll
  for (int u = 0; u < kPostEach; ++u)
    if (e0 + 256 * u < total) dst[e0 + 256 * u] = v[u];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(flags + blockIdx.x, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// lb / ub of all sets (known on the device) to the host; either pointer may be null.
int post_ranges(nnvhip_ctx* c, int64_t count, nnvhip_star* const* s, double* lb, double* ub) {
  const int64_t N = s[0]->N, total = 2 * N * count, blocks = ceil_div(total, kPostBlock);
  const PostSet* table = nullptr;
  BufRef tab;
  if (count > 1) {
    std::vector<PostSet> ps((size_t)count);
    for (int64_t i = 0; i < count; ++i) ps[(size_t)i] = PostSet{s[i]->lb, s[i]->ub};
    NNV_TRY(c->upload_table(ps.data(), sizeof(PostSet) * count, &tab));
    table = tab->as<PostSet>();
  }
  void* slot = nullptr;
  const size_t flag_bytes = ((size_t)blocks * sizeof(uint32_t) + 255) & ~size_t(255);
  NNV_TRY(c->stage(flag_bytes + sizeof(double) * (size_t)total, &slot));
  uint32_t* flags = static_cast<uint32_t*>(slot);
  double* vals = reinterpret_cast<double*>(static_cast<char*>(slot) + flag_bytes);
  for (int64_t b = 0; b < blocks; ++b) reinterpret_cast<volatile uint32_t*>(flags)[b] = 0;
  std::atomic_thread_fence(std::memory_order_seq_cst);
  hipLaunchKernelGGL(post_ranges_kernel, dim3((unsigned)blocks), dim3(256), 0, c->stream, table, PostSet{s[0]->lb, s[0]->ub}, (uint32_t)N,
                     (uint32_t)total, vals, flags);
  NNV_HIP_TRY(hipGetLastError());
  const auto t0 = std::chrono::steady_clock::now();
  long spins = 0;
  for (int64_t b = 0; b < blocks; ++b)
    while (__atomic_load_n(flags + b, __ATOMIC_ACQUIRE) == 0) {
      if (!c->deferred.empty()) c->drain_deferred(16);  // something useful to do while the device works
      if ((++spins & 0xfff) == 0 && std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count() > 10.0) {
        NNV_HIP_TRY(hipStreamSynchronize(c->stream));  // surfaces a launch failure, if any
        if (__atomic_load_n(flags + b, __ATOMIC_ACQUIRE) == 0) NNV_FAIL(NNVHIP_ERR_HIP, "the ranges did not arrive");
      }
    }
  if (lb) memcpy(lb, vals, sizeof(double) * (size_t)(total / 2));
  if (ub) memcpy(ub, vals + total / 2, sizeof(double) * (size_t)(total / 2));
  return NNVHIP_OK;
}

// Above this many values the copy engine is the better way: the blocks' stores reach some 20 GB/s, and a call that
// large no longer notices 20 us.
constexpr int64_t kPostMax = int64_t(1) << 17;

}  // namespace

extern "C" {

/* ------------------------------------------------------------------------------------------ */
/* sets                                                                                        */
/* ------------------------------------------------------------------------------------------ */

// Uploads a host column-major rows x cols matrix into a zero-padded device matrix with leading
// dimension ld.
static int upload_matrix(nnvhip_ctx* c, const double* host, int64_t rows, int64_t cols, int64_t ld,
                         double* dev) {
  if (rows == 0 || cols == 0) return NNVHIP_OK;
  if (ld != rows) NNV_HIP_TRY(hipMemsetAsync(dev, 0, sizeof(double) * ld * cols, c->stream));
  NNV_HIP_TRY(hipMemcpy2DAsync(dev, sizeof(double) * ld, host, sizeof(double) * rows, sizeof(double) * rows,
                               cols, hipMemcpyHostToDevice, c->stream));
  c->h2d_bytes += (int64_t)sizeof(double) * rows * cols;
  // the source is pageable caller memory: finish before returning
  NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  return NNVHIP_OK;
}

int nnvhip_star_create(nnvhip_ctx* c, int64_t N, int64_t n, const double* V, const double* pred_lb,
                       const double* pred_ub, const double* C, const double* d, int64_t p,
                       nnvhip_star** out) {
  CHECK_CTX(c);
  if (!out || !V) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  if (N <= 0 || n < 0 || p < 0) NNV_FAIL(NNVHIP_ERR_SHAPE, "invalid set size N=%lld n=%lld p=%lld", (long long)N, (long long)n, (long long)p);
  if ((pred_lb == nullptr) != (pred_ub == nullptr))
    NNV_FAIL(NNVHIP_ERR_SHAPE, "Inconsistency between number of predicate variables and predicate lower- or upper-bounds vector");
  if (p > 0 && (!C || !d)) NNV_FAIL(NNVHIP_ERR_SHAPE, "Inconsistency between constraint matrix and constraint vector");
  nnvhip_star* s = new_star(c);
  std::unique_ptr<nnvhip_star, int (*)(nnvhip_star*)> guard(s, nnvhip_star_release);
  s->N = N;
  s->n = n;
  s->ld = round_up(N, kLdAlign);
  NNV_TRY(c->alloc(sizeof(double) * s->ld * (n + 1), &s->Vbuf));
  s->V = s->Vbuf->as<double>();
  NNV_TRY(upload_matrix(c, V, N, n + 1, s->ld, s->V));
  int64_t npad = round_up(std::max<int64_t>(n, 1), kLdAlign);
  NNV_TRY(c->alloc(sizeof(double) * 2 * npad, &s->pbuf));
  s->plb = s->pbuf->as<double>();
  s->pub = s->plb + npad;
  if (n > 0) {
    std::vector<double> tmp(2 * npad, 0.0);
    for (int64_t i = 0; i < n; ++i) {
      tmp[i] = pred_lb ? pred_lb[i] : -1.0;  // default of Star.estimateRanges, set/Star.m:1091-1096
      tmp[npad + i] = pred_ub ? pred_ub[i] : 1.0;
    }
    NNV_HIP_TRY(hipMemcpyAsync(s->plb, tmp.data(), sizeof(double) * 2 * npad, hipMemcpyHostToDevice, c->stream));
    c->h2d_bytes += (int64_t)sizeof(double) * 2 * npad;
    NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  }
  auto base = make_cons(c);
  base->p_total = p;
  base->n_total = n;
  if (p > 0 && n > 0) {
    base->ldc = round_up(p, kLdAlign);
    NNV_TRY(c->alloc(sizeof(double) * base->ldc * n, &base->C0));
    NNV_TRY(upload_matrix(c, C, p, n, base->ldc, base->C0->as<double>()));
  }
  if (p > 0) {
    NNV_TRY(c->alloc(sizeof(double) * p, &base->d0));
    NNV_HIP_TRY(hipMemcpyAsync(base->d0->ptr, d, sizeof(double) * p, hipMemcpyHostToDevice, c->stream));
    c->h2d_bytes += (int64_t)sizeof(double) * p;
    NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  }
  s->cons = base;
  *out = guard.release();
  return NNVHIP_OK;
}

// Star(lb, ub) for every column of two N x count matrices.  A box's generators are scaled unit vectors, and the handle
// says which (oh_idx, oh_scale): only the centres go to memory (vcols = 1), back to back, and whoever reads the whole
// matrix has the columns written then (ensure_dense).  Everything the call puts on the device - centres, half-widths,
// predicate bounds, index lists - is laid out in pinned memory and travels from there together (nnvhip_ctx::copy_staged; pieces of kBoxPiece entries,
// so that the staging ring stays at 16 MB whatever the array's size).  (Writing the matrices took 133 us for 100 boxes of 784 dimensions, 1.54 ms for 1024 of them, 6.4 GB nobody read; seven small
// copies and kernels took 60 us of a single set's reach.)
constexpr int64_t kBoxPiece = int64_t(1) << 20;
// Host arrays of 1.5 MB and more are worth waking the context's workers for (some 20 us); several parts to a thread, so that
// one that starts late costs little.  Boxes on one thread and on four: 1400 of 100 dimensions (1.1 MB) 287 -> 305 us, 2000 of them
// (1.6 MB) 422 -> 401, 170 of 784 (1.1 MB) 224 -> 203, 512 of 784 (3.2 MB) 733 -> 599, 8000 of 20 (1.3 MB) 777 -> 787, 14 000 1813 -> 1716.
constexpr int64_t kPoolDoubles = int64_t(3) << 16;
static int host_parts(const nnvhip_ctx* c, int64_t doubles) { return doubles >= kPoolDoubles && !c->no_host_pool ? 4 * (HostPool::kWorkers + 1) : 1; }

int nnvhip_copy_host(nnvhip_ctx* c, int64_t n, const double* src, double* dst) {
  if (!c) NNV_FAIL(NNVHIP_ERR_ARG, "null context");
  if (n < 0 || (n > 0 && (!src || !dst))) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  const int parts = host_parts(c, n);
  c->host_pool.run(parts, [&](int part) {
    const int64_t a = n * part / parts, b = n * (part + 1) / parts;
    if (b > a) memcpy(dst + a, src + a, sizeof(double) * (size_t)(b - a));
  });
  return NNVHIP_OK;
}

int nnvhip_star_from_box(nnvhip_ctx* c, int64_t N, int64_t count, const double* lb, const double* ub,
                         nnvhip_star** out) {
  if (!c) NNV_FAIL(NNVHIP_ERR_ARG, "null context");
  NNV_TRY(nnvhip::enter_ctx(c, true));
  if (!lb || !ub || !out) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  if (N <= 0 || count <= 0 || count > 65535) NNV_FAIL(NNVHIP_ERR_SHAPE, "Inconsistent dimensions between lb and ub");
  const int64_t ld = round_up(N, kLdAlign);
  // Sets with the same half-widths, bit for bit (the boxes of a regular partition), share one scale vector and one
  // index list on the device: layers downstream recognise by the pointers that such sets gather the same scaled
  // weight columns.  shape_of[s] = the first set with set s's half-widths (among the first few distinct shapes).
  // Every shape that is not another set's has a record here.
  struct Shape {
    int64_t n = 0;        // dimensions with a width: generator columns
    int64_t idx_of = -1;  // the shape whose index list it uses (its own, or the first one with all dimensions)
    int64_t idx_off = 0, pb_off = 0;
    bool neg = false;
  };
  std::vector<int64_t> shape_of((size_t)count);  // index into shapes
  std::vector<Shape> shapes;
  std::vector<double> vecs;  // half-widths of the shapes, ld apart
  int64_t kept_shapes = 0;   // how many of them later sets are compared with
  std::vector<double> vec((size_t)ld, 0.0);
  // First pass: half-widths only (they decide the sizes); the centres are formed below, in their place.  Both passes over the
  // host arrays are bound by one thread's share of the memory bandwidth, so those of a large array are shared out: 1024 boxes of
  // 784 dimensions take 340 + 390 us on one thread (and their private copies 250); a reach of them 2.95 -> 2.03 - 2.10 ms, on bounds
  // not seen before 3.6 - 4.4 -> 2.8 - 3.5.  What the workers have read lies in their caches too, and whoever writes it next has those
  // copies invalidated first: a caller that makes its next bounds in the same memory takes 2.46 ms for it where it took 2.27 (26 MB
  // written by one thread after it was read by itself 0.77 ms, after four 1.2 - 1.6, after four have written it 0.77).
  const int parts = host_parts(c, count * N);
  auto half_widths = [&](int64_t s) {
    const double *l = lb + s * N, *u = ub + s * N;
    for (int64_t i = 0; i < N; ++i) vec[(size_t)i] = 0.5 * (u[i] - l[i]);  // Box constructor, set/Box.m:36
  };
  std::vector<char> as_first((size_t)count, 0);  // has the first set's half-widths, bit for bit (known where threads have looked)
  if (parts > 1) half_widths(0);
  if (parts > 1) c->host_pool.run(parts, [&](int part) {
    for (int64_t s = std::max<int64_t>(1, count * part / parts); s < count * (part + 1) / parts; ++s) {
      const double *l = lb + s * N, *u = ub + s * N;
      bool same = true;
      for (int64_t i0 = 0; i0 < N && same; i0 += 64) {
        double v[64];
        const int64_t m = std::min<int64_t>(64, N - i0);
        for (int64_t i = 0; i < m; ++i) v[i] = 0.5 * (u[i0 + i] - l[i0 + i]);
        same = memcmp(v, vec.data() + i0, sizeof(double) * (size_t)m) == 0;
      }
      as_first[(size_t)s] = same;
    }
  });
  for (int64_t s = 0; s < count; ++s) {
    if (as_first[(size_t)s]) continue;  // (shape 0)
    if (s > 0 || parts == 1) half_widths(s);
    int64_t found = -1;
    for (int64_t k = 0; k < kept_shapes && found < 0; ++k)
      if (memcmp(&vecs[(size_t)(k * ld)], vec.data(), sizeof(double) * N) == 0) found = k;
    if (found < 0) {
      found = (int64_t)shapes.size();
      Shape sh;
      if (N == 1) {
        sh.n = 1;  // zero columns are deleted only when the generator matrix has more than one element (set/Box.m:41-43)
      } else {
        for (int64_t i = 0; i < N; ++i) sh.n += vec[(size_t)i] != 0.0;
      }
      for (int64_t i = 0; i < N; ++i) sh.neg = sh.neg || vec[(size_t)i] < 0.0;
      shapes.push_back(sh);
      vecs.insert(vecs.end(), vec.begin(), vec.end());
      if (kept_shapes < 16 && found == kept_shapes) ++kept_shapes;
    }
    shape_of[(size_t)s] = found;
  }
  // layout of the one device block, in doubles: centres | half-widths by shape | predicate bounds by column count | lists
  const int64_t vec_off = ld * count;
  int64_t doubles = vec_off + ld * (int64_t)shapes.size();
  std::map<int64_t, int64_t> pb_at;  // column count -> offset of its -1 / +1 vectors
  for (Shape& sh : shapes) {
    auto at = pb_at.find(sh.n);
    if (at == pb_at.end()) {
      at = pb_at.emplace(sh.n, doubles).first;
      doubles += 2 * round_up(std::max<int64_t>(sh.n, 1), kLdAlign);
    }
    sh.pb_off = at->second;
  }
  int64_t ints = 0, full = -1;
  for (size_t k = 0; k < shapes.size(); ++k) {
    Shape& sh = shapes[k];
    if (sh.n == N && full >= 0) {
      sh.idx_of = full;
      continue;
    }
    sh.idx_of = (int64_t)k;
    sh.idx_off = ints;
    ints += round_up(std::max<int64_t>(sh.n, 1), kLdAlign);
    if (sh.n == N) full = (int64_t)k;
  }
  // (sets whose whole matrices no reader could be given are refused here, as they were when they were written)
  double whole = 0.0;
  for (int64_t s = 0; s < count; ++s) whole += 8.0 * (double)ld * (double)(shapes[(size_t)shape_of[(size_t)s]].n + 1);
  if (whole > (double)c->device_bytes) NNV_FAIL(NNVHIP_ERR_OOM, "out of device memory allocating %.0f bytes", whole);
  NNV_TRY(c->check_room((size_t)whole));
  // bounds and lists (what follows the half-widths)
  const int64_t tail_off = vec_off + ld * (int64_t)shapes.size(), total = doubles + (ints + 1) / 2;
  auto write_tail = [&](double* tail) {
    for (const auto& pb : pb_at) {
      const int64_t npad = round_up(std::max<int64_t>(pb.first, 1), kLdAlign);
      double* at = tail + (pb.second - tail_off);
      std::fill(at, at + npad, -1.0);
      std::fill(at + npad, at + 2 * npad, 1.0);
    }
    int32_t* lists = reinterpret_cast<int32_t*>(tail + (doubles - tail_off));
    for (size_t k = 0; k < shapes.size(); ++k) {
      const Shape& sh = shapes[k];
      if (sh.idx_of != (int64_t)k) continue;
      int32_t* list = lists + sh.idx_off;
      int64_t t = 0;
      for (int64_t i = 0; i < N; ++i)
        if (N == 1 || vecs[k * ld + i] != 0.0) list[t++] = (int32_t)i;
      for (const int64_t end = round_up(std::max<int64_t>(sh.n, 1), kLdAlign); t < end; ++t) list[t] = 0;
    }
  };
  std::vector<double> tail;  // (in one piece they are written in their place)
  if (total > kBoxPiece) {
    tail.resize((size_t)(total - tail_off));
    write_tail(tail.data());
  }
  const size_t bytes = sizeof(double) * (size_t)total;
  BufRef buf;
  NNV_TRY(c->alloc(bytes, &buf));
  for (int64_t e0 = 0; e0 < total; e0 += kBoxPiece) {
    const int64_t e1 = std::min(total, e0 + kBoxPiece);
    void* st = nullptr;
    NNV_TRY(c->stage(sizeof(double) * (size_t)(e1 - e0), &st));
    double* h = static_cast<double*>(st);  // the block's entries [e0, e1)
    int64_t e = std::max(e0, std::min(e1, vec_off));
    const int64_t np = host_parts(c, e - e0);
    c->host_pool.run((int)np, [&](int part) {  // centres
      int64_t q = e0 + (e - e0) * part / np;
      for (const int64_t q1 = e0 + (e - e0) * (part + 1) / np; q < q1;) {
        const int64_t s = q / ld, i0 = q - s * ld, i1 = std::min(ld, i0 + q1 - q);
        const double *l = lb + s * N, *u = ub + s * N;
        double* col = h + (q - e0);
        for (int64_t i = i0; i < std::min(i1, N); ++i) col[i - i0] = 0.5 * (l[i] + u[i]);  // set/Box.m:35
        for (int64_t i = std::max(i0, N); i < i1; ++i) col[i - i0] = 0.0;
        q += i1 - i0;
      }
    });
    if (e < std::min(e1, tail_off)) {
      const int64_t end = std::min(e1, tail_off);
      memcpy(h + (e - e0), vecs.data() + (e - vec_off), sizeof(double) * (size_t)(end - e));
      e = end;
    }
    if (e < e1 && tail.empty()) write_tail(h + tail_off);
    else if (e < e1) memcpy(h + (e - e0), tail.data() + (e - tail_off), sizeof(double) * (size_t)(e1 - e));
    NNV_TRY(c->copy_staged(buf, sizeof(double) * (size_t)e0, st, sizeof(double) * (size_t)(e1 - e0), e1 == total && e0 == 0));
  }
  c->h2d_bytes += (int64_t)bytes;
  double* d = buf->as<double>();
  const int32_t* di = reinterpret_cast<const int32_t*>(d + doubles);
  for (int64_t s = 0; s < count; ++s) {
    const int64_t k = shape_of[(size_t)s];
    const Shape& sh = shapes[(size_t)k];
    nnvhip_star* o = new_star(c);
    o->N = N;
    o->n = sh.n;
    o->ld = ld;
    o->Vbuf = buf;
    o->V = d + s * ld;
    o->pbuf = buf;
    o->plb = d + sh.pb_off;
    o->pub = o->plb + round_up(std::max<int64_t>(sh.n, 1), kLdAlign);
    // C = zeros(1, n), d = 0 (set/Star.m:226-227): a base node with one all-zero row
    auto base = make_cons(c);
    base->p_total = 1;
    base->n_total = o->n;
    o->cons = base;  // C0/d0 left null = all zeros
    o->has_zono = true;  // Z = Zono(center, gens), set/Star.m:230-236
    if (o->n > 0) {  // every generator column is vec(dim) * e_dim
      o->vcols = 1;
      o->oh_from = 1;
      o->oh_idx_buf = buf;
      o->oh_idx = di + shapes[(size_t)sh.idx_of].idx_off;
      o->oh_scale_buf = buf;
      o->oh_scale = d + vec_off + k * ld;
      o->oh_scale_neg = sh.neg;
    }
    out[s] = o;
  }
  return NNVHIP_OK;
}

// info[2k] = offset (in doubles) of block k, info[2k+1] = npad: lb half := -1, ub half := +1
__global__ void fill_pm_one_kernel(double* __restrict__ bounds, const int64_t* __restrict__ info) {
  const int64_t off = info[2 * blockIdx.y], npad = info[2 * blockIdx.y + 1];
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < npad) {
    bounds[off + i] = -1.0;
    bounds[off + npad + i] = 1.0;
  }
}

// Columns of the set the reduceMem suffix of the ReLU layer builds: column 0 the centre, column 1 + g the value
// val[g] on every channel of pixel pix[g] (rows pix[g] + k * HW), every other entry zero.
__global__ void rebox_fill_kernel(double* __restrict__ V, int64_t ld, int N, int HW, int64_t ncols, int ngen,
                                  const double* __restrict__ center, const int32_t* __restrict__ pix,
                                  const double* __restrict__ val) {
  for (int64_t j = blockIdx.y; j < ncols; j += gridDim.y) {
    double* col = V + j * ld;
    const int p = (j >= 1 && j - 1 < ngen) ? pix[j - 1] : -1;
    const double pv = p >= 0 ? val[j - 1] : 0.0;
    for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < ld; r += gridDim.x * blockDim.x) {
      double v = 0.0;
      if (r < N) {
        if (j == 0) v = center[r];
        else if (p >= 0 && r % HW == p) v = pv;
      }
      col[r] = v;
    }
  }
}

int nnvhip_relu_reduce_mem(nnvhip_ctx* c, nnvhip_star* in, int64_t H, int64_t W, int64_t C, nnvhip_star** out, double* im_lb,
                           double* im_ub) {
  CHECK_CTX(c);
  if (!in || in->ctx != c || !out) NNV_FAIL(NNVHIP_ERR_ARG, "invalid set handle");
  if (H <= 0 || W <= 0 || C <= 0 || H * W * C != in->N)
    NNV_FAIL(NNVHIP_ERR_SHAPE, "Inconsistent dimension in the ImageStar and the original Star set");
  const int64_t N = in->N, HW = H * W;
  // [l, u] = images(i).estimateRanges
  NNV_TRY(compute_ranges(c, 1, &in));
  std::vector<double> l((size_t)N), u((size_t)N);
  NNV_HIP_TRY(hipMemcpyAsync(l.data(), in->lb, sizeof(double) * N, hipMemcpyDeviceToHost, c->stream));
  NNV_HIP_TRY(hipMemcpyAsync(u.data(), in->ub, sizeof(double) * N, hipMemcpyDeviceToHost, c->stream));
  NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  // center = 0.5*(u+l); v = 0.5*(u-l); n = numel(find(l-u)); one generator per pixel (i1 outer, i2 inner) whose
  // first-channel half-width is non-zero
  std::vector<double> center((size_t)N), val;
  std::vector<int32_t> pix;
  int64_t n = 0;
  for (int64_t i = 0; i < N; ++i) {
    center[i] = 0.5 * (u[i] + l[i]);
    if (l[i] - u[i] != 0.0) ++n;
  }
  for (int64_t i1 = 0; i1 < H; ++i1)
    for (int64_t i2 = 0; i2 < W; ++i2) {
      const double bv = 0.5 * (u[i1 + i2 * H] - l[i1 + i2 * H]);
      if (bv != 0.0) {
        pix.push_back((int32_t)(i1 + i2 * H));
        val.push_back(bv);
      }
    }
  if ((int64_t)pix.size() > n) NNV_FAIL(NNVHIP_ERR_SHAPE, "Index exceeds the number of array elements");  // (cannot happen: C >= 1)
  nnvhip_star* s = new_star(c);
  std::unique_ptr<nnvhip_star, int (*)(nnvhip_star*)> guard(s, nnvhip_star_release);
  s->N = N;
  s->n = n;
  s->ld = round_up(N, kLdAlign);
  NNV_TRY(c->alloc(sizeof(double) * s->ld * (n + 1), &s->Vbuf));
  s->V = s->Vbuf->as<double>();
  BufRef dcen, dpix, dval;
  NNV_TRY(c->upload(center.data(), sizeof(double) * N, &dcen));
  const int ngen = (int)pix.size();
  if (pix.empty()) {  // (something to upload)
    pix.push_back(0);
    val.push_back(0.0);
  }
  NNV_TRY(c->upload(pix.data(), sizeof(int32_t) * pix.size(), &dpix));
  NNV_TRY(c->upload(val.data(), sizeof(double) * val.size(), &dval));
  dim3 grid((unsigned)std::min<int64_t>(ceil_div(s->ld, 256), 64), (unsigned)std::min<int64_t>(n + 1, 4096));
  hipLaunchKernelGGL(rebox_fill_kernel, grid, dim3(256), 0, c->stream, s->V, s->ld, (int)N, (int)HW, n + 1, ngen,
                     dcen->as<double>(), dpix->as<int32_t>(), dval->as<double>());
  NNV_HIP_TRY(hipGetLastError());
  // predicate bounds -1 / +1; C = zeros(1, n), d = 0
  const int64_t npad = round_up(std::max<int64_t>(n, 1), kLdAlign);
  NNV_TRY(c->alloc(sizeof(double) * 2 * npad, &s->pbuf));
  s->plb = s->pbuf->as<double>();
  s->pub = s->plb + npad;
  {
    const int64_t pinfo[2] = {0, npad};
    BufRef dinfo;
    NNV_TRY(c->upload(pinfo, sizeof(pinfo), &dinfo));
    hipLaunchKernelGGL(fill_pm_one_kernel, dim3((unsigned)ceil_div(npad, 256), 1), dim3(256), 0, c->stream, s->plb, dinfo->as<int64_t>());
    NNV_HIP_TRY(hipGetLastError());
  }
  auto base = make_cons(c);
  base->p_total = 1;
  base->n_total = n;
  s->cons = base;
  if (C == 1 && ngen == n && n > 0) {  // a plain box star: every generator is val * e_pix
    std::vector<double> scale((size_t)N, 0.0);
    bool neg = false;
    for (size_t g = 0; g < (size_t)ngen; ++g) {
      scale[pix[g]] = val[g];
      neg = neg || val[g] < 0.0;
    }
    BufRef dscale;
    NNV_TRY(c->upload(scale.data(), sizeof(double) * N, &dscale));
    s->oh_from = 1;
    s->oh_idx_buf = dpix;
    s->oh_idx = dpix->as<int32_t>();
    s->oh_scale_buf = dscale;
    s->oh_scale = dscale->as<double>();
    s->oh_scale_neg = neg;
  }
  if (im_lb) memcpy(im_lb, l.data(), sizeof(double) * N);
  if (im_ub) memcpy(im_ub, u.data(), sizeof(double) * N);
  *out = guard.release();
  return NNVHIP_OK;
}

int nnvhip_star_retain(nnvhip_star* s) {
  if (!s) NNV_FAIL(NNVHIP_ERR_ARG, "null set handle");
  s->refs.fetch_add(1);
  return NNVHIP_OK;
}

int nnvhip_star_release(nnvhip_star* s) {
  if (!s) return NNVHIP_OK;
  if (s->refs.fetch_sub(1) == 1) {
    delete_star(s);
  }
  return NNVHIP_OK;
}

int nnvhip_star_release_array(int64_t count, nnvhip_star* const* sets) {
  if (count < 0 || (count > 0 && !sets)) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  // a large array is let go later, where the host waits for the device anyway (nnvhip_ctx::deferred)
  const bool later = count >= 256;
  for (int64_t i = 0; i < count; ++i) {
    if (later && sets[i] != nullptr)
      sets[i]->ctx->deferred.push_back(sets[i]);
    else
      nnvhip_star_release(sets[i]);
  }
  return NNVHIP_OK;
}

int nnvhip_star_dims(const nnvhip_star* s, int64_t* N, int64_t* n, int64_t* p) {
  if (!s) NNV_FAIL(NNVHIP_ERR_ARG, "null set handle");
  if (N) *N = s->N;
  if (n) *n = s->n;
  if (p) *p = s->cons ? s->cons->p_total : 0;
  return NNVHIP_OK;
}

int nnvhip_star_has_zono(const nnvhip_star* s, int32_t* flag) {
  if (!s || !flag) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  *flag = s->has_zono ? 1 : 0;
  return NNVHIP_OK;
}

int nnvhip_star_has_user_constraints(const nnvhip_star* s, int32_t* flag) {
  if (!s || !flag) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  const ConsNode* nd = s->cons.get();
  while (nd && nd->prev) nd = nd->prev.get();
  *flag = (nd && nd->C0) ? 1 : 0;  // the base node holds dense rows only when a caller handed some in
  return NNVHIP_OK;
}

// Centre, scales (by row) and rows (by column) of a box of which only the centre is in memory.
// (In the staging ring; a box too large for a piece of it goes to `own`.)
static int fetch_box(const nnvhip_star* s, std::vector<char>* own, const double** centre, const double** scale, const int32_t** idx) {
  nnvhip_ctx* c = s->ctx;
  const size_t nd = sizeof(double) * (size_t)s->ld, bytes = 2 * nd + sizeof(int32_t) * (size_t)s->n;
  char* at = nullptr;
  if (bytes <= sizeof(double) * (size_t)kBoxPiece) {
    void* st = nullptr;
    NNV_TRY(c->stage(bytes, &st));
    at = static_cast<char*>(st);
  } else {
    own->resize(bytes);
    at = own->data();
  }
  NNV_HIP_TRY(hipMemcpyAsync(at, s->V, sizeof(double) * s->N, hipMemcpyDeviceToHost, c->stream));
  NNV_HIP_TRY(hipMemcpyAsync(at + nd, s->oh_scale, sizeof(double) * s->N, hipMemcpyDeviceToHost, c->stream));
  NNV_HIP_TRY(hipMemcpyAsync(at + 2 * nd, s->oh_idx, sizeof(int32_t) * s->n, hipMemcpyDeviceToHost, c->stream));
  NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  *centre = reinterpret_cast<const double*>(at);
  *scale = reinterpret_cast<const double*>(at + nd);
  *idx = reinterpret_cast<const int32_t*>(at + 2 * nd);
  return NNVHIP_OK;
}

int nnvhip_star_fetch_V(const nnvhip_star* s, double* V) {
  if (!s || !V) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  nnvhip_ctx* c = s->ctx;
  NNV_TRY(nnvhip::enter_ctx(c));
  // A box's matrix is put together here: nothing is written on the device for it (500 boxes of 10 dimensions, read one by one:
  // 52 ms with a pass on the device each, 46 when the constructor wrote them).
  if (is_unwritten_box(s)) {
    const double *centre, *scale;
    const int32_t* idx;
    std::vector<char> own;
    NNV_TRY(fetch_box(s, &own, &centre, &scale, &idx));
    memcpy(V, centre, sizeof(double) * (size_t)s->N);
    memset(V + s->N, 0, sizeof(double) * (size_t)(s->N * s->n));
    for (int64_t t = 0; t < s->n; ++t) V[(1 + t) * s->N + idx[t]] = scale[idx[t]];
    return NNVHIP_OK;
  }
  NNV_TRY(ensure_dense(c, const_cast<nnvhip_star*>(s)));  // implicit columns are written out on first read
  NNV_HIP_TRY(hipMemcpy2DAsync(V, sizeof(double) * s->N, s->V, sizeof(double) * s->ld, sizeof(double) * s->N,
                               s->n + 1, hipMemcpyDeviceToHost, c->stream));
  NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  return NNVHIP_OK;
}

int nnvhip_star_fetch_rows(const nnvhip_star* s, int64_t R, const int32_t* rows, double* out) {
  if (!s || (R > 0 && (!rows || !out)) || R < 0) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  if (R == 0) return NNVHIP_OK;
  nnvhip_ctx* c = s->ctx;
  for (int64_t t = 0; t < R; ++t)
    if (rows[t] < 0 || rows[t] >= s->N) NNV_FAIL(NNVHIP_ERR_ARG, "Invalid index");
  NNV_TRY(nnvhip::enter_ctx(c));
  if (is_unwritten_box(s)) {  // (as above; a column's row is found from the rows asked for: idx ascends)
    const double *centre, *scale;
    const int32_t* idx;
    std::vector<char> own;
    NNV_TRY(fetch_box(s, &own, &centre, &scale, &idx));
    memset(out, 0, sizeof(double) * (size_t)(R * (s->n + 1)));
    for (int64_t t = 0; t < R; ++t) {
      out[t] = centre[rows[t]];
      const int32_t* hit = std::lower_bound(idx, idx + s->n, rows[t]);
      if (hit != idx + s->n && *hit == rows[t]) out[(1 + (hit - idx)) * R + t] = scale[rows[t]];
    }
    return NNVHIP_OK;
  }
  NNV_TRY(ensure_dense(c, const_cast<nnvhip_star*>(s)));
  // gather on the device into an Rp x (n+1) matrix (Rp = R rounded up to whole K-tiles, the packing
  // kernel's granularity), one contiguous copy, then drop the padding rows on the host
  const int64_t Rp = round_up(R, kLdAlign), nc = s->n + 1;
  std::vector<int32_t> list((size_t)Rp, -1);
  std::copy(rows, rows + R, list.begin());
  BufRef dlist, packed;
  NNV_TRY(c->upload(list.data(), sizeof(int32_t) * Rp, &dlist));
  NNV_TRY(c->alloc(sizeof(double) * Rp * nc, &packed));
  PackSet ps{s->V, dlist->as<int32_t>(), packed->as<double>(), s->ld, (int32_t)Rp, (int32_t)nc};
  NNV_TRY(launch_pack_rows(c, 1, &ps));
  std::vector<double> tmp((size_t)(Rp * nc));
  NNV_HIP_TRY(hipMemcpyAsync(tmp.data(), packed->ptr, sizeof(double) * Rp * nc, hipMemcpyDeviceToHost, c->stream));
  NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  for (int64_t j = 0; j < nc; ++j) memcpy(out + j * R, tmp.data() + j * Rp, sizeof(double) * R);
  return NNVHIP_OK;
}

int nnvhip_star_fetch_pred_bounds(const nnvhip_star* s, double* lb, double* ub) {
  if (!s) NNV_FAIL(NNVHIP_ERR_ARG, "null set handle");
  nnvhip_ctx* c = s->ctx;
  NNV_TRY(nnvhip::enter_ctx(c));
  if (s->n > 0) {
    if (lb) NNV_HIP_TRY(hipMemcpyAsync(lb, s->plb, sizeof(double) * s->n, hipMemcpyDeviceToHost, c->stream));
    if (ub) NNV_HIP_TRY(hipMemcpyAsync(ub, s->pub, sizeof(double) * s->n, hipMemcpyDeviceToHost, c->stream));
  }
  NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  return NNVHIP_OK;
}

int nnvhip_star_fetch_constraints(const nnvhip_star* s, double* C, double* d) {
  if (!s) NNV_FAIL(NNVHIP_ERR_ARG, "null set handle");
  NNV_TRY(nnvhip::enter_ctx(s->ctx));
  return materialize_constraints(s, C, d);
}

int nnvhip_star_relu_counts(const nnvhip_star* s, int64_t* n_inactive, int64_t* n_crossing) {
  if (!s) NNV_FAIL(NNVHIP_ERR_ARG, "null set handle");
  if (s->n_crossing < 0) NNV_FAIL(NNVHIP_ERR_ARG, "set was not produced by the ReLU step");
  if (n_inactive) *n_inactive = s->n_inactive;
  if (n_crossing) *n_crossing = s->n_crossing;
  return NNVHIP_OK;
}

int nnvhip_star_fetch_crossing(const nnvhip_star* s, int32_t* index, double* lb, double* ub) {
  if (!s) NNV_FAIL(NNVHIP_ERR_ARG, "null set handle");
  if (s->n_crossing < 0) NNV_FAIL(NNVHIP_ERR_ARG, "set was not produced by the ReLU step");
  nnvhip_ctx* c = s->ctx;
  NNV_TRY(nnvhip::enter_ctx(c));
  const ConsNode* node = s->cons.get();
  int64_t m = s->n_crossing;
  if (m > 0) {
    if (index) NNV_HIP_TRY(hipMemcpyAsync(index, node->index->as<int32_t>() + node->index_off, sizeof(int32_t) * m, hipMemcpyDeviceToHost, c->stream));
    const double* lbub = node->lbub->as<double>() + node->lbub_off;
    if (lb) NNV_HIP_TRY(hipMemcpyAsync(lb, lbub, sizeof(double) * m, hipMemcpyDeviceToHost, c->stream));
    if (ub) NNV_HIP_TRY(hipMemcpyAsync(ub, lbub + node->ld_lbub, sizeof(double) * m, hipMemcpyDeviceToHost, c->stream));
  }
  NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  return NNVHIP_OK;
}

int nnvhip_estimate_ranges(nnvhip_ctx* c, nnvhip_star* s, double* lb, double* ub) {
  return nnvhip_estimate_ranges_batch(c, 1, &s, lb, ub);
}

int nnvhip_estimate_ranges_static(nnvhip_ctx* c, const nnvhip_star* s, double* lb_dev, double* ub_dev) {
  CHECK_CTX(c);
  if (!s || s->ctx != c) NNV_FAIL(NNVHIP_ERR_ARG, "invalid set handle");
  if (!lb_dev && !ub_dev) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  return ranges_into_static(c, s, lb_dev, ub_dev);
}

int nnvhip_estimate_ranges_batch(nnvhip_ctx* c, int64_t count, nnvhip_star* const* s, double* lb, double* ub) {
  CHECK_CTX(c);
  if (!s || count <= 0) NNV_FAIL(NNVHIP_ERR_ARG, "null argument");
  for (int64_t i = 0; i < count; ++i) {
    if (!s[i] || s[i]->ctx != c) NNV_FAIL(NNVHIP_ERR_ARG, "invalid set handle %lld", (long long)i);
    if (s[i]->N != s[0]->N) NNV_FAIL(NNVHIP_ERR_SHAPE, "sets of one array must have the same dimension");
  }
  NNV_TRY(c->begin_op());
  NNV_TRY(compute_ranges(c, count, s));
  NNV_TRY(c->end_op());
  if (lb || ub) {
    int64_t N = s[0]->N;
    if (2 * N * count <= kPostMax) return post_ranges(c, count, s, lb, ub);
    // ranges computed by one call sit at a fixed stride in one buffer
    const int64_t stride = count > 1 ? s[1]->lb - s[0]->lb : 0;
    bool regular = count > 1 && stride >= N;
    for (int64_t i = 1; i < count && regular; ++i)
      regular = s[i]->rbuf == s[0]->rbuf && s[i]->lb == s[0]->lb + i * stride && s[i]->ub == s[0]->ub + i * stride;
    if (regular && stride <= 4 * N + 64) {
      // one contiguous copy of the whole range buffer, unpacked on the host (strided 2-D copies of
      // short rows are issued row by row by the runtime)
      const int64_t off_ub = s[0]->ub - s[0]->lb;
      std::vector<double> tmp((size_t)(stride * (count - 1) + std::max<int64_t>(N, off_ub + N)));
      NNV_HIP_TRY(hipMemcpyAsync(tmp.data(), s[0]->lb, sizeof(double) * tmp.size(), hipMemcpyDeviceToHost, c->stream));
      NNV_HIP_TRY(hipStreamSynchronize(c->stream));
      for (int64_t i = 0; i < count; ++i) {
        if (lb) std::copy(tmp.begin() + i * stride, tmp.begin() + i * stride + N, lb + i * N);
        if (ub) std::copy(tmp.begin() + i * stride + off_ub, tmp.begin() + i * stride + off_ub + N, ub + i * N);
      }
      return NNVHIP_OK;
    } else {
      for (int64_t i = 0; i < count; ++i) {
        if (lb) NNV_HIP_TRY(hipMemcpyAsync(lb + i * N, s[i]->lb, sizeof(double) * N, hipMemcpyDeviceToHost, c->stream));
        if (ub) NNV_HIP_TRY(hipMemcpyAsync(ub + i * N, s[i]->ub, sizeof(double) * N, hipMemcpyDeviceToHost, c->stream));
      }
    }
    NNV_HIP_TRY(hipStreamSynchronize(c->stream));
  }
  return NNVHIP_OK;
}

}  // extern "C"
