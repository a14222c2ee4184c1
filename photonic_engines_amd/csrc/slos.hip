// SLOS strong simulation on MI355X (gfx950): plan, C ABI and kernels.
//
// Forward path (replaces FockSLOSKernel._amplitudes / probs, photonic_engines/slos/kernel.py:201-283):
// one launch per photon layer, pull form — each child state sums its parents, whose lex ranks
// are computed from the child's own sorted positions with the counting table (space.hpp), so no
// state or edge table exists anywhere. Every child is written exactly once; there are no atomics.
// The last layer's launch squares, normalises and writes float32 probabilities (or scaled
// complex64 amplitudes) directly.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include <rocprofiler-sdk-roctx/roctx.h>

#include "../../include/slos_mi355x.h"
#include "space.hpp"
#include "layer_block.hpp"
#include "descend_block.hpp"
#include "layer_f64.hpp"
#include "layer_simple.hpp"
#include "pull_index.hpp"
#include "block_launch.hpp"
#include "front.hpp"
#include "raise.hpp"
#include "adjoint_modes.hpp"
#include "descend_tail.hpp"

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(expr)                                                            \
  do {                                                                           \
    hipError_t e_ = (expr);                                                      \
    if (e_ != hipSuccess)                                                        \
      return fail(SLOS_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

constexpr int kMaxPhotons = 32;

}  // namespace

struct DevTables {
  int device = -1;
  uint64_t* cg = nullptr;
  int* lo = nullptr;
  int* modes = nullptr;                    // the plan's input modes (spot permanents)
  slos::TupleWord* tuples = nullptr;       // block-kernel suffix-tuple words (may be absent)
  uint64_t* tuples5 = nullptr;             // the same for 5-position suffixes (may be absent)
  uint32_t* xm[33] = {};                   // x-model rows of the levels 0..L (see xmodel_tables)
  uint32_t* insert = nullptr;              // insert table of the pulls over children (see insert_table)
  uint4* items[33] = {};                   // group-order work items of layer K (may be absent)
  uint32_t n_items[33] = {};
  uint4* fine[33] = {};                    // the same in small items (may be absent)
  uint32_t n_fine[33] = {};
  // the items for a launch of `states` states in all
  std::pair<const uint4*, uint32_t> group_items(int K, uint64_t states) const {
    return fine[K] && states < kFineItems ? std::make_pair((const uint4*)fine[K], n_fine[K])
                                          : std::make_pair((const uint4*)items[K], n_items[K]);
  }
  static constexpr uint64_t kFineItems = 1ull << 23;
};

// The rows of the x-model's levels 0..L (raise.hpp): masks of a level from at[level] on, and from
// off[level] on, per row of the level, the index of its first source in the next level (one more entry:
// their number); `zeros`: as many zero entries as the largest level has rows, and one.
struct XRows {
  std::vector<uint32_t> words;
  std::vector<size_t> at, off, rows;
  size_t zeros = 0;
  uint64_t most = 0;
};

struct slos_plan {
  int n = 0, m = 0, mask = 0, me = 0, multiset = 1, shift = 0;
  std::vector<int> modes;
  std::vector<uint64_t> cg;  // (n + 2) x (me + 1)
  std::vector<int> lo;
  double s_fact = 1.0;       // prod_i s_i!
  std::vector<slos::TupleWord> tuples;   // suffix-tuple words of the block kernel (empty: unused)
  std::vector<uint64_t> tuples5;         // 5-position suffix-tuple words (empty: unused)
  std::vector<uint32_t> items[33];       // group-order work items of layer K, 4 words each (empty: unused)
  std::vector<uint32_t> fine[33];        // the same in small items, for layers of fewer than kFineItems states
  std::unique_ptr<const XRows> xrows[33];  // x-model rows of the levels 0..L, built by the first call
  std::vector<DevTables> dev;
  std::mutex mu;
  slos::SpaceView host_view() const { return slos::SpaceView{cg.data(), lo.data(), me, me + 1}; }
  uint64_t size(int k) const { return cg[(size_t)k * (me + 1)]; }
};

namespace {

// A roctx range over a scope (rocprofv3 --marker-trace shows it; without a profiler it is a no-op
// call): the forward, each of its layers and each descent step are named ranges, so a trace ties
// every kernel to its layer.
struct RoctxRange {
  explicit RoctxRange(const char* name) { roctxRangePushA(name); }
  ~RoctxRange() { roctxRangePop(); }
  RoctxRange(const RoctxRange&) = delete;
  RoctxRange& operator=(const RoctxRange&) = delete;
};

// LDS one work group may use on the current GPU (hipDeviceAttributeMaxSharedMemoryPerBlock; 160 KB
// on gfx950), read once per device. Should the query fail, 64 KB (the LDS of every earlier CDNA
// part) is assumed, so launches only get more conservative.
size_t lds_limit() {
  static std::mutex mu;
  static std::vector<std::pair<int, size_t>> seen;
  int d = 0;
  if (hipGetDevice(&d) != hipSuccess) return 64 * 1024;
  std::lock_guard<std::mutex> g(mu);
  for (const auto& e : seen)
    if (e.first == d) return e.second;
  int v = 0;
  size_t lim = 64 * 1024;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, d) == hipSuccess && v > 0) lim = (size_t)v;
  seen.emplace_back(d, lim);
  return lim;
}

__global__ void k_insert_table(const uint64_t* cg, const slos::TupleWord* tuples, int me, uint32_t n4, uint32_t words,
                               uint32_t* ins) {
  const int W = me + 1, X = slos::insert_from(me);
  const uint32_t first = n4 * (uint32_t)me, n5 = (uint32_t)cg[5 * W + X];
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += gridDim.x * blockDim.x) {
    if (i < first) {
      const slos::TupleWord w = tuples[i % n4];
      const int t[4] = {(int)(w & 63u), (int)((w >> 8) & 63u), (int)((w >> 16) & 63u), (int)((w >> 24) & 63u)};
      ins[i] = slos::insert_word<4>(cg, W, t, (int)(i / n4), 0);
    } else {
      uint64_t r = (i - first) % n5;
      int t[5], x = X;
      for (int l = 0; l < 5; ++l) {  // 5-tuple r of the modes from X on
        const uint64_t* c = cg + (5 - l) * W;
        const uint64_t top = c[x];
        while (x < me - 1 && top - c[x + 1] <= r) ++x;
        r -= top - c[x];
        t[l] = x;
      }
      ins[i] = slos::insert_word<5>(cg, W, t, X + (int)((i - first) / n5), X);
    }
  }
}

int device_tables(const slos_plan* cp, DevTables* out) {
  slos_plan* p = const_cast<slos_plan*>(cp);
  int d = 0;
  HIP_TRY(hipGetDevice(&d));
  std::lock_guard<std::mutex> g(p->mu);
  for (auto& t : p->dev)
    if (t.device == d) {
      *out = t;
      return SLOS_OK;
    }
  DevTables t;
  t.device = d;
  HIP_TRY(hipMalloc(&t.cg, p->cg.size() * sizeof(uint64_t)));
  HIP_TRY(hipMalloc(&t.lo, std::max<size_t>(1, p->lo.size()) * sizeof(int)));
  HIP_TRY(hipMemcpy(t.cg, p->cg.data(), p->cg.size() * sizeof(uint64_t), hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(t.lo, p->lo.data(), p->lo.size() * sizeof(int), hipMemcpyHostToDevice));
  HIP_TRY(hipMalloc(&t.modes, p->modes.size() * sizeof(int)));
  HIP_TRY(hipMemcpy(t.modes, p->modes.data(), p->modes.size() * sizeof(int), hipMemcpyHostToDevice));
  if (!p->tuples.empty()) {
    HIP_TRY(hipMalloc(&t.tuples, p->tuples.size() * sizeof(slos::TupleWord)));
    HIP_TRY(hipMemcpy(t.tuples, p->tuples.data(), p->tuples.size() * sizeof(slos::TupleWord),
                      hipMemcpyHostToDevice));
  }
  if (!p->tuples5.empty()) {
    HIP_TRY(hipMalloc(&t.tuples5, p->tuples5.size() * sizeof(uint64_t)));
    HIP_TRY(hipMemcpy(t.tuples5, p->tuples5.data(), p->tuples5.size() * sizeof(uint64_t), hipMemcpyHostToDevice));
  }
  for (int K = 0; K <= p->n; ++K)
    if (!p->items[K].empty()) {
      HIP_TRY(hipMalloc(&t.items[K], p->items[K].size() * sizeof(uint32_t)));
      HIP_TRY(hipMemcpy(t.items[K], p->items[K].data(), p->items[K].size() * sizeof(uint32_t), hipMemcpyHostToDevice));
      t.n_items[K] = (uint32_t)(p->items[K].size() / 4);
      if (!p->fine[K].empty()) {
        HIP_TRY(hipMalloc(&t.fine[K], p->fine[K].size() * sizeof(uint32_t)));
        HIP_TRY(hipMemcpy(t.fine[K], p->fine[K].data(), p->fine[K].size() * sizeof(uint32_t), hipMemcpyHostToDevice));
        t.n_fine[K] = (uint32_t)(p->fine[K].size() / 4);
      }
    }
  p->dev.push_back(t);
  *out = t;
  return SLOS_OK;
}

// Allocations in its scope neither fail for nor end a graph capture of another thread (whose mode may
// forbid them to every thread).
struct BesideCaptures {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  BesideCaptures() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~BesideCaptures() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  BesideCaptures(const BesideCaptures&) = delete;
  BesideCaptures& operator=(const BesideCaptures&) = delete;
};

bool has_insert_table(const slos_plan* p) {
  return p->multiset && !p->tuples.empty() && p->n >= 5 && p->size(5) <= slos::kInsertTuples &&
         p->tuples.size() * (uint64_t)p->me <= slos::kInsertWords;
}

// The plan's insert table on the current GPU, built by the first pull over children that asks for it
// (1.7 MB and about 50 us at 24 modes); null where the space has none, where there is no memory for it, or
// while `st` is captured and it is not there yet (nothing is allocated inside a capture).
int insert_table(const slos_plan* cp, hipStream_t st, const uint32_t** out) {
  slos_plan* p = const_cast<slos_plan*>(cp);
  *out = nullptr;
  if (!has_insert_table(p)) return SLOS_OK;
  const uint64_t n4 = p->tuples.size(), first = n4 * (uint64_t)p->me;
  const int X = slos::insert_from(p->me);
  const uint64_t words = first + (uint64_t)(p->me - X) * p->cg[(size_t)5 * (p->me + 1) + X];
  int d = 0;
  HIP_TRY(hipGetDevice(&d));
  std::lock_guard<std::mutex> g(p->mu);
  for (auto& t : p->dev)
    if (t.device == d) {
      if (!t.insert) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        HIP_TRY(hipStreamIsCapturing(st, &cap));
        if (cap != hipStreamCaptureStatusNone) return SLOS_OK;
        uint32_t* ins = nullptr;
        const BesideCaptures guard;
        if (hipMalloc(&ins, words * sizeof(uint32_t)) != hipSuccess) {
          (void)hipGetLastError();  // no memory: the kernels without the table
          return SLOS_OK;
        }
        hipLaunchKernelGGL(k_insert_table, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, t.cg, t.tuples, p->me,
                           (uint32_t)n4, (uint32_t)words, ins);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(st);  // other streams may read it from here on
        if (e != hipSuccess) {
          (void)hipFree(ins);
          HIP_TRY(e);
        }
        t.insert = ins;
      }
      *out = t.insert;
    }
  return SLOS_OK;
}

__global__ void k_fill_ones(float2* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = make_float2(1.f, 0.f);
}

// the output of layer 0, the vacuum (one state a batch row): probability |scale|^2, amplitude scale
__global__ void k_vacuum_out(void* out, int64_t n, int probs, float scale) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    if (probs) static_cast<float*>(out)[i] = scale * scale;
    else static_cast<float2*>(out)[i] = make_float2(scale, 0.f);
  }
}

// ------------------------------------------------------------------------------------------
// FP64 mass: per-block partial sums, then one block per batch row
// ------------------------------------------------------------------------------------------

constexpr int kMassBlocks = 1024;

__device__ double block_sum(double v) {
  __shared__ double sh[16];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = 0;
  if (threadIdx.x == 0)
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r += sh[i];
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(256) void k_mass_partial(const float* p, uint64_t count, double* part) {
  const int64_t b = blockIdx.y;
  const float* row = p + (size_t)b * count;
  double s = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (uint64_t)gridDim.x * blockDim.x)
    s += (double)row[i];
  s = block_sum(s);
  if (threadIdx.x == 0) part[(size_t)b * gridDim.x + blockIdx.x] = s;
}

__global__ __launch_bounds__(256) void k_mass_final(const double* part, int nb, double* out) {
  double s = 0;
  for (int i = threadIdx.x; i < nb; i += blockDim.x) s += part[(size_t)blockIdx.x * nb + i];
  s = block_sum(s);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// ------------------------------------------------------------------------------------------
// Group sums (GroupedSLOSKernel): a keyed reduction without atomics. The states are listed in group
// order (`order`), cut into chunks (4096 entries balance the waves); one wave sums a chunk's
// probabilities in FP64 (lane-strided, then a fixed butterfly), and one thread per group sums its
// chunks' partials in ascending order. Every addition has a fixed place, so the sums are
// reproducible run to run. T: float32 or float64 probabilities (and sums).
// ------------------------------------------------------------------------------------------
template <class T>
__global__ __launch_bounds__(256) void k_group_partial(const T* probs, uint64_t count, const int64_t* order,
                                                       const int64_t* chunks, uint32_t n_chunks, double* part) {
  const uint32_t c = blockIdx.x * 4u + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (c >= n_chunks) return;
  const int64_t b = blockIdx.y;
  const T* pb = probs + (size_t)b * count;
  const int64_t i0 = chunks[2 * (size_t)c], i1 = chunks[2 * (size_t)c + 1];
  double s = 0.0;
  for (int64_t i = i0 + lane; i < i1; i += 64) s += (double)pb[order[i]];
#pragma unroll
  for (int w = 32; w >= 1; w >>= 1) s += __shfl_xor(s, w, 64);
  if (lane == 0) part[(size_t)b * n_chunks + c] = s;
}

template <class T>
__global__ __launch_bounds__(256) void k_group_final(const double* part, uint32_t n_chunks, const uint32_t* first,
                                                     int n_groups, T* out) {
  const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (g >= n_groups) return;
  const int64_t b = blockIdx.y;
  double s = 0.0;
  for (uint32_t c = first[g]; c < first[g + 1]; ++c) s += part[(size_t)b * n_chunks + c];
  out[(size_t)b * n_groups + g] = (T)s;
}

// ------------------------------------------------------------------------------------------
// FP64 Ryser permanents for spot checks (one thread per output state)
// ------------------------------------------------------------------------------------------

__global__ __launch_bounds__(64) void k_spot_ryser(const uint64_t* cg_g, const int* lo_g, int me, int n, int m,
                                                   const double2* U, const int* modes, double s_fact,
                                                   int multiset, const uint64_t* idx, int64_t count,
                                                   double* out) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= count) return;
  const slos::SpaceView sv{cg_g, lo_g, me, me + 1};
  int p[kMaxPhotons];
  sv.unrank(idx[q], n, p);
  double tf = 1.0, run = 1.0;
  if (multiset)
    for (int i = 1; i < n; ++i) {
      run = (p[i] == p[i - 1]) ? run + 1.0 : 1.0;
      tf *= run;
    }
  double rre[kMaxPhotons], rim[kMaxPhotons];
  for (int i = 0; i < n; ++i) rre[i] = rim[i] = 0.0;
  double tre = 0.0, tim = 0.0;
  uint64_t prev = 0;
  for (uint64_t k = 1; k < (1ull << n); ++k) {
    const uint64_t gray = k ^ (k >> 1);
    const uint64_t diff = gray ^ prev;
    prev = gray;
    const int c = __builtin_ctzll(diff);
    const double sg = (gray & diff) ? 1.0 : -1.0;
    double pre = 1.0, pim = 0.0;
    for (int i = 0; i < n; ++i) {
      const double2 u = U[(size_t)p[i] * m + modes[c]];
      rre[i] += sg * u.x;
      rim[i] += sg * u.y;
      const double nr = pre * rre[i] - pim * rim[i];
      pim = pre * rim[i] + pim * rre[i];
      pre = nr;
    }
    const int pc = __builtin_popcountll(gray);
    if ((n - pc) & 1) { tre -= pre; tim -= pim; } else { tre += pre; tim += pim; }
  }
  out[q] = (tre * tre + tim * tim) / (s_fact * tf);
}


// ------------------------------------------------------------------------------------------
// uniform loss: q_{k-1}(t) = sum_j q_k(t + e_j) (t_j + 1) / k  (pull over children, no atomics)
// ------------------------------------------------------------------------------------------
// (child ranks: slos::children_fixed in pull_index.hpp; k - 1 <= KM)
template <int KM, class SV = slos::SpaceView, bool EXACT = false>
__global__ __launch_bounds__(256) void k_descend(const uint64_t* cg_g, const int* lo_g, int me, int multiset, int kk,
                                                 const float* __restrict__ qk, uint64_t Sk,
                                                 float* __restrict__ qout, uint64_t Sp, int64_t B, float scale) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef slos::RankT<SV> R;
  const int k = EXACT ? KM + 1 : kk;
  const int stride = me + 1;
  const int ncg = (k + 1) * stride;
  R* cg = reinterpret_cast<R*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = (R)cg_g[i];
  for (int i = threadIdx.x; i < me; i += blockDim.x) lo[i] = lo_g[i];
  __syncthreads();
  const SV sv{cg, lo, me, stride};
  const float invk = 1.f / (float)k;
  for (int64_t b = blockIdx.y; b < B; b += gridDim.y) {
    const float* qb = qk + (size_t)b * Sk;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < Sp; t += (uint64_t)gridDim.x * blockDim.x) {
      int p[KM];
      slos::unrank_fixed<KM>(sv, (R)t, k - 1, p);
      float acc = 0.f;
      if constexpr (EXACT) acc = slos::children_sum<KM>(sv, multiset, k, p, qb);
      else slos::children_fixed<KM>(sv, multiset, k, p, [&](R c, int, int cnt) { acc = fmaf(qb[c], (float)cnt, acc); });
      qout[(size_t)b * Sp + t] = (acc * invk) * scale;
    }
  }
}

// probability-level raise (a photon that interferes with nothing, partial distinguishability):
// q_k(c) = sum_{j distinct in c} w[b][j] q_{k-1}(c - e_j), w = |U[:, col]|^2 (pull over parents,
// ascending photon position, no atomics; k <= KM)
template <int KM>
__global__ __launch_bounds__(256) void k_raise(const uint64_t* cg_g, const int* lo_g, int me, int multiset, int k, int m,
                                               const float* __restrict__ w, const float* __restrict__ qp, uint64_t Sp,
                                               float* __restrict__ qout, uint64_t Sk, int64_t B) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int stride = me + 1;
  const int ncg = (k + 1) * stride;
  uint64_t* cg = reinterpret_cast<uint64_t*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  float* wl = reinterpret_cast<float*>(lo + me);
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = cg_g[i];
  for (int i = threadIdx.x; i < me; i += blockDim.x) lo[i] = lo_g[i];
  const slos::SpaceView sv{cg, lo, me, stride};
  for (int64_t b = blockIdx.y; b < B; b += gridDim.y) {
    __syncthreads();
    for (int j = threadIdx.x; j < m; j += blockDim.x) wl[j] = w[(size_t)b * m + j];
    __syncthreads();
    const float* qb = qp + (size_t)b * Sp;
    for (uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; c < Sk; c += (uint64_t)gridDim.x * blockDim.x) {
      int p[KM];
      slos::unrank_fixed<KM>(sv, c, k, p);
      float acc = 0.f;
      slos::parents_fixed<KM>(sv, multiset, k, p, [&](uint64_t pr, int mode, int) { acc = fmaf(wl[mode], qb[pr], acc); });
      qout[(size_t)b * Sk + c] = acc;
    }
  }
}

// adjoint of the descent (gradient of q_{k-1} w.r.t. q_k): g_k[c] = sum_{j distinct in c}
// g_{k-1}[c - e_j] * count_j(c) / k  — the forward pull structure with real weights (k <= KM)
template <int KM>
__global__ __launch_bounds__(256) void k_ascend(const uint64_t* cg_g, const int* lo_g, int me, int multiset, int k,
                                                const float* __restrict__ gp, uint64_t Sp,
                                                float* __restrict__ gk, uint64_t Sk, int64_t B) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int stride = me + 1;
  const int ncg = (k + 1) * stride;
  uint64_t* cg = reinterpret_cast<uint64_t*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = cg_g[i];
  for (int i = threadIdx.x; i < me; i += blockDim.x) lo[i] = lo_g[i];
  __syncthreads();
  const slos::SpaceView sv{cg, lo, me, stride};
  const int K = k;
  const float invk = 1.f / (float)k;
  for (int64_t b = blockIdx.y; b < B; b += gridDim.y) {
    const float* pb = gp + (size_t)b * Sp;
    for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < Sk; g += (uint64_t)gridDim.x * blockDim.x) {
      int p[KM];
      slos::unrank_fixed<KM>(sv, g, K, p);
      float acc = 0.f;
      slos::parents_fixed<KM>(sv, multiset, K, p, [&](uint64_t pr, int, int cnt) { acc += pb[pr] * (float)cnt; });
      gk[(size_t)b * Sk + g] = acc * invk;
    }
  }
}


// ------------------------------------------------------------------------------------------
// adjoint (reverse-mode) kernels; torch's convention for complex leaves: grad z = dL/dRe z + i dL/dIm z
// ------------------------------------------------------------------------------------------

// readout: p = |a s|^2 f  =>  g_a = 2 s^2 f grad_p a. grad_p is read first: where it is zero the
// gradient is zero, and neither the amplitude nor the state's factor (its unrank) is needed. A loss
// over a few sampled outputs leaves grad_p zero almost everywhere, so the pass then reads grad_p and
// writes g only; elsewhere it computes the same products as without the test.
__global__ __launch_bounds__(256) void k_readout_adjoint(const uint64_t* cg_g, const int* lo_g, int me, int multiset, int K,
                                                         const float2* __restrict__ a, const float* __restrict__ gp,
                                                         float2* __restrict__ g, uint64_t S, int64_t B, float s2) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int stride = me + 1;
  const int ncg = (K + 1) * stride;
  uint64_t* cg = reinterpret_cast<uint64_t*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = cg_g[i];
  for (int i = threadIdx.x; i < me; i += blockDim.x) lo[i] = lo_g[i];
  __syncthreads();
  const slos::SpaceView sv{cg, lo, me, stride};
  for (uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; c < S; c += (uint64_t)gridDim.x * blockDim.x) {
    bool have_f = false;
    float f = 0.f;
    for (int64_t b = blockIdx.y; b < B; b += gridDim.y) {
      const float gv = gp[(size_t)b * S + c];
      float2 r = make_float2(0.f, 0.f);
      if (gv != 0.f) {
        if (!have_f) {
          int p[kMaxPhotons];
          sv.unrank(c, K, p);
          f = slos::run_factorial(p, K, multiset);
          have_f = true;
        }
        const float2 v = a[(size_t)b * S + c];
        const float w = 2.f * s2 * f * gv;
        r = make_float2(w * v.x, w * v.y);
      }
      g[(size_t)b * S + c] = r;
    }
  }
}

// The same adjoint from layer K - 1 instead of layer K: where grad_p is nonzero the state's raw
// amplitude is pulled from its parents in `par` (the parent sum of k_layer_simple, plain sums);
// elsewhere the gradient is zero. For a grad_p that is zero almost everywhere this replaces the
// recompute of layer K and the read of its amplitudes by one pass that reads grad_p and writes g.
template <int KM>
__global__ __launch_bounds__(256) void k_readout_adjoint_pull(const uint64_t* cg_g, const int* lo_g, int me, int multiset,
                                                              int K, int m, int col, const float2* __restrict__ U,
                                                              const float2* __restrict__ par, uint64_t S_par,
                                                              const float* __restrict__ gp, float2* __restrict__ g,
                                                              uint64_t S, int64_t B, float s2) {
  // the counting tables are read from global memory: only the rare nonzero entries unrank, so
  // staging them in LDS per work group would cost more than it saves
  const slos::SpaceView sv{cg_g, lo_g, me, me + 1};
  for (uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; c < S; c += (uint64_t)gridDim.x * blockDim.x) {
    bool have_p = false;
    int p[KM];
    float f = 0.f;
    for (int64_t b = blockIdx.y; b < B; b += gridDim.y) {
      const float gv = gp[(size_t)b * S + c];
      float2 r = make_float2(0.f, 0.f);
      if (gv != 0.f) {
        if (!have_p) {
          slos::unrank_fixed<KM>(sv, c, K, p);
          f = slos::run_factorial_fixed<KM>(p, K, multiset);
          have_p = true;
        }
        const float2* ub = U + (size_t)b * m * m;
        const float2* pb = par + (size_t)b * S_par;
        slos::BlockAcc<false> acc;
        slos::parents_fixed<KM>(sv, multiset, K, p,
                                [&](uint64_t pr, int mode, int) { slos::bk_cmac(acc, ub[(size_t)mode * m + col], pb[pr]); });
        const float w = 2.f * s2 * f * gv;
        r = make_float2(w * acc.re, w * acc.im);
      }
      g[(size_t)b * S + c] = r;
    }
  }
}

// g_{k-1}[t] = sum_{children c = t + e_j} conj(U[b, j, col]) g_k[c]   (pull over children)
// and, per thread, gU_j += conj(psi_{k-1}[t]) g_k[t + e_j] in a private LDS row (no atomics);
// each block then reduces its rows to partial[b][block][j] (FP64 stage in k_reduce_gu)
// (k - 1 <= KM)
constexpr int kAdjThreads = 64;
template <int KM, class SV = slos::SpaceView, bool EXACT = false>
__global__ __launch_bounds__(kAdjThreads) void k_adjoint_layer(const uint64_t* cg_g, const int* lo_g, int me, int multiset,
                                                             int kk, int m, int col, const float2* __restrict__ U,
                                                             const float2* __restrict__ psi, const float2* __restrict__ gk,
                                                             uint64_t Sk, float2* __restrict__ gout, uint64_t Sp,
                                                             double2* __restrict__ partial, int want_psi_grad) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef slos::RankT<SV> R;
  const int k = EXACT ? KM + 1 : kk;
  const int stride = me + 1;
  const int ncg = (k + 1) * stride;
  R* cg = reinterpret_cast<R*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  float2* ucol = reinterpret_cast<float2*>(smem + ((ncg * 8 + me * 4 + 15) & ~15));
  float2* slots = ucol + m;  // [kAdjThreads][me]
  const int64_t b = blockIdx.y;
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = (R)cg_g[i];
  for (int i = threadIdx.x; i < me; i += blockDim.x) lo[i] = lo_g[i];
  for (int j = threadIdx.x; j < m; j += blockDim.x) ucol[j] = U[(size_t)b * m * m + (size_t)j * m + col];
  float2* my = slots + (size_t)threadIdx.x * me;
  for (int j = 0; j < me; ++j) my[j] = make_float2(0.f, 0.f);
  __syncthreads();
  const SV sv{cg, lo, me, stride};
  const float2* gb = gk + (size_t)b * Sk;
  const float2* pb = psi + (size_t)b * Sp;
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < Sp; t += (uint64_t)gridDim.x * blockDim.x) {
    const float2 ps = pb[t];
    int p[KM];
    slos::unrank_fixed<KM>(sv, (R)t, k - 1, p);
    float gr = 0.f, gi = 0.f;
    slos::children_fixed<KM>(sv, multiset, k, p, [&](R c, int j, int) {
      const float2 gv = gb[c];
      const float2 u = ucol[j];
      gr += u.x * gv.x + u.y * gv.y;   // conj(u) * gv
      gi += u.x * gv.y - u.y * gv.x;
      my[j].x += ps.x * gv.x + ps.y * gv.y;   // conj(psi) * gv
      my[j].y += ps.x * gv.y - ps.y * gv.x;
    });
    if (want_psi_grad) gout[(size_t)b * Sp + t] = make_float2(gr, gi);
  }
  __syncthreads();
  for (int j = threadIdx.x; j < me; j += blockDim.x) {
    double sr = 0, si = 0;
    for (int r = 0; r < kAdjThreads; ++r) {
      sr += slots[(size_t)r * me + j].x;
      si += slots[(size_t)r * me + j].y;
    }
    partial[((size_t)b * gridDim.x + blockIdx.x) * me + j] = make_double2(sr, si);
  }
}

// gU[b][j][col] += sum over blocks of partial[b][block][j]
constexpr int kReduceThreads = 256;
__global__ __launch_bounds__(kReduceThreads) void k_reduce_gu(const double2* __restrict__ partial, int nblk, int me, int m, int col,
                                                  float2* __restrict__ gU, int accumulate) {
  const int64_t b = blockIdx.y;
  const int j = blockIdx.x;
  double sr = 0, si = 0;
  for (int r = threadIdx.x; r < nblk; r += blockDim.x) {
    const double2 v = partial[((size_t)b * nblk + r) * me + j];
    sr += v.x;
    si += v.y;
  }
  for (int o = 32; o > 0; o >>= 1) {
    sr += __shfl_down(sr, o, 64);
    si += __shfl_down(si, o, 64);
  }
  __shared__ double2 wave[kReduceThreads / 64];
  if ((threadIdx.x & 63) == 0) wave[threadIdx.x >> 6] = make_double2(sr, si);
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kReduceThreads / 64; ++w) {
      sr += wave[w].x;
      si += wave[w].y;
    }
    float2* dst = gU + (size_t)b * m * m + (size_t)j * m + col;
    if (accumulate) *dst = make_float2(dst->x + (float)sr, dst->y + (float)si);
    else *dst = make_float2((float)sr, (float)si);
  }
}

// All of dL/dU in one launch: work group (j, b) sums the partials of mode j of every layer in FP64 and
// writes row j of gU[b], the layers' sums added to their columns from the last layer down (columns that
// are no input mode, and modes outside the space, are zero).
struct ReduceArgs {
  uint64_t part[kMaxPhotons];  // layer k's partials [B][nblk][me], at k - 1
  uint32_t nblk[kMaxPhotons];
  int col[kMaxPhotons];
  int layers;
};
// Work groups of 1,024 threads, or of 128 where there are many (1024 / 256 / 128 / 64 threads, us of a whole backward: 20,000
// rows of n = 5, m = 10, dual rail, 1374 / 614 / 538 / 530, 2,000 of n = 2, m = 22 186 / 69 / 54 / 55, 100 of n = 6, m = 12 68 / 64 /
// 63 / 65; one row of n = 8, m = 24 226 / 223 / 229 / 241, n = 5, m = 64 314 / 309 / 326 / 395).
constexpr int kReduceAllThreads = 1024, kReduceManyThreads = 128;
constexpr uint32_t kFew = 512;  // partials of a layer that one wave sums
__global__ __launch_bounds__(kReduceAllThreads) void k_reduce_all(ReduceArgs a, const double2* __restrict__ partial, int me,
                                                                  int m, float2* __restrict__ gU) {
  const int kW = (int)blockDim.x / 64;
  __shared__ double2 wave[kMaxPhotons][kReduceAllThreads / 64];
  __shared__ float2 sum[kMaxPhotons];
  const int64_t b = blockIdx.y;
  const int j = blockIdx.x;
  const int w = threadIdx.x >> 6;
  if (j < me) {
    // a layer of few partials is one wave's, the layers in turn; the others take all waves
    for (int l = 0; l < a.layers; ++l) {
      const uint32_t nblk = a.nblk[l];
      const bool few = nblk <= kFew;
      double sr = 0, si = 0;
      if (!few || l % kW == w) {
        const double2* src = partial + a.part[l] + (size_t)b * nblk * me + j;
        for (uint32_t r = few ? threadIdx.x & 63u : threadIdx.x; r < nblk; r += few ? 64u : blockDim.x) {
          const double2 v = src[(size_t)r * me];
          sr += v.x;
          si += v.y;
        }
        for (int o = 32; o > 0; o >>= 1) {
          sr += __shfl_down(sr, o, 64);
          si += __shfl_down(si, o, 64);
        }
      }
      if ((threadIdx.x & 63) == 0) wave[l][w] = make_double2(sr, si);
    }
    __syncthreads();
    if (threadIdx.x < a.layers) {
      double sr = 0, si = 0;
      for (int i = 0; i < kW; ++i) {
        sr += wave[threadIdx.x][i].x;
        si += wave[threadIdx.x][i].y;
      }
      sum[threadIdx.x] = make_float2((float)sr, (float)si);
    }
    __syncthreads();
  }
  for (int c = threadIdx.x; c < m; c += blockDim.x) {
    float2 v = make_float2(0.f, 0.f);
    if (j < me)
      for (int l = a.layers - 1; l >= 0; --l)
        if (a.col[l] == c) v = make_float2(v.x + sum[l].x, v.y + sum[l].y);
    gU[(size_t)b * m * m + (size_t)j * m + c] = v;
  }
}

// dynamic LDS of the single-plan block kernel for layer K with suffix length suf, or 0 if it
// does not fit the GPU's LDS
size_t block_lds_fit(int K, int me, int suf) {
  const size_t sh = slos::block_dyn_lds(K, me, slos::block_maxd(K - suf));
  return sh + slos::kBlockStaticLds <= lds_limit() ? sh : 0;
}

// suffix length of the single-plan block kernel for layer K: 5-position suffixes where their table
// exists and the prefix is 1..8 positions long (5.4x fewer, larger blocks than with 4 at
// n = 11, m = 32: less per-block set-up and fewer part-filled sweep steps), else 4
int block_suffix(const slos_plan* p, const DevTables& dt, int K) {
  return (dt.tuples5 && K - 5 >= 1 && K - 5 <= 8 && block_lds_fit(K, p->me, 5)) ? 5 : slos::kSuf;
}

// (K - suf)-position prefixes of layer K that have children: those that end at or below the last mode with suf admissible
// positions behind it, as many as tuples of as many modes from the other end
uint64_t full_blocks(const slos_plan* p, int K, int suf) {
  const uint64_t* rest = p->cg.data() + (size_t)suf * (p->me + 1);
  int x = p->me - 1;
  while (x > 0 && rest[p->lo[x]] == 0) --x;
  return std::max<uint64_t>(1, p->cg[(size_t)(K - suf) * (p->me + 1) + (p->me - 1 - x)]);
}

// Whether layer K (S states, B rows) runs on the block or group-order kernel rather than one thread a
// state, where both can. The block kernels share index work between states but wait on their own
// set-up, and a block must be long enough to fill waves; the two give the same bits. Measured (us, block
// or group order against thread):
//   group order: 347k states 21 / 14, 2.0M 28 / 29, 7.9M 56 / 94; compensated 490k 44 / 17; where a group, the
//   states of one (K - 6)-position prefix, is short (many rows of few modes), 20,000 rows of 364 states (6 a group)
//   1904 / 137, 1,000 of 6,435 (179) 81 / 75, 3,000 of 1,716 (245) 54 / 53, 800 of 12,870 (286) 116 / 107, 300 of 92,378 (323) 285 / 301, of
//   24,310 (442) 60 / 82; 2.5M states (291) 46 / 41, 30 rows of them 893 / 1045 (compensated 1673 / 1757), 200 of 352,716 (258) 810 /
//   845 (1622 / 1604); complex128 300 of 92,378 412 / 375, 9 of 646,646 (355) 82 / 76, one of 4.5M (383) 71 / 74;
//   blocks, multiset: 98k states 18.4 / 13.8, 475k 18.9 / 14.9, 2.3M (72,000 a block) 33 / 30, 9.3M (3,400 a
//   block) 74 / 78, 17.4M (102 a block, 12 photons) 368 / 274;
//   blocks, collision-free: 126k 41 / 15, 3.1M (522 a block) 93 / 47, 54.6M (308 a block) 1235 / 970, 7.6M (119,000 a
//   block) 57 / 118.
// Shorter blocks pay where the layer is large: a state costs 6 us / 10^6 in blocks and 13 to 25 by threads, a
// block some 2 us / 1000 besides, and the launch some 40 us of waves that wait on their first blocks. So
// the line of set masks is one of states times states a block that has any (full_blocks), by mask, since their threads
// take longer the fewer modes a photon may enter, by sums, since those in 64 bits gain most (compensated) and least (complex128),
// and lower for rows of a batch, whose blocks hide one another's set-up (not on the smallest launches of dual rail):
//   collision-free, 1.5e10 (5.9M states) 93 / 81, 3.8e10 (10.5M) 121 / 130, 1.6e10 (14.3M) 230 / 188, 4.5e10 (28M) 355 / 364, 1.7e10
//   (30M) 585 / 421, 5.2e10 (64.5M) 867 / 949, 5.6e10 (129M) 1836 / 2348, 2.8e11 (94M) 803 / 1285; compensated 1.7e10 928 / 841;
//   rows 5.6e9 (10 of 735k) 107 / 94, 9.9e9 (9 of 7.7M) 1307 / 1191, 1.5e10 (3 of 13.1M) 653 / 565, 2.1e10 (9 of
//   13.0M) 1885 / 2008, 2.8e10 (3 of 20.0M) 723 / 855, compensated 1.2e10 (9 of 5.3M) 1184 / 1301, 1.4e10 (3 of 21.5M) 2114 / 1956,
//   2.8e10 1276 / 1634, complex128 2.1e10 (200 of 500k) 1558 / 1454, 2.8e10 1114 / 1114, 4.8e10 (9 of 6.9M) 900 / 988;
//   dual rail, 8e9 (3.3M) 55 / 47, 6.3e9 (25M) 531 / 479, 1.1e10 436 / 439, 1.5e10 (70M) 1387 / 2474, 2.6e10 (76M) 1116 / 1507, 5.5e10
//   (11M) 107 / 138, compensated 1.3e9 (7.5M) 243 / 229, 2.7e9 (8.9M) 249 / 252, 4.5e9 193 / 212, complex128 1.6e10 (20M) 421 / 383,
//   2e10 (12M) 192 / 217; rows 1.4e9 (200 of 68k) 219 / 197, 2.1e9 (20 of 745k) 248 / 249, 4.5e9 (200 of 113k) 271 / 323, 3.7e9 (3M states in
//   all) 39 / 34, 1.2e10 (4M) 45 / 43, 1.3e10 (7M) 62 / 65, compensated 4.3e8 (5M) 157 / 138, 6.6e8 (10M) 296 / 317, 1.1e9 (3M) 83 / 84, 3.3e9
//   (23M) 475 / 611, complex128 2.1e9 326 / 320, 4.5e9 362 / 382;
//   sparse_1in4, 1.1e9 (1.0M) 21 / 22, 4.3e9 (4.2M) 62 / 78, 1.4e10 (2.9M) 39 / 41, 1.7e10 (16.8M) 178 / 402, 2.2e11 (69M) 534 / 1119; rows
//   2.4e9 (9 of 262k) 33 / 37, compensated 50 / 59; complex128 by states alone, 2.6M 52 / 45, 5.4M 76 / 67, 3 rows of 2.9M 134 / 119, 9
//   of 1.0M 188 / 199, 10.8M 145 / 152, 16.8M 342 / 460;
// and 2^33 for the multiset layers that have no group order: 12 photons, 1.8e9 (17.4M, 101 a block) 364 / 268, 7.7e9 (52M, 149)
//   768 / 790 (compensated 1607 / 1334, complex128 948 / 917), 3e10 (141M, 214) 1482 / 2317.
// The thread kernel's exact forms are those of at most 12 photons and 2^32 states. The line holds for
// compensated sums (8 photons, 1.1M states 27 / 24, 2.2M 33 / 45, 9 photons, 3.1M 46 / 63; collision-free 3.1M (209 a
// block) 115 / 72, 10.7M 106 / 153) and for complex128 (f64: 1.1M 26 / 18, 2.2M 28 / 32, 3.1M 39 / 45; 3.1M (209 a
// block) 101 / 54, 10.7M 80 / 117). At 13 photons, the most the complex128 block kernel takes, its blocks of tens of
// states lose to the thread kernel's 16-photon form up to some ten million: 203k states 96 / 15, 5.2M 229 / 172,
// 10.4M 350 / 336 (raw layers 424 / 296), 37M 959 / 1220 (1113 / 1096), 120M 2209 / 3978; and in rows of short blocks at
// any size: 2,000 of (13, 7), 9 states a block, 4146 / 1721, 20 of (13, 12), 33, 1889 / 1581, 4 of (13, 14), 51, 1149 / 1338.
bool use_blocks(const slos_plan* p, int K, int suf, uint64_t S, int64_t B, bool comp, bool f64) {
  const double states = (double)S * (double)B;
  if (S >= (1ull << 32) || (K > 12 && !f64)) return true;
  if (K > 12 && p->multiset) return S * (uint64_t)B >= (1ull << 25) && S >= 48 * full_blocks(p, K, suf);
  if (K > 12 && S * (uint64_t)B < (1ull << 25)) return false;
  if (S * (uint64_t)B < (1ull << 21)) return false;
  if (suf == 5 && !p->items[K].empty())
    return S >= (f64 ? 370 : S >= (1ull << 20) && states >= (double)(1ull << 23) ? 280 : 320) * p->size(K - 6);
  const double per = (double)S / (double)full_blocks(p, K, suf);
  if (p->multiset) return per >= 256.0 || states * per >= (double)(1ull << 33);
  const bool rows = B > 1, large = states >= (double)(1ull << 23);
  if (p->shift == 0) return states * per >= (f64 ? 4e10 : comp ? (rows ? 1.2e10 : 2.2e10) : rows ? 1.7e10 : 3e10);
  if (p->shift == 1) return states * per >= (comp ? (rows && large ? 6e8 : 2.7e9) : rows ? (large ? 2.5e9 : 1.2e10) : f64 ? 2e10 : 1.4e10);
  return f64 ? states >= 9e6 : states * per >= 2e9;
}

// The grid of `wgs` work groups a row (see slos::batch_item): 1-D over all rows from 8 rows on, where
// there is one for every XCD and the grid's thread count stays below 2^32, else a row per grid y. A row's
// parent layer (par_bytes) is of use to the one XCD it is read into while a fair part of it stays in the L2;
// rows far larger only crowd one another out of the 256 MB behind it. Last layer, us, 1-D against 2-D: 5 MiB of
// parents (32 rows of (8, 20)) 344 / 355, 12 MiB (9 of (9, 26), collision-free) 330 / 341, 24 MiB (9 of (9, 28)) 571 / 569, 29
// MiB (sparse_1in4's layer 7 of 12) 604 / 569, 58 MiB (9 of (6, 60)) 3663 / 2719, 109 MiB (9 of (10, 30)) 2557 / 2327; complex128
// 10 MiB 661 / 704, 22 MiB (dual rail's layer 8 of 16) 410 / 443, 25 MiB (9 of (7, 30)) 675 / 665, 127 MiB 3283 / 3179.
dim3 batch_grid(uint64_t wgs, int64_t B, uint64_t par_bytes, slos::BlockLayer* L) {
  L->row_wgs = (uint32_t)wgs;
  const bool flat = B >= 8 && par_bytes <= (24ull << 20) && wgs * (uint64_t)B < (1ull << 32) / slos::kBlockThreads;
  L->rows = flat ? (uint32_t)B : 1u;
  return flat ? dim3((unsigned)(wgs * (uint64_t)B)) : dim3((unsigned)wgs, (unsigned)B);
}

int launch_block(const slos_plan* p, const DevTables& dt, const slos::LayerArgs& a, int kind, bool comp, hipStream_t st) {
  slos::BlockLayer L;
  L.K = a.K; L.m = a.m; L.col = a.col; L.U = a.U; L.us = a.us; L.S_par = a.S_par; L.S = a.S; L.gp = a.gp;
  L.par_lo = a.par_lo; L.out_lo = a.out_lo;
  const int suf = block_suffix(p, dt, a.K);
  L.S_pre = p->size(a.K - suf);
  L.scale = a.scale; L.flags = a.flags;
  // children per wave: enough waves to fill the chip several times, but long ranges at scale
  uint64_t pw = (a.S / 16384 + 63) & ~63ull;
  // (2048 at most for the complex64 intermediate layers, 4096 for the read-out layer: measured best
  // at n = 11, m = 32)
  L.per_wave = std::min<uint64_t>(std::max<uint64_t>(pw, 256), kind == 0 ? 2048 : 4096);
  // XCD chunks of about 2^20 children (64 work groups at 4096 children per wave)
  L.xcd_chunk = (uint32_t)std::max<uint64_t>(1, (1ull << 20) / ((uint64_t)slos::kWaves * L.per_wave));
  const uint64_t waves = (a.S + L.per_wave - 1) / L.per_wave;
  const uint64_t wgs = (waves + slos::kWaves - 1) / slos::kWaves;
  if (wgs > 0x7fffffffull) return fail(SLOS_ERANGE, "layer too large for one launch");
  if (a.B > 65535) return fail(SLOS_ERANGE, "batch > 65535");
  const uint64_t par_bytes = a.S_par * sizeof(float2) * (a.par_lo ? 2 : 1);
  // layers in group order where their work items exist (plain or compensated sums; probabilities or
  // complex64)
  if (suf == 5 && kind != 2 && dt.items[a.K]) {
    const auto [gitems, gn] = dt.group_items(a.K, a.S * (uint64_t)a.B);
    const size_t shg = slos::group_dyn_lds(a.K, p->me);
    const uint64_t gwgs = ((uint64_t)gn + slos::kWaves - 1) / slos::kWaves;
    if (shg + slos::kBlockStaticLds <= lds_limit() && gwgs <= 0x7fffffffull) {
      L.xcd_chunk = (uint32_t)std::max<uint64_t>(1, (1ull << 20) / ((uint64_t)slos::kWaves * slos::kGroupItemChildren));
      const slos::BlockGrid bg{batch_grid(gwgs, a.B, par_bytes, &L), shg, st, dt.cg, dt.lo, dt.tuples5, p->me, p->multiset};
      slos::launch_layer_group(a.K - suf, kind, comp, bg, a.par, a.out, L, gitems, gn);
      HIP_TRY(hipGetLastError());
      return SLOS_OK;
    }
  }
  const size_t sh = block_lds_fit(a.K, p->me, suf);
  if (!sh) return fail(SLOS_ERANGE, "block kernel LDS exceeds the GPU's LDS");
  const slos::BlockGrid bg{batch_grid(wgs, a.B, par_bytes, &L), sh, st, dt.cg, dt.lo,
                           suf == 5 ? static_cast<const void*>(dt.tuples5) : dt.tuples, p->me, p->multiset};
  if (kind == 0) slos::launch_layer_block<0>(comp, a.K - suf, suf, bg, a.par, a.out, L);
  else if (kind == 1) slos::launch_layer_block<1>(comp, a.K - suf, suf, bg, a.par, a.out, L);
  else if (kind == 4) slos::launch_layer_block<4>(false, a.K - suf, suf, bg, a.par, a.out, L);
  else slos::launch_layer_block<2>(comp, a.K - suf, suf, bg, a.par, a.out, L);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

// calls f with the smallest photon bound KM (8, 16 or 32) of the thread-per-state kernels that
// holds `photons` (their per-state arrays are sized by it and stay in registers)
template <class F>
void with_km(int photons, F&& f) {
  if (photons <= 8) f(std::integral_constant<int, 8>{});
  else if (photons <= 16) f(std::integral_constant<int, 16>{});
  else f(std::integral_constant<int, 32>{});
}

// par_hilo / out_hilo (compensated sums only): the parent layer / the complex64 output layer is a
// hi/lo pair [2][B][S], the low-order parts after the high ones
int launch_layer(const slos_plan* p, const DevTables& dt, int K, int col, const float2* U, slos::MatrixStride us, int64_t B,
                 const float2* par, uint64_t S_par, void* out, uint64_t S, int kind, float scale,
                 unsigned flags, hipStream_t st, bool par_hilo = false, bool out_hilo = false,
                 const float* gp = nullptr) {
  slos::LayerArgs a;
  a.gp = gp;
  a.cg = dt.cg; a.lo = dt.lo; a.me = p->me; a.multiset = p->multiset; a.K = K; a.m = p->m; a.col = col;
  a.U = U; a.us = us; a.words = dt.tuples5; a.par = par; a.S_par = S_par; a.out = out; a.S = S; a.B = B;
  a.scale = scale; a.flags = flags;
  const bool comp = flags & SLOS_FLAG_COMPENSATED;
  a.par_lo = (comp && par_hilo) ? B * (int64_t)S_par : 0;
  a.out_lo = (comp && out_hilo && kind == 0) ? B * (int64_t)S : 0;
  if (!(flags & SLOS_FLAG_SIMPLE) && dt.tuples && K > slos::kSuf && K - slos::kSuf <= 16 &&
      block_lds_fit(K, p->me, slos::kSuf) && (flags & SLOS_FLAG_BLOCK || use_blocks(p, K, block_suffix(p, dt, K), S, B, comp, false)))
    return launch_block(p, dt, a, kind, comp, st);
  const size_t sh = (((size_t)(K + 1) * (p->me + 1) * 8 + p->me * 4 + 15) & ~(size_t)15) + (size_t)p->m * 8;
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  const uint64_t blocks = std::min<uint64_t>((S + 255) / 256, 1u << 20);
  dim3 grid((unsigned)std::max<uint64_t>(blocks, 1), (unsigned)std::min<int64_t>(B, 65535));
  slos::launch_layer_simple(kind, comp, grid, sh, st, a);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

// one complex128 layer on the block or group-order kernel; -1 where they do not apply (layers of
// fewer than 5 photons, prefixes of more than 8 positions, spaces without tuple words, and by use_blocks)
int launch_block_f64(const slos_plan* p, const DevTables& dt, int K, int col, const void* U, slos::MatrixStride us, int64_t B, const void* par,
                     uint64_t S_par, void* out, uint64_t S, int kind, double scale, unsigned flags, hipStream_t st) {
  if (!dt.tuples || K <= slos::kSuf || B > 65535) return -1;
  const int suf = dt.tuples5 && K > 5 ? 5 : slos::kSuf;
  const int d = K - suf;
  if (d > 8 || !(flags & SLOS_FLAG_BLOCK || use_blocks(p, K, suf, S, B, false, true))) return -1;
  slos::BlockLayerF64 L{};
  L.l.K = K; L.l.m = p->m; L.l.col = col; L.l.S_par = S_par; L.l.S = S; L.l.S_pre = p->size(d);
  L.l.flags = flags;
  L.U = static_cast<const double2*>(U);
  L.l.us = us;
  L.scale = scale;
  if (suf == 5 && kind <= 1 && dt.items[K]) {
    const size_t sh = slos::group_dyn_lds64(K, p->me);
    const auto [items, n_items] = dt.group_items(K, S * (uint64_t)B);
    const uint64_t wgs = ((uint64_t)n_items + slos::kWaves - 1) / slos::kWaves;
    if (sh + slos::kBlockStaticLds64 <= lds_limit() && wgs <= 0x7fffffffull) {
      L.l.xcd_chunk = (uint32_t)std::max<uint64_t>(1, (1ull << 20) / ((uint64_t)slos::kWaves * slos::kGroupItemChildren));
      const slos::BlockGrid bg{batch_grid(wgs, B, S_par * sizeof(double2), &L.l), sh, st, dt.cg, dt.lo, dt.tuples5, p->me, p->multiset};
      slos::launch_layer_group_f64(d, kind, bg, static_cast<const double2*>(par), out, L, items, n_items);
      HIP_TRY(hipGetLastError());
      return SLOS_OK;
    }
  }
  const size_t sh = slos::block_dyn_lds(K, p->me, slos::block_maxd_f64(d));
  if (sh + slos::kBlockStaticLds64 > lds_limit()) return -1;
  // children per wave as the complex64 block kernel
  const uint64_t pw = (S / 16384 + 63) & ~63ull;
  L.l.per_wave = std::min<uint64_t>(std::max<uint64_t>(pw, 256), kind == 0 ? 2048 : 4096);
  L.l.xcd_chunk = (uint32_t)std::max<uint64_t>(1, (1ull << 20) / ((uint64_t)slos::kWaves * L.l.per_wave));
  const uint64_t wgs = ((S + L.l.per_wave - 1) / L.l.per_wave + slos::kWaves - 1) / slos::kWaves;
  if (wgs > 0x7fffffffull) return -1;
  const slos::BlockGrid bg{batch_grid(wgs, B, S_par * sizeof(double2), &L.l), sh, st, dt.cg, dt.lo,
                           suf == 5 ? static_cast<const void*>(dt.tuples5) : dt.tuples, p->me, p->multiset};
  slos::launch_layer_block_f64(kind, d, suf, bg, static_cast<const double2*>(par), out, L);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

// one complex128 layer, on the block or group-order kernel where launch_block_f64 takes it, else thread per
// state: kind 0 raw complex128, 1 float64 probabilities, 2 scaled complex128 amplitudes (SLOS_FLAG_IMMEDIATE:
// times sqrt(prod t!))
int launch_layer_f64(const slos_plan* p, const DevTables& dt, int K, int col, const void* U, slos::MatrixStride us, int64_t B, const void* par,
                     uint64_t S_par, void* out, uint64_t S, int kind, double scale, unsigned flags, hipStream_t st) {
  if (!(flags & SLOS_FLAG_SIMPLE)) {
    const int rc = launch_block_f64(p, dt, K, col, U, us, B, par, S_par, out, S, kind, scale, flags, st);
    if (rc >= 0) return rc;
  }
  slos::LayerArgsF64 a;
  a.cg = dt.cg; a.lo = dt.lo; a.words = dt.tuples5; a.me = p->me; a.multiset = p->multiset; a.K = K; a.m = p->m; a.col = col;
  a.U = static_cast<const double2*>(U); a.us = us; a.par = static_cast<const double2*>(par); a.S_par = S_par;
  a.out = out; a.S = S; a.B = B; a.scale = scale;
  a.immediate = (flags & SLOS_FLAG_IMMEDIATE) ? 1u : 0u;
  const size_t sh = slos::space_lds_f64(K, p->me) + (size_t)p->m * 16;
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  const uint64_t blocks = std::min<uint64_t>((S + 255) / 256, 1u << 20);
  dim3 grid((unsigned)std::max<uint64_t>(blocks, 1), (unsigned)std::min<int64_t>(B, 65535));
  slos::launch_layer_f64_simple(kind, grid, sh, st, a);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

// The layers 1..kf that one launch of k_front takes (0: none): the largest kf <= layer for which the
// layers below kf fit LDS with at most kFrontStates states, which computes at most 2^21 states again (all
// work groups together; with more the chip is full and a launch a layer costs less), and whose work
// groups, of every row, are at most 512: two a CU, the chip once. Each takes 10 us or more however few
// states its row has, so that with many rows a launch a layer is the shorter way, us, so / a launch a layer:
// n = 4, m = 8, 512 work groups 17 / 27, 1024 31 / 27, 2048 59 / 29; n = 5, m = 10, 512 19 / 30, 1024 34 / 33,
// 2048 66 / 49; n = 6, m = 6, 1024 32 / 30; n = 3, m = 6, 60000 1117 / 153; n = 2, m = 4, 60000 818 / 84. From
// 128 modes on a thread's search for its positions, which k_front shortens, outweighs that: n = 2, m = 200,
// 5120 113 / 145; n = 1, m = 300, 2048 28 / 45; n = 2, m = 1500, 1100 52 / 704; but n = 2, m = 100, 5120 107 / 89.
int front_layers(const slos_plan* p, int64_t B, int layer, size_t elem, bool comp, size_t* lds, uint32_t* buf) {
  int kf = 0;
  if (B > 65535) return 0;
  uint64_t below = 1, most = 1;  // states of the layers 0..k-1, the largest of them
  for (int k = 1; k <= std::min(layer, slos::kFrontMax); ++k) {
    const uint64_t S = p->size(k);
    if (S >= (1ull << 31) || most > slos::kFrontStates) break;
    const uint64_t wgs = (S + slos::kFrontThreads - 1) / slos::kFrontThreads;
    if (wgs * below * (uint64_t)B > (1ull << 21)) break;
    const size_t need = slos::front_lds(k, p->me, p->m, elem, most, comp);
    if (need > lds_limit()) break;
    if (p->me >= 128 || wgs * (uint64_t)B <= 512u) {
      kf = k;
      *lds = need;
      *buf = (uint32_t)most;
    }
    below += S;
    most = std::max(most, S);
  }
  return kf;
}

// layers 1..kf (front_layers) in one launch; kind: of layer kf
int run_front(const slos_plan* p, const DevTables& dt, int kf, const int* cols, const void* U, slos::MatrixStride us, int64_t B, void* out,
              int kind, double scale, unsigned flags, size_t lds, uint32_t buf, bool hilo_out, hipStream_t st,
              void* const* below = nullptr) {
  slos::FrontArgs a{};
  if (below)
    for (int k = 0; k < kf; ++k) a.below[k] = below[k];
  a.cg = dt.cg; a.lo = dt.lo; a.tuples = dt.tuples; a.tuples5 = dt.tuples5;
  a.me = p->me; a.multiset = p->multiset; a.m = p->m; a.kf = kf; a.kind = kind; a.U = U; a.us = us;
  for (int k = 0; k < kf; ++k) a.cols[k] = cols[k];
  for (int k = 0; k <= kf; ++k) a.S[k] = (uint32_t)p->size(k);
  a.buf = buf; a.out = out; a.scale = scale;
  a.immediate = (flags & SLOS_FLAG_IMMEDIATE) ? 1u : 0u;
  a.out_lo = hilo_out ? B * (int64_t)p->size(kf) : 0;
  const uint64_t wgs = (p->size(kf) + slos::kFrontThreads - 1) / slos::kFrontThreads;
  const RoctxRange range("slos first layers");
  slos::launch_front((flags & SLOS_FLAG_F64) != 0, (flags & SLOS_FLAG_COMPENSATED) != 0,
                     dim3((unsigned)wgs, (unsigned)B), lds, st, a);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

bool mul_overflow(uint64_t a, uint64_t b, uint64_t* r) { return __builtin_mul_overflow(a, b, r); }

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct WsLayout {
  size_t ones = 0, odd = 0, even = 0, total = 0;
};

// hilo: the intermediate layers are hi/lo pairs [2][B][S] (compensated sums carry their rounding
// errors from layer to layer), twice the bytes; f64: complex128 layers (16 bytes a state)
int forward_layout(const slos_plan* p, int64_t B, int layer, WsLayout* w, bool hilo = false, bool f64 = false) {
  uint64_t maxodd = 0, maxeven = 0;
  for (int k = 1; k < layer; ++k) (k & 1 ? maxodd : maxeven) = std::max(k & 1 ? maxodd : maxeven, p->size(k));
  uint64_t a = 0, b = 0;
  const uint64_t elem = f64 ? 16 : 8;
  const uint64_t per = (uint64_t)B * elem * (hilo ? 2 : 1);
  if (mul_overflow(maxodd, per, &a) || mul_overflow(maxeven, per, &b))
    return fail(SLOS_ERANGE, "workspace size overflows");
  w->ones = 0;
  w->odd = align256((size_t)B * elem);
  w->even = w->odd + align256(a);
  w->total = w->even + align256(b);
  return SLOS_OK;
}

// ------------------------------------------------------------------------------------------
// strong-then-sample: two-level inverse CDF over float32 probabilities in FP64, every addition in
// a fixed order (chunk = 64 entries summed in index order, block = 64 chunks summed in chunk
// order, block prefix = sequential inside segments of kSampleSeg blocks plus the sequential
// prefix of the segment totals), then the per-shot search. Replaces the float64 cumsum +
// searchsorted of imperfections.py:221-237 (above 2^24 categories) without an [S] float64 copy.
// ------------------------------------------------------------------------------------------
constexpr int kSampleChunk = 64;
constexpr int kSampleBlock = kSampleChunk * 64;   // 4096 entries
constexpr int kSampleSeg = 1024;                   // blocks per prefix segment

// One wave per block of 4096 entries; lane c loads its own chunk c (64 consecutive entries, 16 bytes
// at a time: the two cache lines of a chunk are read by one lane in consecutive loads) and sums it
// in index order (FP64, from 0.0; entries past S count as 0), then every lane sums the 64 chunk
// sums in chunk order. No LDS, so many waves stay resident to cover the stream.
constexpr int kSumWaves = 4;
__global__ __launch_bounds__(64 * kSumWaves) void k_sample_block_sums(const float* __restrict__ p, uint64_t S, uint64_t nb,
                                                                      double* __restrict__ bsum,
                                                                      double* __restrict__ csum) {
  const int lane = threadIdx.x & 63;
  const uint64_t b = (uint64_t)blockIdx.x * kSumWaves + (uint64_t)(threadIdx.x >> 6);
  if (b >= nb) return;
  const uint64_t i0 = b * kSampleBlock + (uint64_t)lane * kSampleChunk;
  double cs = 0.0;
  if (i0 + kSampleChunk <= S) {
    float4 v[kSampleChunk / 4];
#pragma unroll
    for (int j = 0; j < kSampleChunk / 4; ++j) __builtin_memcpy(&v[j], p + i0 + 4 * j, 16);
#pragma unroll
    for (int j = 0; j < kSampleChunk / 4; ++j) {
      cs += (double)v[j].x;
      cs += (double)v[j].y;
      cs += (double)v[j].z;
      cs += (double)v[j].w;
    }
  } else {
    for (int k = 0; k < kSampleChunk; ++k) cs += (double)(i0 + k < S ? p[i0 + k] : 0.f);
  }
  csum[b * 64 + (uint64_t)lane] = cs;
  double tot = 0.0;
  for (int c = 0; c < 64; ++c) tot += __shfl(cs, c, 64);
  if (lane == 0) bsum[b] = tot;
}

// Block prefix over segments of kSampleSeg blocks: one work group per segment stages its block sums
// in LDS (coalesced), one thread takes their inclusive prefix in order (from 0.0) and the group
// writes it back (coalesced); segtot[seg] = the segment's total.
__global__ __launch_bounds__(256) void k_sample_seg_prefix(const double* __restrict__ bsum, uint64_t nb,
                                                           double* __restrict__ cdf, double* __restrict__ segtot) {
  __shared__ double seg[kSampleSeg];
  const uint64_t a = (uint64_t)blockIdx.x * kSampleSeg;
  const int len = (int)(nb - a < (uint64_t)kSampleSeg ? nb - a : (uint64_t)kSampleSeg);
  for (int i = threadIdx.x; i < len; i += blockDim.x) seg[i] = bsum[a + i];
  __syncthreads();
  if (threadIdx.x == 0) {
    double acc = 0.0;
    for (int i = 0; i < len; ++i) {
      acc += seg[i];
      seg[i] = acc;
    }
    segtot[blockIdx.x] = acc;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < len; i += blockDim.x) cdf[a + i] = seg[i];
}

// exclusive prefix of the segment totals, in order (one thread; at most 1024 segments)
__global__ __launch_bounds__(64) void k_sample_seg_offsets(double* __restrict__ segtot, int nseg) {
  if (threadIdx.x != 0) return;
  double run = 0.0;
  for (int i = 0; i < nseg; ++i) {
    const double v = segtot[i];
    segtot[i] = run;
    run += v;
  }
}

// cdf = segment offset + the segment's own prefix
__global__ __launch_bounds__(256) void k_sample_add_offsets(double* __restrict__ cdf, uint64_t nb,
                                                            const double* __restrict__ segoff) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nb; i += (uint64_t)gridDim.x * blockDim.x)
    cdf[i] = segoff[i / kSampleSeg] + cdf[i];
}

// one thread per shot: u = uniform * total; block = first cdf >= u (binary search), then the chunk
// and the entry by in-order prefix sums of the block pass's chunk sums and of the chunk's entries
__global__ __launch_bounds__(256) void k_sample_search(const float* __restrict__ p, uint64_t S, uint64_t nb,
                                                       const double* __restrict__ cdf, const double* __restrict__ csum,
                                                       const double* __restrict__ uni, int64_t shots,
                                                       uint64_t* __restrict__ idx) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= shots) return;
  const double total = cdf[nb - 1];
  const double u = uni[s] * total;
  uint64_t lo = 0, hi = nb - 1;  // first b with cdf[b] >= u, else nb - 1
  while (lo < hi) {
    const uint64_t mid = lo + (hi - lo) / 2;
    if (cdf[mid] >= u) hi = mid;
    else lo = mid + 1;
  }
  const uint64_t b = lo;
  double r = u - (b > 0 ? cdf[b - 1] : 0.0);
  const double* cb = csum + b * 64;
  int c = 63;
  double pre = 0.0;
  for (int q = 0; q < 64; ++q) {
    const double v = cb[q];
    if (pre + v >= r) {
      c = q;
      break;
    }
    pre += v;
  }
  r -= pre;
  const uint64_t first = b * kSampleBlock + (uint64_t)c * kSampleChunk;
  int k = 63;
  double acc = 0.0;
  for (int q = 0; q < kSampleChunk; ++q) {
    acc += (double)(first + q < S ? p[first + q] : 0.f);
    if (acc >= r) {
      k = q;
      break;
    }
  }
  uint64_t out = first + (uint64_t)k;
  if (out >= S) out = S - 1;
  idx[s] = out;
}

// lex index -> occupation row (int32 [m]) of layer k, one thread per index
// (an index >= S_k gives a row of -1)
__global__ __launch_bounds__(256) void k_unrank_occ(const uint64_t* cg_g, const int* lo_g, int me, int k, int m,
                                                    const uint64_t* __restrict__ idx, int64_t count,
                                                    int32_t* __restrict__ occ) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int stride = me + 1;
  const int ncg = (k + 1) * stride;
  uint64_t* cg = reinterpret_cast<uint64_t*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = cg_g[i];
  for (int i = threadIdx.x; i < me; i += blockDim.x) lo[i] = lo_g[i];
  __syncthreads();
  const slos::SpaceView sv{cg, lo, me, stride};
  for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < count; s += (int64_t)gridDim.x * blockDim.x) {
    int32_t* row = occ + (size_t)s * m;
    const uint64_t g = idx[s];
    if (g >= cg[(size_t)k * stride]) {
      for (int j = 0; j < m; ++j) row[j] = -1;
      continue;
    }
    int pos[kMaxPhotons];
    sv.unrank(g, k, pos);
    for (int j = 0; j < m; ++j) row[j] = 0;
    for (int i = 0; i < k; ++i) row[pos[i]] += 1;
  }
}

// ------------------------------------------------------------------------------------------
// uneven batches: a group of plans, one launch per photon layer (see layer_block.hpp)
// ------------------------------------------------------------------------------------------

// thread-per-state form of a group layer: item = (plan, instance, 256 * spt consecutive states)
// (K <= KM)
template <bool COMP, int KM>
__global__ __launch_bounds__(256) void k_layer_simple_group(slos::GroupLaunch gl) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int K = gl.K;
  const uint64_t* cur = nullptr;
  slos::for_each_item(gl.total, [&](uint32_t item) {
    const slos::GroupItem& it = gl.it[slos::group_index(gl, item)];
    const uint32_t rel = item - it.wg_begin;
    const uint32_t b = rel / it.wgs_per_inst, w = rel - b * it.wgs_per_inst;
    const int stride = it.me + 1;
    const int ncg = (K + 1) * stride;
    uint64_t* cg = reinterpret_cast<uint64_t*>(smem);
    int* lo = reinterpret_cast<int*>(cg + ncg);
    float2* ucol = reinterpret_cast<float2*>(smem + ((ncg * 8 + it.me * 4 + 15) & ~15));
    __syncthreads();  // the previous item is done with LDS
    if (it.cg != cur) {
      for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = it.cg[i];
      for (int i = threadIdx.x; i < it.me; i += blockDim.x) lo[i] = it.lo[i];
      cur = it.cg;
    }
    for (int j = threadIdx.x; j < it.m; j += blockDim.x)
      ucol[j] = it.U[(size_t)b * it.m * it.m + (size_t)j * it.m + it.col];
    __syncthreads();
    const slos::SpaceView sv{cg, lo, it.me, stride};
    const float2* pb = it.par + (size_t)b * it.S_par;
    const uint32_t spt = (uint32_t)it.per_wave;
    const uint64_t g0 = (uint64_t)w * 256u * spt + threadIdx.x;
    for (uint32_t i = 0; i < spt; ++i) {
      const uint64_t g = g0 + 256ull * i;
      if (g >= it.S) break;
      int pos[KM];
      slos::unrank_fixed<KM>(sv, g, K, pos);
      slos::BlockAcc<COMP> acc;
      slos::parents_fixed<KM>(sv, it.multiset, K, pos,
                              [&](uint64_t pr, int mode, int) { slos::bk_cmac(acc, ucol[mode], pb[pr]); });
      if constexpr (COMP) {
        if (it.par_lo)  // the parents' low-order parts
          slos::parents_fixed<KM>(sv, it.multiset, K, pos,
                                  [&](uint64_t pr, int mode, int) { slos::bk_lo_mac(acc, ucol[mode], pb[it.par_lo + pr]); });
      }
      const float2 sum = acc.value();
      float re = sum.x, im = sum.y;
      if (it.kind == 1) {
        const float f = slos::run_factorial_fixed<KM>(pos, K, it.multiset);
        re *= it.scale;
        im *= it.scale;
        reinterpret_cast<float*>(it.out)[(size_t)b * it.S + g] = slos::prob_readout(re, im, f);
      } else {
        reinterpret_cast<float2*>(it.out)[(size_t)b * it.S + g] = make_float2(re, im);
        if constexpr (COMP) {
          if (it.out_lo) reinterpret_cast<float2*>(it.out)[it.out_lo + (size_t)b * it.S + g] = acc.rest(sum);
        }
      }
    }
  });
}

size_t simple_lds_bytes(int K, int me, int m) {
  return (((size_t)(K + 1) * (me + 1) * 8 + (size_t)me * 4 + 15) & ~(size_t)15) + (size_t)m * 8;
}

}  // namespace

// a group of plans run together (uneven batches)
struct slos_group {
  struct Cfg {
    int block = -1;         // 1 block kernel, 0 thread-per-state, 2 one single-plan launch per plan, -1 default
    uint64_t per_wave = 0;  // children per wave (block) / states per thread (simple); 0: default
    uint32_t grid = 0;      // work groups of the persistent launch; 0: one per item
  };
  std::vector<const slos_plan*> plans;
  int nmax = 0;
  std::vector<Cfg> cfg;     // [nmax + 1]
  hipStream_t cap = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int cap_device = -1;
};

namespace {

struct GroupArgs {
  std::vector<const float2*> U;
  std::vector<int64_t> B;
  std::vector<float*> out;
  std::vector<float> scale;
  unsigned flags = 0;
  unsigned char* ws = nullptr;
  size_t ws_bytes = 0;
};

struct GroupWs {
  std::vector<size_t> ones, buf0, buf1;
  size_t total = 0;
};

// hilo (compensated sums): every plan's intermediate layers are hi/lo pairs [2][B][S]
int group_layout(const slos_group* G, const int64_t* B, GroupWs* w, bool hilo) {
  size_t off = 0;
  for (size_t g = 0; g < G->plans.size(); ++g) {
    const slos_plan* p = G->plans[g];
    if (B[g] < 1 || B[g] > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
    uint64_t maxS = 0, bytes = 0;
    for (int k = 1; k < p->n; ++k) maxS = std::max(maxS, p->size(k));
    if (mul_overflow(maxS, (uint64_t)B[g] * 8 * (hilo ? 2 : 1), &bytes))
      return fail(SLOS_ERANGE, "workspace size overflows");
    w->ones.push_back(off);
    off += align256((size_t)B[g] * 8);
    w->buf0.push_back(off);
    off += align256(bytes);
    w->buf1.push_back(off);
    off += align256(bytes);
  }
  w->total = off;
  return SLOS_OK;
}

int group_args(const slos_group* G, const void* const* U, const int64_t* B, float* const* out, const double* scale,
               unsigned flags, void* ws, size_t ws_bytes, GroupArgs* a, GroupWs* w) {
  if (!G || !U || !B || !out || !scale) return fail(SLOS_EINVAL, "NULL argument");
  int rc = group_layout(G, B, w, (flags & SLOS_FLAG_COMPENSATED) != 0);
  if (rc) return rc;
  if (!ws || ws_bytes < w->total)
    return fail(SLOS_ENOMEM, "workspace too small: need " + std::to_string(w->total) + " bytes");
  for (size_t g = 0; g < G->plans.size(); ++g) {
    if (!U[g] || !out[g]) return fail(SLOS_EINVAL, "NULL unitary or output");
    a->U.push_back(static_cast<const float2*>(U[g]));
    a->B.push_back(B[g]);
    a->out.push_back(out[g]);
    a->scale.push_back((float)scale[g]);
  }
  a->flags = flags;
  a->ws = static_cast<unsigned char*>(ws);
  a->ws_bytes = ws_bytes;
  return SLOS_OK;
}

bool group_can_block(const slos_group* G, const std::vector<DevTables>& dts, int K, unsigned flags) {
  if ((flags & SLOS_FLAG_SIMPLE) || K <= slos::kSuf || K - slos::kSuf > 16) return false;
  size_t off = 0;
  for (size_t g = 0; g < G->plans.size(); ++g)
    if (G->plans[g]->n >= K) {
      if (!dts[g].tuples) return false;
      off = std::max(off, slos::block_table_offset(K, G->plans[g]->me));
    }
  const size_t sh = off + (size_t)slos::kWaves * slos::kBlockBatch * slos::block_words(slos::block_maxd(K - slos::kSuf)) * 4;
  return sh + slos::kBlockStaticLds <= lds_limit();
}

// layer K of every plan with n >= K as one launch per plan, through the single-plan path (the
// 5-position-suffix and group-order kernels where they apply): the same values as the group kernel
int group_layer_per_plan(const slos_group* G, int K, const GroupArgs& a, const GroupWs& w,
                         const std::vector<DevTables>& dts, hipStream_t st) {
  const bool hilo = (a.flags & SLOS_FLAG_COMPENSATED) != 0;
  for (size_t g = 0; g < G->plans.size(); ++g) {
    const slos_plan* p = G->plans[g];
    if (p->n < K) continue;
    float2* bufs[2] = {reinterpret_cast<float2*>(a.ws + w.buf0[g]), reinterpret_cast<float2*>(a.ws + w.buf1[g])};
    const float2* par = K == 1 ? reinterpret_cast<const float2*>(a.ws + w.ones[g]) : bufs[(K - 1) & 1];
    const bool last = K == p->n;
    void* out = last ? static_cast<void*>(a.out[g]) : static_cast<void*>(bufs[K & 1]);
    const int rc = launch_layer(p, dts[g], K, p->modes[K - 1], a.U[g], slos::packed_stride(p->m), a.B[g], par, p->size(K - 1), out, p->size(K),
                                last ? 1 : 0, last ? a.scale[g] : 1.f, a.flags & ~SLOS_FLAG_HILO, st, hilo && K >= 2,
                                hilo && !last);
    if (rc) return rc;
  }
  return SLOS_OK;
}

// layer K of every plan with n >= K, in one launch (or one per plan: Cfg.block 2, and by default
// where a single plan reaches layer K)
int group_layer(const slos_group* G, int K, const GroupArgs& a, const GroupWs& w, const std::vector<DevTables>& dts,
                const slos_group::Cfg& c, hipStream_t st) {
  int active = 0;
  for (size_t g = 0; g < G->plans.size(); ++g) active += G->plans[g]->n >= K;
  if (c.block == 2 || (c.block == -1 && active == 1)) return group_layer_per_plan(G, K, a, w, dts, st);
  slos::GroupLaunch gl{};
  gl.K = K;
  const bool block = group_can_block(G, dts, K, a.flags) && c.block != 0;
  uint64_t children = 0;
  for (size_t g = 0; g < G->plans.size(); ++g)
    if (G->plans[g]->n >= K) children += G->plans[g]->size(K) * (uint64_t)a.B[g];
  uint64_t pw_default = std::min<uint64_t>(std::max<uint64_t>((children / 16384 + 63) & ~63ull, 256), 4096);
  size_t sh = 0;
  uint64_t total = 0;
  int cnt = 0;
  for (size_t g = 0; g < G->plans.size(); ++g) {
    const slos_plan* p = G->plans[g];
    if (p->n < K) continue;
    slos::GroupItem& it = gl.it[cnt++];
    const DevTables& dt = dts[g];
    it.cg = dt.cg;
    it.lo = dt.lo;
    it.tuples = dt.tuples;
    it.U = a.U[g];
    const float2* bufs[2] = {reinterpret_cast<const float2*>(a.ws + w.buf0[g]),
                             reinterpret_cast<const float2*>(a.ws + w.buf1[g])};
    it.par = K == 1 ? reinterpret_cast<const float2*>(a.ws + w.ones[g]) : bufs[(K - 1) & 1];
    const bool last = K == p->n;
    it.out = last ? static_cast<void*>(a.out[g]) : const_cast<float2*>(bufs[K & 1]);
    it.S_par = p->size(K - 1);
    it.S = p->size(K);
    it.S_pre = block ? p->size(K - slos::kSuf) : 0;
    it.kind = last ? 1 : 0;
    it.scale = last ? a.scale[g] : 1.f;
    it.flags = a.flags;
    // compensated sums carry hi/lo layers (the vacuum row of layer 0 has no low part)
    const bool hilo = (a.flags & SLOS_FLAG_COMPENSATED) != 0;
    it.par_lo = (hilo && K >= 2) ? a.B[g] * (int64_t)it.S_par : 0;
    it.out_lo = (hilo && !last) ? a.B[g] * (int64_t)it.S : 0;
    it.me = p->me;
    it.multiset = p->multiset;
    it.m = p->m;
    it.col = p->modes[K - 1];
    uint64_t wgs;
    if (block) {
      it.per_wave = c.per_wave ? c.per_wave : pw_default;
      wgs = ((it.S + it.per_wave - 1) / it.per_wave + slos::kWaves - 1) / slos::kWaves;
      sh = std::max(sh, slos::block_table_offset(K, p->me));
    } else {
      it.per_wave = c.per_wave ? c.per_wave : 1;
      wgs = (it.S + 256 * it.per_wave - 1) / (256 * it.per_wave);
      sh = std::max(sh, simple_lds_bytes(K, p->me, p->m));
    }
    it.wg_begin = (uint32_t)total;
    it.wgs_per_inst = (uint32_t)wgs;
    total += wgs * (uint64_t)a.B[g];
    if (total > 0x7fffffffull) return fail(SLOS_ERANGE, "group layer too large for one launch");
  }
  if (cnt == 0) return SLOS_OK;
  gl.count = cnt;
  gl.total = (uint32_t)total;
  if (block) {
    gl.table_off = (uint32_t)sh;
    sh += (size_t)slos::kWaves * slos::kBlockBatch * slos::block_words(slos::block_maxd(K - slos::kSuf)) * 4;
  }
  if (sh + (block ? slos::kBlockStaticLds : 0) > lds_limit()) return fail(SLOS_ERANGE, "group layer LDS exceeds the GPU's LDS");
  const uint32_t all = (uint32_t)(8 * ((total + 7) / 8));
  const uint32_t grid = c.grid ? std::min<uint32_t>(std::max<uint32_t>(c.grid & ~7u, 8), all) : all;
  const bool comp = a.flags & SLOS_FLAG_COMPENSATED;
  if (block) slos::launch_layer_block_group(comp, K - slos::kSuf, grid, sh, st, gl);
  else
    with_km(K, [&](auto km) {
      constexpr int KM = decltype(km)::value;
      if (comp) hipLaunchKernelGGL((k_layer_simple_group<true, KM>), dim3(grid), dim3(256), sh, st, gl);
      else hipLaunchKernelGGL((k_layer_simple_group<false, KM>), dim3(grid), dim3(256), sh, st, gl);
    });
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

int group_tables(const slos_group* G, std::vector<DevTables>* dts) {
  dts->resize(G->plans.size());
  for (size_t g = 0; g < G->plans.size(); ++g) {
    int rc = device_tables(G->plans[g], &(*dts)[g]);
    if (rc) return rc;
  }
  return SLOS_OK;
}

int group_forward(const slos_group* G, const GroupArgs& a, const GroupWs& w, const std::vector<DevTables>& dts,
                  hipStream_t st) {
  for (size_t g = 0; g < G->plans.size(); ++g) {
    hipLaunchKernelGGL(k_fill_ones, dim3((unsigned)std::min<int64_t>((a.B[g] + 255) / 256, 4096)), dim3(256), 0, st,
                       reinterpret_cast<float2*>(a.ws + w.ones[g]), a.B[g]);
    HIP_TRY(hipGetLastError());
  }
  for (int K = 1; K <= G->nmax; ++K) {
    int rc = group_layer(G, K, a, w, dts, G->cfg[K], st);
    if (rc) return rc;
  }
  return SLOS_OK;
}

void group_drop_graph(slos_group* G) {
  if (G->exec) (void)hipGraphExecDestroy(G->exec);
  if (G->graph) (void)hipGraphDestroy(G->graph);
  G->exec = nullptr;
  G->graph = nullptr;
}

}  // namespace

void build_tuples(slos_plan* p) {
  const auto sv = p->host_view();
  const uint64_t N = p->size(slos::kSuf);
  p->tuples.resize(N);
  for (uint64_t u = 0; u < N; ++u) p->tuples[u] = slos::make_tuple_word(sv, p->multiset, u);
  // 5-position suffixes: positions < 64 keep every rank term inside its packed field
  // (cg[4][1] < 2^24, cg[3][1] and cg[2][1] < 2^16, cg[1][0] < 2^8)
  if (p->n > 5 && p->size(5) <= (4u << 20)) {
    const uint64_t N5 = p->size(5);
    p->tuples5.resize(N5);
    for (uint64_t u = 0; u < N5; ++u) p->tuples5[u] = slos::make_tuple_word<5>(sv, p->multiset, u);
    // the last layer in group order: multiset spaces, prefixes of 2..6 positions
    // (item ranks are 32-bit; at most about 32M items a layer)
    for (int K = 7; K <= p->n && K <= 11; ++K)
      if (p->multiset && p->size(K - 6) <= 0xffffffffull &&
          p->size(K) / slos::kGroupItemChildren + p->size(K - 6) <= (32u << 20))
      {
        slos::group_items(sv, K, p->items[K]);
        if (p->size(K) < DevTables::kFineItems)
          slos::group_items(sv, K, p->fine[K], slos::kGroupFineChildren, slos::kGroupFineWidth);
      }
  }
}

// the keyed group sums of slos_group_sums / slos_group_sums_f64 (k_group_partial, k_group_final)
namespace {

template <class T>
int group_sums(const T* probs, int64_t batch, uint64_t count, const int64_t* order, const int64_t* chunks,
               uint32_t n_chunks, const uint32_t* first, int n_groups, T* out, void* ws, size_t ws_bytes,
               slos_stream_t stream) {
  if (!probs || !order || !first || !out || batch < 1 || batch > 65535 || n_groups < 1 || (n_chunks && !chunks))
    return fail(SLOS_EINVAL, "bad argument");
  if (n_chunks && (!ws || ws_bytes < (size_t)batch * n_chunks * sizeof(double)))
    return fail(SLOS_ENOMEM, "workspace too small");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  double* part = static_cast<double*>(ws);
  if (n_chunks) {
    hipLaunchKernelGGL(k_group_partial<T>, dim3((n_chunks + 3) / 4, (unsigned)batch), dim3(256), 0, st, probs, count,
                       order, chunks, n_chunks, part);
    HIP_TRY(hipGetLastError());
  }
  hipLaunchKernelGGL(k_group_final<T>, dim3((unsigned)((n_groups + 255) / 256), (unsigned)batch), dim3(256), 0, st,
                     part, n_chunks, first, n_groups, out);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

}  // namespace

extern "C" {

const char* slos_version(void) { return "slos_mi355x 0.1 (gfx950)"; }

const char* slos_last_error(void) { return g_err.c_str(); }

int slos_plan_create(int n, int m, int mask, const int32_t* input_modes, slos_plan** out) {
  if (!out) return fail(SLOS_EINVAL, "out is NULL");
  *out = nullptr;
  if (n < 0) return fail(SLOS_EINVAL, "n must be >= 0");
  if (n > kMaxPhotons) return fail(SLOS_ERANGE, "at most 32 photons");
  if (m < 1 || m > 4096) return fail(SLOS_EINVAL, "m must be in [1, 4096]");
  if (!input_modes) return fail(SLOS_EINVAL, "input_modes is NULL");
  auto* p = new slos_plan();
  p->n = n; p->m = m; p->mask = mask;
  switch (mask) {
    case SLOS_MASK_FOCK: p->me = m; p->multiset = 1; break;
    case SLOS_MASK_UNBUNCHED: p->me = m; p->multiset = 0; p->shift = 0; break;
    case SLOS_MASK_DUAL_RAIL: p->me = m; p->multiset = 0; p->shift = 1; break;
    case SLOS_MASK_SPARSE_1IN4: p->me = m; p->multiset = 0; p->shift = 2; break;
    case SLOS_MASK_TAIL_EMPTY: p->me = m - 2; p->multiset = 1; break;
    default: delete p; return fail(SLOS_EINVAL, "unknown mask id " + std::to_string(mask));
  }
  if (p->me < 1) { delete p; return fail(SLOS_EINVAL, "empty output space (too few modes for the mask)"); }
  std::vector<int> cnt(m, 0);
  for (int k = 0; k < n; ++k) {
    if (input_modes[k] < 0 || input_modes[k] >= m) { delete p; return fail(SLOS_EINVAL, "input mode out of range"); }
    p->modes.push_back(input_modes[k]);
    cnt[input_modes[k]]++;
  }
  for (int c : cnt) for (int i = 2; i <= c; ++i) p->s_fact *= i;
  p->lo.resize(p->me);
  for (int x = 0; x < p->me; ++x) {
    const int v = p->multiset ? x : (((x >> p->shift) + 1) << p->shift);
    p->lo[x] = std::min(v, p->me);
  }
  const int st = p->me + 1;
  p->cg.assign((size_t)(n + 2) * st, 0);
  for (int x = 0; x <= p->me; ++x) p->cg[x] = 1;
  for (int r = 1; r <= n + 1; ++r)
    for (int x = p->me - 1; x >= 0; --x) {
      uint64_t v;
      if (__builtin_add_overflow(p->cg[(size_t)r * st + x + 1], p->cg[(size_t)(r - 1) * st + p->lo[x]], &v)) {
        if (r <= n) { delete p; return fail(SLOS_ERANGE, "layer size exceeds 64 bits"); }
        v = UINT64_MAX;  // row n+1 is only a guard
      }
      p->cg[(size_t)r * st + x] = v;
    }
  // the block kernel's tuple words hold positions < 64 (6 bits and a mark bit per byte)
  if (n > slos::kSuf && p->m <= slos::kBlockModes && p->size(slos::kSuf) <= (4u << 20)) build_tuples(p);
  if (p->size(n) == 0) {
    delete p;
    return fail(SLOS_EINVAL, "empty output space for n=" + std::to_string(n) + " m=" + std::to_string(m));
  }
  *out = p;
  return SLOS_OK;
}

int slos_plan_destroy(slos_plan* p) {
  if (!p) return SLOS_OK;
  int cur = 0;
  (void)hipGetDevice(&cur);
  for (auto& t : p->dev) {
    (void)hipSetDevice(t.device);
    (void)hipFree(t.cg);
    (void)hipFree(t.lo);
    (void)hipFree(t.modes);
    if (t.tuples) (void)hipFree(t.tuples);
    if (t.tuples5) (void)hipFree(t.tuples5);
    if (t.insert) (void)hipFree(t.insert);
    for (auto* x : t.xm)
      if (x) (void)hipFree(x);
    for (auto* it : t.items)
      if (it) (void)hipFree(it);
    for (auto* it : t.fine)
      if (it) (void)hipFree(it);
  }
  (void)hipSetDevice(cur);
  delete p;
  return SLOS_OK;
}

int slos_layer_size(const slos_plan* p, int k, uint64_t* size) {
  if (!p || !size) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 0 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  *size = p->size(k);
  return SLOS_OK;
}

int slos_rank(const slos_plan* p, int k, const int32_t* pos, int64_t count, uint64_t* idx) {
  if (!p || (!pos && count) || (!idx && count)) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 0 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  const auto sv = p->host_view();
  for (int64_t q = 0; q < count; ++q) {
    const int32_t* t = pos + q * k;
    int l = 0, run = 0;
    for (int i = 0; i < k; ++i) {
      if (t[i] < l || t[i] >= p->me) return fail(SLOS_EINVAL, "positions do not describe an admissible sorted state");
      run = (i > 0 && t[i] == t[i - 1]) ? run + 1 : 1;
      if (sv.C(k - i - 1, p->lo[t[i]]) == 0) return fail(SLOS_EINVAL, "state has no admissible completion");
      l = p->lo[t[i]];
    }
    (void)run;
    idx[q] = sv.rank(reinterpret_cast<const int*>(t), k);
  }
  return SLOS_OK;
}

int slos_unrank(const slos_plan* p, int k, const uint64_t* idx, int64_t count, int32_t* pos) {
  if (!p || (!pos && count) || (!idx && count)) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 0 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  const auto sv = p->host_view();
  const uint64_t S = p->size(k);
  for (int64_t q = 0; q < count; ++q) {
    if (idx[q] >= S) return fail(SLOS_ERANGE, "index >= layer size");
    sv.unrank(idx[q], k, reinterpret_cast<int*>(pos + q * k));
  }
  return SLOS_OK;
}

int slos_prob_norms(const slos_plan* p, int k, uint64_t first, int64_t count, double* out) {
  if (!p || (!out && count)) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 0 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  const uint64_t S = p->size(k);
  if (count < 0 || first > S || (uint64_t)count > S - first) return fail(SLOS_ERANGE, "range outside the layer");
  const auto sv = p->host_view();
  int t[kMaxPhotons];
  for (int64_t q = 0; q < count; ++q) {
    sv.unrank(first + q, k, t);
    double f = 1, run = 1;
    if (p->multiset)
      for (int i = 1; i < k; ++i) {
        run = (t[i] == t[i - 1]) ? run + 1 : 1;
        f *= run;
      }
    out[q] = f;
  }
  return SLOS_OK;
}

int slos_forward_workspace(const slos_plan* p, int64_t batch, int layer, unsigned flags, size_t* bytes) {
  if (!p || !bytes) return fail(SLOS_EINVAL, "NULL argument");
  if (batch < 1) return fail(SLOS_EINVAL, "batch must be >= 1");
  if (layer < 0 || layer > p->n) return fail(SLOS_EINVAL, "layer out of range");
  if ((flags & SLOS_FLAG_F64) && (flags & (SLOS_FLAG_COMPENSATED | SLOS_FLAG_HILO)))
    return fail(SLOS_EINVAL, "SLOS_FLAG_F64 computes in FP64: no compensated sums");
  WsLayout w;
  int rc = forward_layout(p, batch, layer, &w, (flags & SLOS_FLAG_COMPENSATED) != 0, (flags & SLOS_FLAG_F64) != 0);
  if (rc) return rc;
  *bytes = w.total;
  return SLOS_OK;
}

namespace {

// argument checks shared by slos_forward and slos_forward_noalloc: the input columns and the
// workspace layout
int forward_check(const slos_plan* p, const void* U, int64_t batch, const int32_t* modes, int layer, int out_kind,
                  void* out, unsigned flags, int* cols, WsLayout* w) {
  if (!p || !U || !out) return fail(SLOS_EINVAL, "NULL argument");
  if (batch < 1) return fail(SLOS_EINVAL, "batch must be >= 1");
  if (layer < 0 || layer > p->n) return fail(SLOS_EINVAL, "layer out of range");
  if (out_kind != SLOS_OUT_PROBS && out_kind != SLOS_OUT_AMPS) return fail(SLOS_EINVAL, "unknown output kind");
  for (int k = 0; k < layer; ++k) {
    cols[k] = modes ? modes[k] : p->modes[k];
    if (cols[k] < 0 || cols[k] >= p->m) return fail(SLOS_EINVAL, "input mode out of range");
  }
  if ((flags & SLOS_FLAG_F64) && (flags & (SLOS_FLAG_COMPENSATED | SLOS_FLAG_HILO)))
    return fail(SLOS_EINVAL, "SLOS_FLAG_F64 computes in FP64: no compensated sums");
  return forward_layout(p, batch, layer, w, (flags & SLOS_FLAG_COMPENSATED) != 0, (flags & SLOS_FLAG_F64) != 0);
}

// the complex128 forward (SLOS_FLAG_F64): the same layer walk as forward_run, FP64 kernels
int forward_run_f64(const slos_plan* p, const DevTables& dt, const void* U, slos::MatrixStride us, int64_t batch, const int* cols, int layer,
                    int out_kind, void* out, double scale, unsigned flags, const WsLayout& w, void* ws,
                    hipStream_t st) {
  auto* base = static_cast<unsigned char*>(ws);
  double2* ones = reinterpret_cast<double2*>(base + w.ones);
  void* bufs[2] = {base + w.even, base + w.odd};
  const dim3 g1((unsigned)std::min<int64_t>((batch + 255) / 256, 4096));
  if (layer == 0) {  // no photon: the vacuum
    hipLaunchKernelGGL(slos::k_vacuum_out_f64, g1, dim3(256), 0, st, out, batch, out_kind == SLOS_OUT_PROBS ? 1 : 0,
                       scale);
    HIP_TRY(hipGetLastError());
    return SLOS_OK;
  }
  const RoctxRange whole("slos_forward");
  const void* par = ones;
  uint64_t S_par = 1;
  size_t lds = 0;
  uint32_t buf = 0;
  const int kf = (flags & (SLOS_FLAG_SIMPLE | SLOS_FLAG_BLOCK)) ? 0 : front_layers(p, batch, layer, 16, false, &lds, &buf);
  if (kf) {
    void* dst = kf == layer ? out : bufs[kf & 1];
    const int rc = run_front(p, dt, kf, cols, U, us, batch, dst, kf < layer ? 0 : out_kind == SLOS_OUT_PROBS ? 1 : 2, scale,
                             flags, lds, buf, false, st);
    if (rc) return rc;
    par = dst;
    S_par = p->size(kf);
  } else {
    hipLaunchKernelGGL(slos::k_fill_ones_f64, g1, dim3(256), 0, st, ones, batch);
    HIP_TRY(hipGetLastError());
  }
  for (int k = kf + 1; k <= layer; ++k) {
    const uint64_t S = p->size(k);
    const bool last = (k == layer);
    void* dst = last ? out : bufs[k & 1];
    const int kind = last ? (out_kind == SLOS_OUT_PROBS ? 1 : 2) : 0;
    char name[32];
    std::snprintf(name, sizeof name, "slos layer %d", k);
    const RoctxRange range(name);
    const int rc = launch_layer_f64(p, dt, k, cols[k - 1], U, us, batch, par, S_par, dst, S, kind, scale, flags, st);
    if (rc) return rc;
    par = dst;
    S_par = S;
  }
  return SLOS_OK;
}

// the layer launches of a forward whose workspace `ws` follows layout `w` (no allocation)
int forward_run(const slos_plan* p, const DevTables& dt, const void* U, slos::MatrixStride us, int64_t batch, const int* cols, int layer,
                int out_kind, void* out, double scale, unsigned flags, const WsLayout& w, void* ws, hipStream_t st) {
  if (flags & SLOS_FLAG_F64) return forward_run_f64(p, dt, U, us, batch, cols, layer, out_kind, out, scale, flags, w, ws, st);
  int rc = SLOS_OK;
  auto* base = static_cast<unsigned char*>(ws);
  float2* ones = reinterpret_cast<float2*>(base + w.ones);
  float2* bufs[2] = {reinterpret_cast<float2*>(base + w.even), reinterpret_cast<float2*>(base + w.odd)};
  if (layer == 0) {  // no photon: the vacuum
    hipLaunchKernelGGL(k_vacuum_out, dim3((unsigned)std::min<int64_t>((batch + 255) / 256, 4096)), dim3(256), 0, st, out,
                       batch, out_kind == SLOS_OUT_PROBS ? 1 : 0, (float)scale);
    HIP_TRY(hipGetLastError());
    return SLOS_OK;
  }
  const float2* Uf = static_cast<const float2*>(U);
  const float2* par = ones;
  uint64_t S_par = 1;
  // compensated sums: every intermediate layer is a hi/lo pair [2][B][S] (the buffers are sized for it)
  const bool hilo = (flags & SLOS_FLAG_COMPENSATED) != 0;
  const RoctxRange whole("slos_forward");
  size_t lds = 0;
  uint32_t buf = 0;
  const int kf = (flags & (SLOS_FLAG_SIMPLE | SLOS_FLAG_BLOCK)) ? 0 : front_layers(p, batch, layer, 8, hilo, &lds, &buf);
  if (kf) {
    void* dst = kf == layer ? out : bufs[kf & 1];
    rc = run_front(p, dt, kf, cols, U, us, batch, dst, kf < layer ? 0 : out_kind == SLOS_OUT_PROBS ? 1 : 2, scale, flags, lds,
                   buf, hilo && kf < layer, st);
    if (rc) return rc;
    par = static_cast<const float2*>(dst);
    S_par = p->size(kf);
  } else {
    hipLaunchKernelGGL(k_fill_ones, dim3((unsigned)std::min<int64_t>((batch + 255) / 256, 4096)), dim3(256), 0, st,
                       ones, batch);
    HIP_TRY(hipGetLastError());
  }
  for (int k = kf + 1; k <= layer; ++k) {
    const uint64_t S = p->size(k);
    const bool last = (k == layer);
    void* dst = last ? out : bufs[k & 1];
    const int kind = last ? (out_kind == SLOS_OUT_PROBS ? 1 : 2) : 0;
    char name[32];
    std::snprintf(name, sizeof name, "slos layer %d", k);
    const RoctxRange range(name);
    rc = launch_layer(p, dt, k, cols[k - 1], Uf, us, batch, par, S_par, dst, S, kind, (float)scale, flags & ~SLOS_FLAG_HILO,
                      st, hilo && k >= 2, hilo && !last);
    if (rc) return rc;
    par = static_cast<const float2*>(dst);
    S_par = S;
  }
  return SLOS_OK;
}

}  // namespace

// Scratch of slos_forward_noalloc: the vacuum row and the two ping-pong layers, one copy per GPU
// (held until the process ends). Host code never passes the symbol itself to a kernel: its device
// address comes from hipGetSymbolAddress, once per device.
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

struct ScratchSlot {
  int device;
  void* ptr;
};
std::mutex g_scratch_mu;
std::vector<ScratchSlot> g_scratch;

// device address of the current GPU's scratch array (looked up on the first call on each GPU)
int scratch_address(void** out) {
  int d = 0;
  HIP_TRY(hipGetDevice(&d));
  std::lock_guard<std::mutex> g(g_scratch_mu);
  for (const auto& s : g_scratch)
    if (s.device == d) {
      *out = s.ptr;
      return SLOS_OK;
    }
  void* ptr = nullptr;
  HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  if (!ptr) return fail(SLOS_EHIP, "hipGetSymbolAddress(scratch) returned NULL");
  g_scratch.push_back(ScratchSlot{d, ptr});
  *out = ptr;
  return SLOS_OK;
}

// the plan's tables on the current GPU if they are already resident (no allocation)
int resident_tables(const slos_plan* cp, DevTables* out) {
  slos_plan* p = const_cast<slos_plan*>(cp);
  int d = 0;
  HIP_TRY(hipGetDevice(&d));
  std::lock_guard<std::mutex> g(p->mu);
  for (auto& t : p->dev)
    if (t.device == d) {
      *out = t;
      return SLOS_OK;
    }
  return fail(SLOS_EINVAL, "the plan has no tables on this GPU yet: run slos_forward (or slos_layer_step) with "
                           "this plan once on it first");
}

}  // namespace

int slos_forward_strided(const slos_plan* p, const void* U, const int64_t* strides, int64_t batch, const int32_t* modes, int layer, int out_kind,
                 void* out, double scale, unsigned flags, void* ws, size_t ws_bytes, slos_stream_t stream) {
  int cols[kMaxPhotons] = {};  // layer <= n <= 32 (checked before cols is written)
  WsLayout w;
  int rc = forward_check(p, U, batch, modes, layer, out_kind, out, flags, cols, &w);
  if (rc) return rc;
  if (!strides) return fail(SLOS_EINVAL, "NULL argument");
  if (!ws || ws_bytes < w.total)
    return fail(SLOS_ENOMEM, "workspace too small: need " + std::to_string(w.total) + " bytes");
  DevTables dt;
  rc = device_tables(p, &dt);
  if (rc) return rc;
  return forward_run(p, dt, U, slos::MatrixStride{strides[0], strides[1], strides[2]}, batch, cols, layer, out_kind, out, scale, flags, w, ws,
                     reinterpret_cast<hipStream_t>(stream));
}

int slos_forward(const slos_plan* p, const void* U, int64_t batch, const int32_t* modes, int layer, int out_kind,
                 void* out, double scale, unsigned flags, void* ws, size_t ws_bytes, slos_stream_t stream) {
  if (!p) return fail(SLOS_EINVAL, "NULL argument");
  const int64_t m = p->m, packed[3] = {m * m, m, 1};
  return slos_forward_strided(p, U, packed, batch, modes, layer, out_kind, out, scale, flags, ws, ws_bytes, stream);
}

int slos_forward_noalloc(const slos_plan* p, const void* U, int64_t batch, const int32_t* modes, int layer,
                         int out_kind, void* out, double scale, unsigned flags, slos_stream_t stream) {
  int cols[kMaxPhotons] = {};  // layer <= n <= 32 (checked before cols is written)
  WsLayout w;
  int rc = forward_check(p, U, batch, modes, layer, out_kind, out, flags, cols, &w);
  if (rc) return rc;
  if (w.total > kNoAllocScratchBytes)
    return fail(SLOS_ERANGE, "slos_forward_noalloc: the intermediate layers need " + std::to_string(w.total) +
                                 " bytes, above its fixed scratch of " + std::to_string(kNoAllocScratchBytes) +
                                 " bytes; use slos_forward with a workspace");
  DevTables dt;
  rc = resident_tables(p, &dt);
  if (rc) return rc;
  void* ws = nullptr;
  rc = scratch_address(&ws);
  if (rc) return rc;
  return forward_run(p, dt, U, slos::packed_stride(p->m), batch, cols, layer, out_kind, out, scale, flags, w, ws,
                     reinterpret_cast<hipStream_t>(stream));
}

int slos_layer_step(const slos_plan* p, const void* U, int64_t batch, int k, int col, const void* psi_prev,
                    int out_kind, void* out, double scale, unsigned flags, slos_stream_t stream) {
  if (!p || !U || !psi_prev || !out) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 1 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  if (col < 0 || col >= p->m) return fail(SLOS_EINVAL, "input mode out of range");
  if (batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
  if (out_kind < 0 || out_kind > 2) return fail(SLOS_EINVAL, "unknown output kind");
  DevTables dt;
  int rc = device_tables(p, &dt);
  if (rc) return rc;
  const int kind = out_kind == 2 ? 0 : (out_kind == SLOS_OUT_PROBS ? 1 : 2);
  if (flags & SLOS_FLAG_F64) {
    if (flags & (SLOS_FLAG_COMPENSATED | SLOS_FLAG_HILO))
      return fail(SLOS_EINVAL, "SLOS_FLAG_F64 computes in FP64: no compensated sums");
    return launch_layer_f64(p, dt, k, col, U, slos::packed_stride(p->m), batch, psi_prev, p->size(k - 1), out, p->size(k), kind, scale, flags,
                            reinterpret_cast<hipStream_t>(stream));
  }
  const bool hilo = (flags & SLOS_FLAG_HILO) && (flags & SLOS_FLAG_COMPENSATED);
  if ((flags & SLOS_FLAG_HILO) && !(flags & SLOS_FLAG_COMPENSATED))
    return fail(SLOS_EINVAL, "SLOS_FLAG_HILO needs SLOS_FLAG_COMPENSATED");
  return launch_layer(p, dt, k, col, static_cast<const float2*>(U), slos::packed_stride(p->m), batch, static_cast<const float2*>(psi_prev),
                      p->size(k - 1), out, p->size(k), kind, (float)scale, flags & ~SLOS_FLAG_HILO,
                      reinterpret_cast<hipStream_t>(stream), hilo, hilo && kind == 0);
}

int slos_readout_adjoint(const slos_plan* p, int64_t batch, const void* amps, const float* grad_p, double scale,
                         void* grad_amps, slos_stream_t stream) {
  if (!p || !amps || !grad_p || !grad_amps) return fail(SLOS_EINVAL, "NULL argument");
  if (batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
  DevTables dt;
  int rc = device_tables(p, &dt);
  if (rc) return rc;
  const uint64_t S = p->size(p->n);
  const size_t sh = (size_t)(p->n + 1) * (p->me + 1) * 8 + (size_t)p->me * 4;
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  dim3 grid((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((S + 255) / 256, 1u << 20)),
            (unsigned)std::min<int64_t>(batch, 16));
  hipLaunchKernelGGL(k_readout_adjoint, grid, dim3(256), sh, reinterpret_cast<hipStream_t>(stream), dt.cg, dt.lo,
                     p->me, p->multiset, p->n, static_cast<const float2*>(amps), grad_p,
                     static_cast<float2*>(grad_amps), S, batch, (float)(scale * scale));
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

namespace {

int run_readout_pull(const slos_plan* p, const DevTables& dt, const float2* U, int64_t batch, int col, const float2* psi_prev,
                     const float* grad_p, double scale, float2* grad_amps, hipStream_t st) {
  const int K = p->n;
  const uint64_t S = p->size(K);
  dim3 grid((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((S + 255) / 256, 1u << 20)),
            (unsigned)std::min<int64_t>(batch, 16));
  with_km(K, [&](auto km) {
    hipLaunchKernelGGL((k_readout_adjoint_pull<decltype(km)::value>), grid, dim3(256), 0, st, dt.cg, dt.lo, p->me,
                       p->multiset, K, p->m, col, U, psi_prev, p->size(K - 1), grad_p, grad_amps, S, batch,
                       (float)(scale * scale));
  });
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

}  // namespace

int slos_readout_adjoint_pull(const slos_plan* p, const void* U, int64_t batch, const void* psi_prev,
                              const float* grad_p, double scale, void* grad_amps, slos_stream_t stream) {
  if (!p || !U || !psi_prev || !grad_p || !grad_amps) return fail(SLOS_EINVAL, "NULL argument");
  if (batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
  if (p->n < 1) return fail(SLOS_EINVAL, "no photon layer");
  DevTables dt;
  const int rc = device_tables(p, &dt);
  if (rc) return rc;
  return run_readout_pull(p, dt, static_cast<const float2*>(U), batch, p->modes[p->n - 1],
                          static_cast<const float2*>(psi_prev), grad_p, scale, static_cast<float2*>(grad_amps),
                          reinterpret_cast<hipStream_t>(stream));
}

// work groups of the thread-per-state adjoint (grid-stride over the parents; one FP64 partial per
// work group and mode)
static int adjoint_blocks(uint64_t Sp) { return (int)std::max<uint64_t>(1, std::min<uint64_t>((Sp + 63) / 64, 1u << 16)); }

namespace {

// parents per XCD chunk of the insert-table adjoint (see slos::xcd_chunk_index)
constexpr uint64_t kAdjChunkParents = 1ull << 18;

// How one adjoint layer runs: the kernel with a lane a mode, the insert-table kernel or the
// thread-per-state kernel; `nblk` work groups, each writing one FP64 partial per mode.
struct AdjLaunch {
  bool walk = false;
  uint32_t turns = 0;  // parents a group, of the kernel with a lane a mode (0: another kernel)
  uint64_t per_wave = 0;
  uint32_t xcd_chunk = 1;
  size_t lds = 0;   // of the thread-per-state kernel
  uint64_t nblk = 0;
};

// the insert-table kernel: parent prefixes of 0..8 positions, up to 32 modes (its sums' registers)
bool adjoint_walk(const slos_plan* p, int k) {
  const int dp = k - 1 - slos::kSuf;
  return has_insert_table(p) && dp >= 0 && dp <= 8 && p->me <= 32;
}

// Whether an adjoint layer takes the kernel with a lane a mode. It is quick to start and computes each
// child's index anew: the one for few parents, and for many modes, where the thread-per-state kernel has
// few waves (its sums' LDS). Adjoint layers with their sums, us, lane a mode / walk: 98k parents in all (24
// modes) 31 / 35, 171k (14) 35 / 29, 377k (32) 68 / 57; lane a mode / thread per state: 17k (24) 26 / 38, 119k (14)
// 30 / 34, 273k (12) 54 / 42, 886k (20) 100 / 116, 209k (32) 44 / 92, 766k (64) 234 / 592, 1.1M (40) 268 / 417. In set
// masks most modes have no child: sparse_1in4, 2.6M (20) 335 / 152, 1.2M (24) 129 / 102, 1.1M (32) 132 / 202; dual rail,
// 672k (20) 73 / 62, 253k (24) 36 / 46; collision-free 1.6M (20) 165 / 171. Where the thread-per-state forms are
// exact (parents of at most 3 photons), and in sparse_1in4, it must fill its 32 or 64 lanes to four fifths: 3 photons, 78k
// (24) 29 / 28, 520k (24) 99 / 89, 598k (32) 123 / 176, 574k (40) 239 / 191, 915k (64) 503 / 696; sparse_1in4 1.9M (36) 363 / 332.
bool adjoint_modes(const slos_plan* p, int k, int64_t batch) {
  if (k - 1 > slos::kModesPhotons || p->me > 64 || p->size(k) >= (1ull << 31)) return false;
  return p->size(k - 1) <= (k - 1 <= 3 ? 1ull << 16 : 1ull << 17) / (uint64_t)batch ||
         (!adjoint_walk(p, k) && p->me >= 20 + 4 * p->shift &&
          ((k - 1 > 3 && p->shift < 2) || 5 * p->me >= 4 * slos::modes_lanes(p->me)));
}

// modes: the kernel with a lane a mode, else the walk or the thread-per-state kernel
int adjoint_launch(const slos_plan* p, int k, bool modes, AdjLaunch* L) {
  const uint64_t Sp = p->size(k - 1);
  L->lds = (((size_t)(k + 1) * (p->me + 1) * 8 + p->me * 4 + 15) & ~(size_t)15) + (size_t)p->m * 8 +
           (size_t)kAdjThreads * p->me * 8;
  if (modes) {
    const uint32_t groups = slos::modes_groups(p->me);
    L->turns = (uint32_t)std::min<uint64_t>(8, std::max<uint64_t>(1, Sp / (groups * 64u)));
    L->nblk = (Sp + groups * L->turns - 1) / (groups * L->turns);
    return SLOS_OK;
  }
  L->walk = adjoint_walk(p, k);
  if (L->walk) {
    // parents per wave: at most about 2^16 work groups (FP64 partials per mode), and else as few as
    // pay for a wave's sum over its lanes (us with 128 / 256 / 512: 2.0M parents 137 / 119 / 112,
    // 475k 55 / 60 / 73, 2.2M 147 / 130 / 153, 76k 57 / 80 / 92)
    uint64_t pw = (Sp / ((uint64_t)slos::kWaves << 16) + slos::kAdjChunk - 1) & ~(uint64_t)(slos::kAdjChunk - 1);
    pw = std::max<uint64_t>(pw, Sp < (1ull << 20) ? 128 : 256);
    const uint64_t wgs = ((Sp + pw - 1) / pw + slos::kWaves - 1) / slos::kWaves;
    if (wgs > 0x7fffffffull) return fail(SLOS_ERANGE, "layer too large for one launch");
    L->per_wave = pw;
    L->xcd_chunk = (uint32_t)std::max<uint64_t>(1, kAdjChunkParents / ((uint64_t)slos::kWaves * pw));
    L->nblk = wgs;
    return SLOS_OK;
  }
  if (L->lds > lds_limit()) return fail(SLOS_ERANGE, "adjoint LDS exceeds the GPU's LDS (too many modes)");
  L->nblk = adjoint_blocks(Sp);
  return SLOS_OK;
}

}  // namespace

int slos_adjoint_workspace(const slos_plan* p, int64_t batch, int k, size_t* bytes) {
  if (!p || !bytes) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 1 || k > p->n || batch < 1) return fail(SLOS_EINVAL, "bad argument");
  // (enough for every smaller batch too, whichever kernel that takes)
  uint64_t nblk = 0;
  for (const bool modes : {false, true}) {
    if (modes && !adjoint_modes(p, k, 1)) break;
    AdjLaunch L;
    const int rc = adjoint_launch(p, k, modes, &L);
    if (rc && !(rc == SLOS_ERANGE && adjoint_modes(p, k, batch))) return rc;
    nblk = std::max(nblk, L.nblk);
  }
  *bytes = (size_t)batch * nblk * p->me * sizeof(double2);
  return SLOS_OK;
}

namespace {

// the FP64 partials of layer k's dL/dU column and (unless null) grad_prev, as `L` (adjoint_launch)
int run_adjoint(const slos_plan* p, const DevTables& dt, const AdjLaunch& L, const float2* U, int64_t batch, int k, int col,
                const float2* psi, const float2* gk, float2* gout, double2* part, hipStream_t st) {
  const uint64_t Sp = p->size(k - 1), Sk = p->size(k);
  if (L.turns) {
    slos::AdjointModesArgs a{};
    a.cg = dt.cg; a.lo = dt.lo; a.tuples = dt.tuples; a.tuples5 = dt.tuples5;
    a.me = p->me; a.multiset = p->multiset; a.m = p->m; a.col = col;
    a.U = U; a.psi = psi; a.gk = gk; a.gout = gout; a.Sp = (uint32_t)Sp; a.Sk = (uint32_t)Sk; a.turns = L.turns;
    a.partial = part;
    slos::launch_adjoint_modes(k - 1, dim3((unsigned)L.nblk, (unsigned)batch), st, a);
    HIP_TRY(hipGetLastError());
    return SLOS_OK;
  }
  const uint32_t* ins = nullptr;
  if (L.walk) {
    const int rc = insert_table(p, st, &ins);
    if (rc) return rc;
  }
  if (ins) {
    const slos::BlockGrid bg{dim3((unsigned)L.nblk, (unsigned)batch), 0, st, dt.cg, dt.lo, dt.tuples, p->me, p->multiset};
    slos::launch_adjoint_insert(k - 1 - slos::kSuf, bg, p->m, col, U, psi, gk, Sk, gout, Sp, L.per_wave, L.xcd_chunk, part,
                                ins);
  } else {  // (also inside a capture that comes before the first use of the table)
    if (L.lds > lds_limit()) return fail(SLOS_ERANGE, "adjoint LDS exceeds the GPU's LDS (too many modes)");
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)L.nblk, (unsigned)batch), dim3(kAdjThreads), L.lds, st, dt.cg, dt.lo, p->me,
                         p->multiset, k, p->m, col, U, psi, gk, Sk, gout, Sp, part, gout != nullptr);
    };
    const bool narrow = Sk < (1ull << 32);
    if (narrow && k == 2) launch(k_adjoint_layer<1, slos::SpaceView32, true>);
    else if (narrow && k == 3) launch(k_adjoint_layer<2, slos::SpaceView32, true>);
    else if (narrow && k == 4) launch(k_adjoint_layer<3, slos::SpaceView32, true>);
    else if (narrow && k == 5) launch(k_adjoint_layer<4, slos::SpaceView32, true>);
    else with_km(k - 1, [&](auto km) { launch(k_adjoint_layer<decltype(km)::value>); });
  }
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

}  // namespace

int slos_adjoint_layer(const slos_plan* p, const void* U, int64_t batch, int k, int col, const void* psi_prev,
                       const void* grad_k, void* grad_prev, void* grad_U, int accumulate, void* ws, size_t ws_bytes,
                       slos_stream_t stream) {
  if (!p || !U || !psi_prev || !grad_k || !grad_U) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 1 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  if (col < 0 || col >= p->m) return fail(SLOS_EINVAL, "input mode out of range");
  if (batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
  AdjLaunch L;
  int rc = adjoint_launch(p, k, adjoint_modes(p, k, batch), &L);
  if (rc) return rc;
  if (!ws || ws_bytes < (size_t)batch * L.nblk * p->me * sizeof(double2)) return fail(SLOS_ENOMEM, "workspace too small");
  DevTables dt;
  rc = device_tables(p, &dt);
  if (rc) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  rc = run_adjoint(p, dt, L, static_cast<const float2*>(U), batch, k, col, static_cast<const float2*>(psi_prev),
                   static_cast<const float2*>(grad_k), static_cast<float2*>(grad_prev), static_cast<double2*>(ws), st);
  if (rc) return rc;
  hipLaunchKernelGGL(k_reduce_gu, dim3((unsigned)p->me, (unsigned)batch), dim3(kReduceThreads), 0, st,
                     static_cast<const double2*>(ws), (int)L.nblk, p->me, p->m, col, static_cast<float2*>(grad_U), accumulate);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

namespace {

// the layers 0..layer-1 a backward pass reads, one after another [batch][S_k] at multiples of 256 bytes
int saved_layout(const slos_plan* p, int64_t batch, int layer, std::vector<size_t>* at, size_t* total) {
  uint64_t sum = 0;
  for (int k = 0; k < layer; ++k) {
    uint64_t bytes;
    at->push_back((size_t)sum);
    if (mul_overflow(p->size(k), (uint64_t)batch * sizeof(float2), &bytes) || bytes > (1ull << 62) ||
        __builtin_add_overflow(sum, align256((size_t)bytes), &sum))
      return fail(SLOS_ERANGE, "layer sizes overflow");
  }
  *total = (size_t)sum;
  return SLOS_OK;
}

// workspace of a backward pass: the partials of every layer, and the gradients of two layers in turn
struct BackLayout {
  std::vector<AdjLaunch> L;       // of layer k at k - 1
  std::vector<size_t> part;       // its partials (bytes from the workspace's begin)
  size_t g[2] = {0, 0};           // gradients of the layers top, top - 2, ..; top - 1, .. (top: `layer`, or the one below)
  size_t total = 0;
};

int back_layout(const slos_plan* p, int64_t batch, int layer, bool readout, BackLayout* b) {
  size_t sum = 0;
  for (int k = 1; k <= layer; ++k) {
    AdjLaunch L;
    const int rc = adjoint_launch(p, k, adjoint_modes(p, k, batch), &L);
    if (rc) return rc;
    b->L.push_back(L);
    b->part.push_back(sum);
    sum += align256((size_t)batch * L.nblk * p->me * sizeof(double2));
  }
  // (a mask's layers need not shrink with the photons: the largest of those a buffer holds in turn)
  for (int i = 0; i < 2; ++i) {
    uint64_t most = 0;
    for (int k = readout ? layer - i : layer - 1 - i; k >= 1; k -= 2) most = std::max(most, p->size(k));
    b->g[i] = sum;
    sum += align256((size_t)batch * most * sizeof(float2));
  }
  b->total = sum;
  return SLOS_OK;
}

}  // namespace

int slos_saved_bytes(const slos_plan* p, int64_t batch, int layer, size_t* bytes) {
  if (!p || !bytes) return fail(SLOS_EINVAL, "NULL argument");
  if (layer < 1 || layer > p->n || batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "bad argument");
  std::vector<size_t> at;
  return saved_layout(p, batch, layer, &at, bytes);
}

int slos_forward_saved(const slos_plan* p, const void* U, int64_t batch, const int32_t* modes, int layer, int probs,
                       void* out, double scale, void* saved, size_t saved_bytes, slos_stream_t stream) {
  int cols[kMaxPhotons] = {};
  WsLayout w;
  int rc = forward_check(p, U, batch, modes, layer, probs ? SLOS_OUT_PROBS : SLOS_OUT_AMPS, out, 0u, cols, &w);
  if (rc) return rc;
  if (layer < 1 || batch > 65535) return fail(SLOS_EINVAL, "bad argument");
  std::vector<size_t> at;
  size_t total = 0;
  rc = saved_layout(p, batch, layer, &at, &total);
  if (rc) return rc;
  if (!saved || saved_bytes < total) return fail(SLOS_ENOMEM, "buffer of the layers too small");
  DevTables dt;
  rc = device_tables(p, &dt);
  if (rc) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  void* layers[kMaxPhotons];
  for (int k = 0; k < layer; ++k) layers[k] = static_cast<unsigned char*>(saved) + at[k];
  const RoctxRange whole("slos_forward");
  size_t lds = 0;
  uint32_t buf = 0;
  const int kf = front_layers(p, batch, layer - 1, 8, false, &lds, &buf);
  if (kf) {
    rc = run_front(p, dt, kf, cols, U, slos::packed_stride(p->m), batch, layers[kf], 0, 1.0, 0u, lds, buf, false, st, layers);
    if (rc) return rc;
  } else {
    hipLaunchKernelGGL(k_fill_ones, dim3((unsigned)std::min<int64_t>((batch + 255) / 256, 4096)), dim3(256), 0, st,
                       static_cast<float2*>(layers[0]), batch);
    HIP_TRY(hipGetLastError());
  }
  for (int k = kf + 1; k <= layer; ++k) {
    const bool last = k == layer;
    rc = launch_layer(p, dt, k, cols[k - 1], static_cast<const float2*>(U), slos::packed_stride(p->m), batch,
                      static_cast<const float2*>(layers[k - 1]), p->size(k - 1), last ? out : layers[k], p->size(k),
                      last && probs ? 1 : 0, last ? (float)scale : 1.f, 0u, st);
    if (rc) return rc;
  }
  return SLOS_OK;
}

int slos_backward_workspace(const slos_plan* p, int64_t batch, int layer, int grad_kind, size_t* bytes) {
  if (!p || !bytes) return fail(SLOS_EINVAL, "NULL argument");
  if (layer < 1 || layer > p->n || batch < 1 || batch > 65535 || grad_kind < 0 || grad_kind > 2)
    return fail(SLOS_EINVAL, "bad argument");
  BackLayout b;
  const int rc = back_layout(p, batch, layer, grad_kind != 0, &b);
  *bytes = b.total;
  return rc;
}

int slos_backward(const slos_plan* p, const void* U, int64_t batch, const int32_t* modes, int layer, const void* saved,
                  size_t saved_bytes, const void* grad, int grad_kind, double scale, void* grad_U, void* ws,
                  size_t ws_bytes, slos_stream_t stream) {
  if (!p || !U || !saved || !grad || !grad_U || !ws) return fail(SLOS_EINVAL, "NULL argument");
  if (layer < 1 || layer > p->n || batch < 1 || batch > 65535 || grad_kind < 0 || grad_kind > 2)
    return fail(SLOS_EINVAL, "bad argument");
  if (grad_kind != 0 && layer != p->n) return fail(SLOS_EINVAL, "probabilities are those of the last layer");
  ReduceArgs ra{};
  std::vector<size_t> at;
  size_t total = 0;
  int rc = saved_layout(p, batch, layer, &at, &total);
  if (rc) return rc;
  if (saved_bytes < total) return fail(SLOS_ENOMEM, "buffer of the layers too small");
  BackLayout b;
  rc = back_layout(p, batch, layer, grad_kind != 0, &b);
  if (rc) return rc;
  if (ws_bytes < b.total) return fail(SLOS_ENOMEM, "workspace too small");
  for (int k = 0; k < layer; ++k) {
    ra.col[k] = modes ? modes[k] : p->modes[k];
    if (ra.col[k] < 0 || ra.col[k] >= p->m) return fail(SLOS_EINVAL, "input mode out of range");
    ra.part[k] = b.part[k] / sizeof(double2);
    ra.nblk[k] = (uint32_t)b.L[k].nblk;
  }
  ra.layers = layer;
  DevTables dt;
  rc = device_tables(p, &dt);
  if (rc) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const RoctxRange whole("slos_backward");
  const auto* Uf = static_cast<const float2*>(U);
  auto* base = static_cast<unsigned char*>(ws);
  auto psi = [&](int k) { return reinterpret_cast<const float2*>(static_cast<const unsigned char*>(saved) + at[k]); };
  const auto* gk = static_cast<const float2*>(grad);
  int next = 0;
  if (grad_kind != 0) {
    auto* g = reinterpret_cast<float2*>(base + b.g[0]);
    const auto* gp = static_cast<const float*>(grad);
    if (grad_kind == 1) {  // the amplitudes again, with the readout's adjoint in the same pass
      rc = launch_layer(p, dt, layer, ra.col[layer - 1], Uf, slos::packed_stride(p->m), batch, psi(layer - 1), p->size(layer - 1), g, p->size(layer), 4,
                        (float)(scale * scale), 0u, st, false, false, gp);
    } else {
      rc = run_readout_pull(p, dt, Uf, batch, ra.col[layer - 1], psi(layer - 1), gp, scale, g, st);
    }
    if (rc) return rc;
    gk = g;
    next = 1;
  }
  for (int k = layer; k >= 1; --k) {
    auto* gout = k > 1 ? reinterpret_cast<float2*>(base + b.g[next]) : nullptr;
    rc = run_adjoint(p, dt, b.L[k - 1], Uf, batch, k, ra.col[k - 1], psi(k - 1), gk, gout,
                     reinterpret_cast<double2*>(base + b.part[k - 1]), st);
    if (rc) return rc;
    gk = gout;
    next ^= 1;
  }
  const int threads = (int64_t)p->m * batch > 1024 ? kReduceManyThreads : kReduceAllThreads;
  hipLaunchKernelGGL(k_reduce_all, dim3((unsigned)p->m, (unsigned)batch), dim3((unsigned)threads), 0, st, ra,
                     reinterpret_cast<const double2*>(base), p->me, p->m, static_cast<float2*>(grad_U));
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

namespace {

// Whether a descent of `batch` rows with prefixes of dp positions takes the insert-table kernel. Its
// waves spend a fixed part of their time on each block, and on a small layer their blocks run one
// after another: with few parents a block the thread-per-state kernel is the faster one. Descents, us,
// walk / thread per state: blocks of 296 parents on average, 203k in all, 25 / 25; of 324, 32k in all,
// 18 / 23; of 189, 76k in all, 29 / 24; of 133, 7.7M in all, 179 / 387; of 34, 4.6M in all, 134 / 186;
// of 24, 7.8M in all, 300 / 312; of 56, 705k in all, 53 / 44; of 10, 1.1M in all, 110 / 58.
bool insert_walk(const slos_plan* p, int dp, uint64_t Sp, int64_t batch) {
  const int X = slos::insert_from(p->me);
  const uint64_t blocks = dp == 0 ? 1 : (X ? p->cg[(size_t)dp * (p->me + 1) + (p->me - X)] : 0) + p->size(dp - 1);
  return Sp / blocks >= 256 || (Sp / blocks >= 32 && Sp >= (1ull << 20) / (uint64_t)batch);
}

// Parents per wave of the insert-table kernels: few, so that the waves in flight read near one
// another (descents, us, with 64 / 128 / 256 / 512: 0.66M parents 17.5 / 20.0 / 21.6 / 27.9, 2.0M 39 / 41 / 40 / 41, 7.9M
// 127 / 111 / 108 / 135, 28M 492 / 383 / 383 / 445, 62M 1212 / 1042 / 1096 / 1203, 93M 1699 / 1257 / 1168 / 1258, 1.1G 23400 /
// 18900 / 18900 / 19900).
uint64_t insert_per_wave(uint64_t Sp) { return Sp < (1ull << 22) ? 64 : Sp < (1ull << 24) ? 128 : 256; }

}  // namespace

namespace {

// one step of the loss recurrence
int run_descend(const slos_plan* p, const DevTables& dt, int k, const float* q_k, float* q_km1, int64_t batch,
                unsigned flags, double scale, hipStream_t st) {
  const uint64_t Sp = p->size(k - 1), Sk = p->size(k);
  const int dp = k - 1 - slos::kSuf;
  char name[32];
  std::snprintf(name, sizeof name, "slos descent %d", k);
  const RoctxRange range(name);
  if (!(flags & SLOS_FLAG_SIMPLE) && p->multiset && dt.tuples && dp >= 0 && dp <= 8) {
    const uint64_t S_pre = p->size(dp);
    const uint32_t* ins = nullptr;
    const int rc = insert_table(p, st, &ins);
    if (rc) return rc;
    if (ins) {
      if (insert_walk(p, dp, Sp, batch)) {
        const uint64_t pw = insert_per_wave(Sp);
        const uint64_t wgs = ((Sp + pw - 1) / pw + slos::kWaves - 1) / slos::kWaves;
        if (wgs > 0x7fffffffull) return fail(SLOS_ERANGE, "layer too large for one launch");
        const slos::BlockGrid bg{dim3((unsigned)wgs, (unsigned)batch), 0, st, dt.cg, dt.lo, dt.tuples, p->me, p->multiset};
        const uint32_t xc = (uint32_t)((1ull << 16) / ((uint64_t)slos::kWaves * pw));
        slos::launch_descend_insert(dp, bg, q_k, Sk, q_km1, Sp, pw, (float)scale, xc, ins);
        HIP_TRY(hipGetLastError());
        return SLOS_OK;
      }
    } else if (dp >= 1) {
      const int maxd = dp <= 4 ? 4 : dp <= 6 ? 6 : 8;
      const size_t shb = slos::desc_dyn_lds(k, p->me, maxd);
      if (shb <= lds_limit()) {
        // more than 41 modes, or no table yet. Parents per wave: 1024 on layers of 2^27 parents or more, 512 below,
        // fewer on small layers; XCD chunks of 2^16 parents
        uint64_t pw = (Sp / 16384 + 63) & ~63ull;
        pw = std::min<uint64_t>(std::max<uint64_t>(pw, 256), Sp >= (1ull << 27) ? 1024 : 512);
        const uint64_t wgs = ((Sp + pw - 1) / pw + slos::kWaves - 1) / slos::kWaves;
        if (wgs > 0x7fffffffull) return fail(SLOS_ERANGE, "layer too large for one launch");
        const uint32_t xc = (uint32_t)std::max<uint64_t>(1, (1ull << 16) / ((uint64_t)slos::kWaves * pw));
        const slos::BlockGrid bg{dim3((unsigned)wgs, (unsigned)batch), shb, st, dt.cg, dt.lo, dt.tuples, p->me, p->multiset};
        slos::launch_descend_block(maxd, bg, k, q_k, Sk, q_km1, Sp, S_pre, pw, (float)scale, xc);
        HIP_TRY(hipGetLastError());
        return SLOS_OK;
      }
    }
  }
  const size_t sh = (size_t)(k + 1) * (p->me + 1) * 8 + (size_t)p->me * 4;
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  dim3 grid((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((Sp + 255) / 256, 1u << 20)), (unsigned)batch);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), sh, st, dt.cg, dt.lo, p->me, p->multiset, k, q_k, Sk, q_km1, Sp, batch,
                       (float)scale);
  };
  // Known photons and 32-bit ranks, as the forward's thread kernel, with the gathers of every mode in turn (children_sum): the
  // step 5 -> 4 at 24 modes 14 -> 6 us. In a set mask most modes take no photon where many are taken, and the walk
  // over the admissible ones is shorter from 6 parent photons on (sparse_1in4: 5): us, walk / every mode, 6 -> 5 at 26 modes
  // 18 / 14, at 40 54 / 52, 7 -> 6 at 26 modes 19 / 23, 8 -> 7 35 / 51, 9 -> 8 75 / 116, at 40 5195 / 6388; sparse_1in4, 36
  // modes, 5 -> 4 16.5 / 16.0, 6 -> 5 15.8 / 18.5, 9 -> 8 19 / 59.
  const int every = p->multiset ? 8 : p->shift == 2 ? 4 : 5;
  switch (Sk < (1ull << 32) && k - 1 <= every ? k - 1 : 0) {
    case 1: launch(k_descend<1, slos::SpaceView32, true>); break;
    case 2: launch(k_descend<2, slos::SpaceView32, true>); break;
    case 3: launch(k_descend<3, slos::SpaceView32, true>); break;
    case 4: launch(k_descend<4, slos::SpaceView32, true>); break;
    case 5: launch(k_descend<5, slos::SpaceView32, true>); break;
    case 6: launch(k_descend<6, slos::SpaceView32, true>); break;
    case 7: launch(k_descend<7, slos::SpaceView32, true>); break;
    case 8: launch(k_descend<8, slos::SpaceView32, true>); break;
    default: with_km(k - 1, [&](auto km) { launch(k_descend<decltype(km)::value>); }); break;
  }
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

// The layer k from which one launch takes every step down (descend_tail.hpp), or 0: with more rows than CUs its work
// groups of 1,024 threads take turns, and a launch a step is the shorter way (us, so / a launch a step: n = 5, m = 9, 1
// row 18 / 28, 256 19 / 29, 512 30 / 29, 2048 102 / 33, 20000 958 / 136; n = 6, m = 12, 256 40 / 44, 512 66 / 59).
int tail_top(const slos_plan* p, int64_t batch) {
  if (batch > 256) return 0;
  int top = 0;
  for (int k = 1; k <= std::min(p->n, slos::kTailTop); ++k) {
    const uint64_t Sp = p->size(k - 1);
    if (Sp > slos::kTailStates || Sp * (uint64_t)p->me > slos::kTailEdges || p->size(k) >= (1ull << 31)) break;
    top = k;
  }
  return slos::tail_lds(top, p->me) <= lds_limit() ? top : 0;
}

}  // namespace

int slos_loss_descend(const slos_plan* p, int k, const float* q_k, float* q_km1, int64_t batch, unsigned flags,
                      double scale, slos_stream_t stream) {
  if (!p || !q_k || !q_km1) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 1 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  if (batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
  DevTables dt;
  const int rc = device_tables(p, &dt);
  if (rc) return rc;
  return run_descend(p, dt, k, q_k, q_km1, batch, flags, scale, reinterpret_cast<hipStream_t>(stream));
}

int slos_loss_thin(const slos_plan* p, const float* q, float* const* out, const double* scale, int64_t batch,
                   slos_stream_t stream) {
  if (!p || !q || !scale || (p->n > 0 && !out)) return fail(SLOS_EINVAL, "NULL argument");
  if (batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
  for (int k = 0; k < p->n; ++k)
    if (!out[k]) return fail(SLOS_EINVAL, "NULL argument");
  DevTables dt;
  int rc = device_tables(p, &dt);
  if (rc) return rc;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int top = tail_top(p, batch);
  for (int k = p->n; k > top; --k) {
    rc = run_descend(p, dt, k, k == p->n ? q : out[k], out[k - 1], batch, 0u, scale[k - 1], st);
    if (rc) return rc;
  }
  if (top) {
    const RoctxRange range("slos last descents");
    slos::TailArgs a{};
    a.cg = dt.cg; a.lo = dt.lo; a.tuples = dt.tuples; a.me = p->me; a.multiset = p->multiset; a.top = top;
    a.q = top == p->n ? q : out[top];
    for (int k = 0; k <= top; ++k) a.S[k] = (uint32_t)p->size(k);
    for (int k = 0; k < top; ++k) {
      a.out[k] = out[k];
      a.scale[k] = (float)scale[k];
    }
    slos::launch_descend_tail(dim3(1, (unsigned)batch), slos::tail_lds(top, p->me), st, a);
    HIP_TRY(hipGetLastError());
  }
  return SLOS_OK;
}

namespace {

constexpr uint64_t kXRows = 1u << 20;  // rows of all levels together

bool xmodel_rows(int n, int levels, XRows* x) {
  std::vector<uint32_t> level{0u};
  uint64_t total = 0;
  for (int L = 0; L <= levels; ++L) {
    total += level.size();
    if (total > kXRows) return false;
    x->rows.push_back(level.size());
    x->most = std::max<uint64_t>(x->most, level.size());
    x->at.push_back(x->words.size());
    x->words.insert(x->words.end(), level.begin(), level.end());
    x->off.push_back(x->words.size());
    std::vector<uint32_t> next;
    for (const uint32_t t : level) {
      x->words.push_back((uint32_t)next.size());
      const int first = t ? __builtin_ctz(t) : n;
      for (int j = 0; j < first; ++j) next.push_back(t | (1u << j));
      if (next.size() > kXRows) return false;
    }
    x->words.push_back((uint32_t)next.size());
    level.swap(next);
  }
  x->zeros = x->words.size();
  x->words.insert(x->words.end(), x->most + 1, 0u);
  return true;
}

// the plan's rows of the levels 0..levels (null: more than kXRows)
const XRows* xmodel_host_rows(const slos_plan* cp, int levels) {
  slos_plan* p = const_cast<slos_plan*>(cp);
  std::lock_guard<std::mutex> g(p->mu);
  if (!p->xrows[levels]) {
    auto x = std::make_unique<XRows>();
    if (!xmodel_rows(p->n, levels, x.get())) return nullptr;
    p->xrows[levels] = std::move(x);
  }
  return p->xrows[levels].get();
}

// the same on the current GPU
int xmodel_tables(const slos_plan* cp, int levels, const XRows& x, hipStream_t st, const uint32_t** out) {
  slos_plan* p = const_cast<slos_plan*>(cp);
  int d = 0;
  HIP_TRY(hipGetDevice(&d));
  std::lock_guard<std::mutex> g(p->mu);
  for (auto& t : p->dev)
    if (t.device == d) {
      if (!t.xm[levels]) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        HIP_TRY(hipStreamIsCapturing(st, &cap));
        if (cap != hipStreamCaptureStatusNone)
          return fail(SLOS_EINVAL, "the plan's first x-model call cannot be captured: run it once before");
        uint32_t* dev = nullptr;
        const BesideCaptures guard;
        HIP_TRY(hipMalloc(&dev, x.words.size() * sizeof(uint32_t)));
        hipError_t e = hipMemcpyAsync(dev, x.words.data(), x.words.size() * sizeof(uint32_t), hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);  // other streams may read it from here on
        if (e != hipSuccess) {
          (void)hipFree(dev);
          HIP_TRY(e);
        }
        t.xm[levels] = dev;
      }
      *out = t.xm[levels];
      return SLOS_OK;
    }
  return fail(SLOS_EINVAL, "no device tables");
}

struct XLayout {
  const XRows* rows = nullptr;
  int levels = 0;                 // the most distinguishable photons beside at least two interfering ones
  size_t A[2] = {0, 0}, chain[2] = {0, 0}, scale = 0, one = 0, up = 0, fwd = 0, total = 0;
  std::vector<uint32_t> chunk;    // rows of one forward, per level
};

int xmodel_layout(const slos_plan* p, int64_t B, int order, unsigned flags, XLayout* x) {
  const int n = p->n;
  if (n < 3 || n > slos::kRaisePhotons || order < 1 || order > n || B < 1 || B > 65535)
    return fail(SLOS_EINVAL, "bad argument");
  // (a subset's photons are laid out as the columns of an m x m matrix)
  if (n > p->m) return fail(SLOS_EINVAL, "more photons than modes");
  x->levels = std::min(order, n - 2);
  x->rows = xmodel_host_rows(p, x->levels);
  if (!x->rows) return fail(SLOS_ERANGE, "too many subsets");
  uint64_t A[2] = {0, 0}, up = 0, fwd = 0;
  for (int L = 0; L <= x->levels; ++L) {
    const uint64_t R = x->rows->rows[L];
    uint64_t bytes;
    if (mul_overflow(p->size(n - L), R * (uint64_t)B * sizeof(float), &bytes) || bytes > (1ull << 62))
      return fail(SLOS_ERANGE, "layer sizes overflow");
    if (L) A[L & 1] = std::max(A[L & 1], bytes);
    WsLayout w;
    const int rc = forward_layout(p, B, n - L, &w, (flags & SLOS_FLAG_COMPENSATED) != 0, false);
    if (rc) return rc;
    const uint64_t row = w.total + (uint64_t)B * p->m * p->m * sizeof(float2);
    const uint64_t fit = std::min<uint64_t>({R, 65535u / (uint64_t)B, (1ull << 30) / row});
    x->chunk.push_back((uint32_t)std::max<uint64_t>(1, fit));
    WsLayout wc;
    const int rc2 = forward_layout(p, B * (int64_t)x->chunk[L], n - L, &wc, (flags & SLOS_FLAG_COMPENSATED) != 0, false);
    if (rc2) return rc2;
    fwd = std::max<uint64_t>(fwd, wc.total);
    up = std::max<uint64_t>(up, (uint64_t)x->chunk[L] * (uint64_t)B * p->m * p->m * sizeof(float2));
  }
  size_t sum = 0;
  auto take = [&](size_t* at, uint64_t bytes) {
    *at = sum;
    sum += align256((size_t)bytes);
  };
  take(&x->A[0], A[0]);
  take(&x->A[1], A[1]);
  take(&x->chain[0], (uint64_t)B * sizeof(float));
  take(&x->chain[1], (uint64_t)B * p->size(1) * sizeof(float));
  take(&x->scale, x->rows->most * sizeof(float));
  take(&x->one, sizeof(float));
  take(&x->up, up);
  take(&x->fwd, fwd);
  x->total = sum;
  return SLOS_OK;
}

}  // namespace

int slos_xmodel_workspace(const slos_plan* p, int64_t batch, int order, unsigned flags, size_t* bytes) {
  if (!p || !bytes) return fail(SLOS_EINVAL, "NULL argument");
  XLayout x;
  const int rc = xmodel_layout(p, batch, order, flags, &x);
  *bytes = x.total;
  return rc;
}

int slos_xmodel(const slos_plan* p, const void* U, int64_t batch, int order, const float* weights, int weights_on_device,
                float* out, unsigned flags, void* ws, size_t ws_bytes, slos_stream_t stream) {
  if (!p || !U || !weights || !out || !ws) return fail(SLOS_EINVAL, "NULL argument");
  if (flags & ~(unsigned)SLOS_FLAG_COMPENSATED) return fail(SLOS_EINVAL, "unsupported flag");
  XLayout x;
  int rc = xmodel_layout(p, batch, order, flags, &x);
  if (rc) return rc;
  if (ws_bytes < x.total) return fail(SLOS_ENOMEM, "workspace too small");
  DevTables dt;
  rc = device_tables(p, &dt);
  if (rc) return rc;
  const uint32_t* tab = nullptr;
  rc = xmodel_tables(p, x.levels, *x.rows, reinterpret_cast<hipStream_t>(stream), &tab);
  if (rc) return rc;
  const int n = p->n;
  const int B = (int)batch;
  int photons[kMaxPhotons];  // their columns, in order (k_subset_columns counts equal ones next to each other)
  std::copy(p->modes.begin(), p->modes.end(), photons);
  std::sort(photons, photons + n);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const RoctxRange whole("slos_xmodel");
  auto* base = static_cast<unsigned char*>(ws);
  auto* scale = reinterpret_cast<float*>(base + x.scale);
  auto* one = reinterpret_cast<float*>(base + x.one);
  auto level = [&](int L) { return L ? reinterpret_cast<float*>(base + x.A[L & 1]) : out; };
  // the terms of L distinguishable photons: every subset's forward, and the rows' weights
  auto start = [&](int L) {
    const uint32_t R = (uint32_t)x.rows->rows[L];
    const int g = n - L;
    int cols[kMaxPhotons];
    for (int i = 0; i < g; ++i) cols[i] = i;
    for (uint32_t r0 = 0; r0 < R; r0 += x.chunk[L]) {
      slos::SubsetArgs a{};
      a.U = static_cast<const float2*>(U);
      a.Up = reinterpret_cast<float2*>(base + x.up);
      a.masks = tab + x.rows->at[L];
      a.r0 = r0;
      a.rows = std::min(x.chunk[L], R - r0);
      a.B = B; a.m = p->m; a.n = n; a.g = g;
      a.row_scale = scale;
      for (int j = 0; j < n; ++j) a.cols[j] = photons[j];
      slos::launch_subsets(st, a);
      HIP_TRY(hipGetLastError());
      const int64_t rows = (int64_t)a.rows * B;
      WsLayout w;
      int rc = forward_layout(p, rows, g, &w, (flags & SLOS_FLAG_COMPENSATED) != 0, false);
      if (rc) return rc;
      rc = forward_run(p, dt, a.Up, slos::packed_stride(p->m), rows, cols, g, SLOS_OUT_PROBS, level(L) + (size_t)r0 * B * p->size(g), 1.0, flags, w,
                       base + x.fwd, st);
      if (rc) return rc;
    }
    return (int)SLOS_OK;
  };
  // targets += their sources, raised (off: see RaiseArgs), the targets scaled
  auto raise = [&](int K, const float* q, float* to, uint32_t targets, const uint32_t* off, int photon, const float* row_scale,
                   int weight) {
    slos::RaiseArgs a{};
    a.cg = dt.cg; a.lo = dt.lo; a.words = dt.tuples5; a.me = p->me; a.multiset = p->multiset; a.m = p->m; a.K = K; a.B = B;
    a.S_par = p->size(K - 1); a.S = p->size(K);
    a.q = q; a.out = to; a.targets = targets; a.off = off; a.photon = photon; a.photons = off ? n : 1;
    a.row_scale = row_scale;
    if (weight < 0) a.weight_value = 1.f;
    else if (weights_on_device) a.weight = weights + weight;
    else a.weight_value = weights[weight];
    a.U = static_cast<const float2*>(U);
    for (int j = 0; j < n; ++j) a.cols[j] = photons[j];
    const size_t lds = slos::raise_lds(K, p->me, a.photons);
    if (lds > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
    const uint64_t wgs = std::min<uint64_t>((a.S + 255) / 256, 1u << 20);  // (a launch has at most 2^32 threads)
    // a work group takes all targets of its states where there are enough states: 2048 work groups fill
    // the chip
    const uint64_t parts = std::min<uint64_t>({targets, 65535u, (2048 + wgs * B - 1) / (wgs * B)});
    a.rows_per = (uint32_t)((targets + parts - 1) / parts);
    const unsigned z = (targets + a.rows_per - 1) / a.rows_per;
    slos::launch_raise(dim3((unsigned)wgs, (unsigned)B, z), lds, st, a);
    HIP_TRY(hipGetLastError());
    return (int)SLOS_OK;
  };
  const int top = x.levels;
  rc = start(top);
  if (rc) return rc;
  rc = raise(n - top, level(top), level(top), (uint32_t)x.rows->rows[top], tab + x.rows->zeros, 0, scale, top);
  if (rc) return rc;
  if (order >= n - 1) {
    // the terms with fewer than two interfering photons: photons 0 and 1 raised from the vacuum into
    // the set of the others
    auto* c0 = reinterpret_cast<float*>(base + x.chain[0]);
    auto* c1 = reinterpret_cast<float*>(base + x.chain[1]);
    slos::launch_chain_start(st, c0, B, one, weights_on_device ? weights + n + 1 : nullptr,
                             weights_on_device ? 0.f : weights[n + 1]);
    HIP_TRY(hipGetLastError());
    rc = raise(1, c0, c1, 1, nullptr, 0, nullptr, -1);
    if (rc) return rc;
    const uint32_t others = ((1u << n) - 1u) & ~3u;
    const uint32_t* masks = x.rows->words.data() + x.rows->at[top];
    const size_t row = std::find(masks, masks + x.rows->rows[top], others) - masks;
    rc = raise(2, c1, level(top) + row * B * p->size(2), 1, nullptr, 1, one, -1);
    if (rc) return rc;
  }
  for (int L = top; L >= 1; --L) {
    rc = start(L - 1);
    if (rc) return rc;
    rc = raise(n - L + 1, level(L), level(L - 1), (uint32_t)x.rows->rows[L - 1], tab + x.rows->off[L - 1], 0, scale, L - 1);
    if (rc) return rc;
  }
  return SLOS_OK;
}

int slos_raise(const slos_plan* p, int k, const float* w, const float* q_km1, float* q_k, int64_t batch,
               slos_stream_t stream) {
  if (!p || !w || !q_km1 || !q_k) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 1 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  if (batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
  DevTables dt;
  int rc = device_tables(p, &dt);
  if (rc) return rc;
  const uint64_t Sp = p->size(k - 1), Sk = p->size(k);
  const size_t sh = (size_t)(k + 1) * (p->me + 1) * 8 + (size_t)p->me * 4 + (size_t)p->m * 4;
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  dim3 grid((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((Sk + 255) / 256, 1u << 20)), (unsigned)batch);
  with_km(k, [&](auto km) {
    hipLaunchKernelGGL((k_raise<decltype(km)::value>), grid, dim3(256), sh, reinterpret_cast<hipStream_t>(stream),
                       dt.cg, dt.lo, p->me, p->multiset, k, p->m, w, q_km1, Sp, q_k, Sk, batch);
  });
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

int slos_loss_ascend(const slos_plan* p, int k, const float* g_km1, float* g_k, int64_t batch, slos_stream_t stream) {
  if (!p || !g_km1 || !g_k) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 1 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  if (batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
  DevTables dt;
  int rc = device_tables(p, &dt);
  if (rc) return rc;
  const uint64_t Sp = p->size(k - 1), Sk = p->size(k);
  const size_t sh = (size_t)(k + 1) * (p->me + 1) * 8 + (size_t)p->me * 4;
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  dim3 grid((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((Sk + 255) / 256, 1u << 20)), (unsigned)batch);
  with_km(k, [&](auto km) {
    hipLaunchKernelGGL((k_ascend<decltype(km)::value>), grid, dim3(256), sh, reinterpret_cast<hipStream_t>(stream),
                       dt.cg, dt.lo, p->me, p->multiset, k, g_km1, Sp, g_k, Sk, batch);
  });
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

int slos_mass_workspace(int64_t batch, uint64_t count, size_t* bytes) {
  (void)count;
  if (!bytes || batch < 1) return fail(SLOS_EINVAL, "bad argument");
  *bytes = (size_t)batch * kMassBlocks * sizeof(double);
  return SLOS_OK;
}

int slos_total_mass(const float* probs, int64_t batch, uint64_t count, double* out, void* ws, size_t ws_bytes,
                    slos_stream_t stream) {
  if (!probs || !out || batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "bad argument");
  if (!ws || ws_bytes < (size_t)batch * kMassBlocks * sizeof(double)) return fail(SLOS_ENOMEM, "workspace too small");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  double* part = static_cast<double*>(ws);
  hipLaunchKernelGGL(k_mass_partial, dim3(kMassBlocks, (unsigned)batch), dim3(256), 0, st, probs, count, part);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_mass_final, dim3((unsigned)batch), dim3(256), 0, st, part, kMassBlocks, out);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}


int slos_group_sums(const float* probs, int64_t batch, uint64_t count, const int64_t* order, const int64_t* chunks,
                    uint32_t n_chunks, const uint32_t* first, int n_groups, float* out, void* ws, size_t ws_bytes,
                    slos_stream_t stream) {
  return group_sums(probs, batch, count, order, chunks, n_chunks, first, n_groups, out, ws, ws_bytes, stream);
}

int slos_group_sums_f64(const double* probs, int64_t batch, uint64_t count, const int64_t* order,
                        const int64_t* chunks, uint32_t n_chunks, const uint32_t* first, int n_groups, double* out,
                        void* ws, size_t ws_bytes, slos_stream_t stream) {
  return group_sums(probs, batch, count, order, chunks, n_chunks, first, n_groups, out, ws, ws_bytes, stream);
}

int slos_spot_probs(const slos_plan* p, const void* U, const uint64_t* idx, int64_t count, double* out,
                    slos_stream_t stream) {
  if (!p || !U || (!idx && count) || (!out && count)) return fail(SLOS_EINVAL, "NULL argument");
  if (p->n > 24) return fail(SLOS_ERANGE, "spot permanents support n <= 24");
  if (count == 0) return SLOS_OK;
  DevTables dt;
  int rc = device_tables(p, &dt);
  if (rc) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_spot_ryser, dim3((unsigned)((count + 63) / 64)), dim3(64), 0, st, dt.cg, dt.lo, p->me, p->n,
                     p->m, static_cast<const double2*>(U), dt.modes, p->s_fact, p->multiset, idx, count, out);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

int slos_sample_workspace(uint64_t count, size_t* bytes) {
  if (!bytes) return fail(SLOS_EINVAL, "NULL argument");
  if (count < 1) return fail(SLOS_EINVAL, "count must be >= 1");
  const uint64_t nb = (count + kSampleBlock - 1) / kSampleBlock;
  if (nb > (uint64_t)kSampleSeg * 1024) return fail(SLOS_ERANGE, "too many categories for the sampler");
  // block sums, the cdf, the chunk sums and the segment totals
  *bytes = 2 * align256(nb * sizeof(double)) + align256(nb * 64 * sizeof(double)) + align256(1024 * sizeof(double));
  return SLOS_OK;
}

int slos_sample(const float* probs, uint64_t count, const double* uniforms, int64_t shots, uint64_t* idx, void* ws,
                size_t ws_bytes, slos_stream_t stream) {
  if (shots < 0) return fail(SLOS_EINVAL, "shots must be >= 0");
  if (!probs || (shots > 0 && (!uniforms || !idx))) return fail(SLOS_EINVAL, "NULL argument");
  size_t need = 0;
  int rc = slos_sample_workspace(count, &need);
  if (rc) return rc;
  if (!ws || ws_bytes < need) return fail(SLOS_ENOMEM, "workspace too small: need " + std::to_string(need) + " bytes");
  if (shots == 0) return SLOS_OK;
  const uint64_t nb = (count + kSampleBlock - 1) / kSampleBlock;
  double* bsum = static_cast<double*>(ws);
  double* cdf = reinterpret_cast<double*>(static_cast<unsigned char*>(ws) + align256(nb * sizeof(double)));
  double* csum = reinterpret_cast<double*>(static_cast<unsigned char*>(ws) + 2 * align256(nb * sizeof(double)));
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_sample_block_sums, dim3((unsigned)((nb + kSumWaves - 1) / kSumWaves)), dim3(64 * kSumWaves), 0, st,
                     probs, count, nb, bsum, csum);
  HIP_TRY(hipGetLastError());
  double* segtot = reinterpret_cast<double*>(static_cast<unsigned char*>(ws) + 2 * align256(nb * sizeof(double)) +
                                             align256(nb * 64 * sizeof(double)));
  const uint64_t nseg = (nb + kSampleSeg - 1) / kSampleSeg;  // <= 1024 (slos_sample_workspace)
  hipLaunchKernelGGL(k_sample_seg_prefix, dim3((unsigned)nseg), dim3(256), 0, st, bsum, nb, cdf, segtot);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_sample_seg_offsets, dim3(1), dim3(64), 0, st, segtot, (int)nseg);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_sample_add_offsets, dim3((unsigned)std::min<uint64_t>((nb + 255) / 256, 4096)), dim3(256), 0, st,
                     cdf, nb, segtot);
  HIP_TRY(hipGetLastError());
  const uint64_t g = ((uint64_t)shots + 255) / 256;
  if (g > 0x7fffffffull) return fail(SLOS_ERANGE, "too many shots for one launch");
  hipLaunchKernelGGL(k_sample_search, dim3((unsigned)g), dim3(256), 0, st, probs, count, nb, cdf, csum, uniforms, shots,
                     idx);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

int slos_unrank_device(const slos_plan* p, int k, const uint64_t* idx, int64_t count, int32_t* occ,
                       slos_stream_t stream) {
  if (!p || !idx || !occ) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 0 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  if (count < 0) return fail(SLOS_EINVAL, "count must be >= 0");
  if (count == 0) return SLOS_OK;
  DevTables dt;
  int rc = device_tables(p, &dt);
  if (rc) return rc;
  const size_t sh = (size_t)(k + 1) * (p->me + 1) * 8 + (size_t)p->me * 4;
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  const uint64_t blocks = std::min<uint64_t>(((uint64_t)count + 255) / 256, 1u << 16);
  hipLaunchKernelGGL(k_unrank_occ, dim3((unsigned)blocks), dim3(256), sh, reinterpret_cast<hipStream_t>(stream), dt.cg,
                     dt.lo, p->me, k, p->m, idx, count, occ);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

int slos_group_create(int count, const slos_plan* const* plans, slos_group** out) {
  if (!out || !plans) return fail(SLOS_EINVAL, "NULL argument");
  *out = nullptr;
  if (count < 1 || count > slos::kMaxGroup)
    return fail(SLOS_EINVAL, "a group holds 1 to " + std::to_string(slos::kMaxGroup) + " plans");
  auto* G = new slos_group();
  for (int g = 0; g < count; ++g) {
    const slos_plan* p = plans[g];
    if (!p) {
      delete G;
      return fail(SLOS_EINVAL, "NULL plan");
    }
    if (simple_lds_bytes(p->n, p->me, p->m) > lds_limit()) {
      delete G;
      return fail(SLOS_ERANGE, "plan too large for a group launch (LDS)");
    }
    G->plans.push_back(p);
    G->nmax = std::max(G->nmax, p->n);
  }
  G->cfg.assign(G->nmax + 1, slos_group::Cfg());
  *out = G;
  return SLOS_OK;
}

int slos_group_destroy(slos_group* G) {
  if (!G) return SLOS_OK;
  group_drop_graph(G);
  if (G->cap) (void)hipStreamDestroy(G->cap);
  delete G;
  return SLOS_OK;
}

int slos_group_workspace(const slos_group* G, const int64_t* batch, unsigned flags, size_t* bytes) {
  if (!G || !batch || !bytes) return fail(SLOS_EINVAL, "NULL argument");
  GroupWs w;
  int rc = group_layout(G, batch, &w, (flags & SLOS_FLAG_COMPENSATED) != 0);
  if (rc) return rc;
  *bytes = w.total;
  return SLOS_OK;
}

int slos_group_forward(slos_group* G, const void* const* U, const int64_t* batch, float* const* out,
                       const double* scale, unsigned flags, void* ws, size_t ws_bytes, slos_stream_t stream) {
  GroupArgs a;
  GroupWs w;
  int rc = group_args(G, U, batch, out, scale, flags, ws, ws_bytes, &a, &w);
  if (rc) return rc;
  std::vector<DevTables> dts;
  rc = group_tables(G, &dts);
  if (rc) return rc;
  return group_forward(G, a, w, dts, reinterpret_cast<hipStream_t>(stream));
}

int slos_group_tune(slos_group* G, const void* const* U, const int64_t* batch, float* const* out,
                    const double* scale, unsigned flags, void* ws, size_t ws_bytes, int reps, slos_stream_t stream) {
  GroupArgs a;
  GroupWs w;
  int rc = group_args(G, U, batch, out, scale, flags, ws, ws_bytes, &a, &w);
  if (rc) return rc;
  if (reps < 1) return fail(SLOS_EINVAL, "reps must be >= 1");
  std::vector<DevTables> dts;
  rc = group_tables(G, &dts);
  if (rc) return rc;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  int dev = 0, ncu = 0;
  HIP_TRY(hipGetDevice(&dev));
  HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  group_drop_graph(G);
  std::fill(G->cfg.begin(), G->cfg.end(), slos_group::Cfg());
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  // layers in order: each candidate rewrites layer K from the (already final) layer K - 1
  rc = group_forward(G, a, w, dts, st);
  for (int K = 1; K <= G->nmax && rc == SLOS_OK; ++K) {
    std::vector<slos_group::Cfg> cand;
    const uint32_t grids[4] = {0, (uint32_t)ncu * 2, (uint32_t)ncu * 4, (uint32_t)ncu * 8};
    if (group_can_block(G, dts, K, flags))
      for (uint64_t pw : {256, 512, 1024, 2048, 4096})
        for (uint32_t gr : grids) cand.push_back({1, pw, gr});
    for (uint64_t spt : {1, 2, 4})
      for (uint32_t gr : grids) cand.push_back({0, spt, gr});
    cand.push_back({2, 0, 0});  // one single-plan launch per plan
    float best = 1e30f;
    slos_group::Cfg pick;
    for (const auto& c : cand) {
      rc = group_layer(G, K, a, w, dts, c, st);  // warm-up
      if (rc) break;
      if ((rc = (hipEventRecord(e0, st) == hipSuccess ? SLOS_OK : fail(SLOS_EHIP, "hipEventRecord")))) break;
      for (int r = 0; r < reps && rc == SLOS_OK; ++r) rc = group_layer(G, K, a, w, dts, c, st);
      if (rc) break;
      float ms = 0.f;
      if (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
          hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
        rc = fail(SLOS_EHIP, "event timing failed");
        break;
      }
      if (ms < best) {
        best = ms;
        pick = c;
      }
    }
    G->cfg[K] = pick;
    // leave layer K final under the chosen launch (all candidates compute the same values)
    if (rc == SLOS_OK) rc = group_layer(G, K, a, w, dts, pick, st);
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}

int slos_group_config(const slos_group* G, int K, int* block, uint64_t* per_wave, uint32_t* grid) {
  if (!G || !block || !per_wave || !grid) return fail(SLOS_EINVAL, "NULL argument");
  if (K < 1 || K > G->nmax) return fail(SLOS_EINVAL, "layer out of range");
  *block = G->cfg[K].block;
  *per_wave = G->cfg[K].per_wave;
  *grid = G->cfg[K].grid;
  return SLOS_OK;
}

int slos_group_capture(slos_group* G, const void* const* U, const int64_t* batch, float* const* out,
                       const double* scale, unsigned flags, void* ws, size_t ws_bytes) {
  GroupArgs a;
  GroupWs w;
  int rc = group_args(G, U, batch, out, scale, flags, ws, ws_bytes, &a, &w);
  if (rc) return rc;
  std::vector<DevTables> dts;
  rc = group_tables(G, &dts);  // device tables exist before capture: nothing is allocated inside it
  if (rc) return rc;
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  if (G->cap && G->cap_device != dev) {
    (void)hipStreamDestroy(G->cap);
    G->cap = nullptr;
  }
  if (!G->cap) {
    HIP_TRY(hipStreamCreateWithFlags(&G->cap, hipStreamNonBlocking));
    G->cap_device = dev;
  }
  group_drop_graph(G);
  HIP_TRY(hipStreamBeginCapture(G->cap, hipStreamCaptureModeThreadLocal));
  rc = group_forward(G, a, w, dts, G->cap);
  hipGraph_t graph = nullptr;
  const hipError_t ec = hipStreamEndCapture(G->cap, &graph);
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (ec != hipSuccess) return fail(SLOS_EHIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(ec));
  G->graph = graph;
  HIP_TRY(hipGraphInstantiate(&G->exec, G->graph, nullptr, nullptr, 0));
  return SLOS_OK;
}

int slos_group_replay(slos_group* G, slos_stream_t stream) {
  if (!G) return fail(SLOS_EINVAL, "NULL argument");
  if (!G->exec) return fail(SLOS_EINVAL, "no captured forward: call slos_group_capture first");
  HIP_TRY(hipGraphLaunch(G->exec, reinterpret_cast<hipStream_t>(stream)));
  return SLOS_OK;
}

}  // extern "C"

// ------------------------------------------------------------------------------------------
// complex128 / float64 twins of the entry points that take typed pointers or no flags
// (FockSLOSKernel(dtype=torch.complex128)); thread-per-state FP64 kernels of layer_f64.hpp
// ------------------------------------------------------------------------------------------

namespace {

// plan tables on the device, the batch range and the layer range shared by the twins below
int f64_common(const slos_plan* p, int k, int64_t batch, DevTables* dt) {
  if (k < 1 || k > p->n) return fail(SLOS_EINVAL, "layer out of range");
  if (batch < 1 || batch > 65535) return fail(SLOS_EINVAL, "batch must be in [1, 65535]");
  return device_tables(p, dt);
}

// work groups and dynamic LDS of k_adjoint_layer_f64 for layer k
int adjoint_launch_f64(const slos_plan* p, int k, size_t* lds, uint64_t* nblk) {
  *lds = slos::space_lds_f64(k, p->me) + (size_t)p->m * 16 + (size_t)slos::kAdjThreadsF64 * p->me * 16;
  if (*lds > lds_limit()) return fail(SLOS_ERANGE, "adjoint LDS exceeds the GPU's LDS (too many modes)");
  *nblk = (uint64_t)adjoint_blocks(p->size(k - 1));
  return SLOS_OK;
}

}  // namespace

int slos_loss_descend_f64(const slos_plan* p, int k, const double* q_k, double* q_km1, int64_t batch, double scale,
                          slos_stream_t stream) {
  if (!p || !q_k || !q_km1) return fail(SLOS_EINVAL, "NULL argument");
  DevTables dt;
  int rc = f64_common(p, k, batch, &dt);
  if (rc) return rc;
  const uint64_t Sp = p->size(k - 1), Sk = p->size(k);
  const size_t sh = slos::space_lds_f64(k, p->me);
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  char name[32];
  std::snprintf(name, sizeof name, "slos descent %d", k);
  const RoctxRange range(name);
  dim3 grid((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((Sp + 255) / 256, 1u << 20)), (unsigned)batch);
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define SLOS_F64D(KM) \
  hipLaunchKernelGGL((slos::k_descend_f64<KM>), grid, dim3(256), sh, st, dt.cg, dt.lo, p->me, p->multiset, k, q_k, Sk, \
                     q_km1, Sp, batch, scale)
  if (k - 1 <= 8) { SLOS_F64D(8); }
  else if (k - 1 <= 16) { SLOS_F64D(16); }
  else { SLOS_F64D(32); }
#undef SLOS_F64D
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

int slos_loss_ascend_f64(const slos_plan* p, int k, const double* g_km1, double* g_k, int64_t batch,
                         slos_stream_t stream) {
  if (!p || !g_km1 || !g_k) return fail(SLOS_EINVAL, "NULL argument");
  DevTables dt;
  int rc = f64_common(p, k, batch, &dt);
  if (rc) return rc;
  const uint64_t Sp = p->size(k - 1), Sk = p->size(k);
  const size_t sh = slos::space_lds_f64(k, p->me);
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  dim3 grid((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((Sk + 255) / 256, 1u << 20)), (unsigned)batch);
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define SLOS_F64A(KM)                                                                                                \
  hipLaunchKernelGGL((slos::k_ascend_f64<KM>), grid, dim3(256), sh, st, dt.cg, dt.lo, p->me, p->multiset, k, g_km1, Sp, \
                     g_k, Sk, batch)
  if (k <= 8) { SLOS_F64A(8); }
  else if (k <= 16) { SLOS_F64A(16); }
  else { SLOS_F64A(32); }
#undef SLOS_F64A
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

int slos_readout_adjoint_f64(const slos_plan* p, int64_t batch, const void* amps, const double* grad_p, double scale,
                             void* grad_amps, slos_stream_t stream) {
  if (!p || !amps || !grad_p || !grad_amps) return fail(SLOS_EINVAL, "NULL argument");
  if (p->n < 1) return fail(SLOS_EINVAL, "no photon: nothing depends on U");
  DevTables dt;
  int rc = f64_common(p, p->n, batch, &dt);
  if (rc) return rc;
  const uint64_t S = p->size(p->n);
  const size_t sh = slos::space_lds_f64(p->n, p->me);
  if (sh > lds_limit()) return fail(SLOS_ERANGE, "counting table does not fit LDS");
  dim3 grid((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((S + 255) / 256, 1u << 20)),
            (unsigned)std::min<int64_t>(batch, 16));
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define SLOS_F64R(KM)                                                                                                 \
  hipLaunchKernelGGL((slos::k_readout_adjoint_f64<KM>), grid, dim3(256), sh, st, dt.cg, dt.lo, p->me, p->multiset, p->n, \
                     static_cast<const double2*>(amps), grad_p, static_cast<double2*>(grad_amps), S, batch, scale * scale)
  if (p->n <= 8) { SLOS_F64R(8); }
  else if (p->n <= 16) { SLOS_F64R(16); }
  else { SLOS_F64R(32); }
#undef SLOS_F64R
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}

int slos_adjoint_workspace_f64(const slos_plan* p, int64_t batch, int k, size_t* bytes) {
  if (!p || !bytes) return fail(SLOS_EINVAL, "NULL argument");
  if (k < 1 || k > p->n || batch < 1) return fail(SLOS_EINVAL, "bad argument");
  size_t lds = 0;
  uint64_t nblk = 0;
  int rc = adjoint_launch_f64(p, k, &lds, &nblk);
  if (rc) return rc;
  *bytes = (size_t)batch * nblk * p->me * sizeof(double2);
  return SLOS_OK;
}

int slos_adjoint_layer_f64(const slos_plan* p, const void* U, int64_t batch, int k, int col, const void* psi_prev,
                           const void* grad_k, void* grad_prev, void* grad_U, int accumulate, void* ws,
                           size_t ws_bytes, slos_stream_t stream) {
  if (!p || !U || !psi_prev || !grad_k || !grad_U) return fail(SLOS_EINVAL, "NULL argument");
  if (col < 0 || col >= p->m) return fail(SLOS_EINVAL, "input mode out of range");
  DevTables dt;
  int rc = f64_common(p, k, batch, &dt);
  if (rc) return rc;
  size_t lds = 0;
  uint64_t nblk = 0;
  rc = adjoint_launch_f64(p, k, &lds, &nblk);
  if (rc) return rc;
  if (!ws || ws_bytes < (size_t)batch * nblk * p->me * sizeof(double2)) return fail(SLOS_ENOMEM, "workspace too small");
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define SLOS_F64J(KM)                                                                                              \
  hipLaunchKernelGGL((slos::k_adjoint_layer_f64<KM>), dim3((unsigned)nblk, (unsigned)batch), dim3(slos::kAdjThreadsF64), \
                     lds, st, dt.cg, dt.lo, p->me, p->multiset, k, p->m, col, static_cast<const double2*>(U),         \
                     static_cast<const double2*>(psi_prev), static_cast<const double2*>(grad_k), p->size(k),          \
                     static_cast<double2*>(grad_prev), p->size(k - 1), static_cast<double2*>(ws), grad_prev != nullptr)
  if (k - 1 <= 8) { SLOS_F64J(8); }
  else if (k - 1 <= 16) { SLOS_F64J(16); }
  else { SLOS_F64J(32); }
#undef SLOS_F64J
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(slos::k_reduce_gu_f64, dim3((unsigned)p->me, (unsigned)batch), dim3(64), 0, st,
                     static_cast<const double2*>(ws), (int)nblk, p->me, p->m, col, static_cast<double2*>(grad_U),
                     accumulate);
  HIP_TRY(hipGetLastError());
  return SLOS_OK;
}
