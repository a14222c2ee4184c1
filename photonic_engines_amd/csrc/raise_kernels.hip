// k_raise_rows, k_subset_columns and k_chain_start (raise.hpp).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "raise.hpp"

namespace slos {

// (a sum whose terms are rounded on their own: the layer-by-layer mixture adds tensors)
__device__ __forceinline__ float add_rounded(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

// |u|^2, every operation rounded
__device__ __forceinline__ float square_rounded(float2 u) {
#pragma clang fp contract(off)
  return u.x * u.x + u.y * u.y;
}

// One child a thread: its positions and its parents' ranks once, for all rows of the work group. A row
// costs a gather, an LDS weight and a multiply-add per parent and source; the gathers are 4 bytes a
// lane from one row, near one another. Bound by the cache's rate for them. A source's parents are summed
// in ascending position, then the sources in ascending order of their photon: the bits of the
// layer-by-layer mixture, whose complex layer steps computed every row's index again and whose rows were
// gathered, widened to complex and added by some 350 tensor operations: n = 8, m = 24, every order,
// 4710 -> 856 us.
template <int KM, class SV, bool EXACT>
__global__ __launch_bounds__(256) void k_raise_rows(RaiseArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef RankT<SV> R;
  const int K = EXACT ? KM : a.K;
  const int stride = a.me + 1;
  const int ncg = (K + 1) * stride;
  R* cg = reinterpret_cast<R*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  float* wl = reinterpret_cast<float*>(smem + ((ncg * 8 + a.me * 4 + 15) & ~15));  // [photons][me]
  const int b = blockIdx.y;
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = (R)a.cg[i];
  for (int i = threadIdx.x; i < a.me; i += blockDim.x) lo[i] = a.lo[i];
  for (int i = threadIdx.x; i < a.photons * a.me; i += blockDim.x) {
    const int j = i / a.me, x = i - j * a.me;
    const float2 u = a.U[(size_t)b * a.m * a.m + (size_t)x * a.m + a.cols[a.off ? j : a.photon]];
    wl[i] = square_rounded(u);
  }
  __syncthreads();
  const SV sv{cg, lo, a.me, stride};
  const float wt = a.weight ? *a.weight : a.weight_value;
  const uint32_t r0 = blockIdx.z * a.rows_per;
  const uint32_t r1 = r0 + a.rows_per < a.targets ? r0 + a.rows_per : a.targets;
  for (uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; c < a.S; c += (uint64_t)gridDim.x * blockDim.x) {
    int p[KM];
    unrank_words<KM>(sv, a.words, (R)c, K, p);
    R par[KM];      // the parent without position l
    bool real[KM];  // (a repeated position is no further parent)
    parent_ranks<KM>(sv, a.multiset, K, p, par, real);
    for (uint32_t r = r0; r < r1; ++r) {
      const uint32_t s0 = a.off ? a.off[r] : 0u, s1 = a.off ? a.off[r + 1] : 1u;
      float acc = 0.f;
#pragma unroll 2
      for (uint32_t s = s0; s < s1; ++s) {
        const float* q = a.q + ((size_t)s * a.B + b) * a.S_par;
        const float* w = wl + (size_t)(s - s0) * a.me;
        float v[KM];
#pragma unroll
        for (int l = 0; l < KM; ++l) v[l] = l < K ? q[par[l]] : 0.f;
        float sum = 0.f;
#pragma unroll
        for (int l = 0; l < KM; ++l)
          if (l < K) sum = fmaf(w[p[l]], real[l] ? v[l] : 0.f, sum);
        acc = add_rounded(acc, sum);
      }
      float* o = a.out + ((size_t)r * a.B + b) * a.S + c;
      *o = a.row_scale ? add_rounded((*o * a.row_scale[r]) * wt, acc) : acc;
    }
  }
}

__global__ __launch_bounds__(256) void k_subset_columns(SubsetArgs a) {
  const uint32_t row = blockIdx.x, b = blockIdx.y;
  const uint32_t mask = a.masks[a.r0 + row];
  __shared__ int cols[kRaisePhotons];
  if (threadIdx.x == 0) {
    double s = 1.0;
    int g = 0, run = 0, last = -1;
    for (int j = 0; j < a.n; ++j)
      if (!((mask >> j) & 1u)) {
        const int c = a.cols[j];
        run = c == last ? run + 1 : 1;  // the photons are in order of their columns
        last = c;
        s *= run;
        cols[g++] = c;
      }
    if (b == 0) a.row_scale[a.r0 + row] = (float)(1.0 / s);
  }
  __syncthreads();
  const float2* U = a.U + (size_t)b * a.m * a.m;
  float2* Up = a.Up + ((size_t)row * a.B + b) * a.m * a.m;
  for (int i = threadIdx.x; i < a.m * a.g; i += blockDim.x) {
    const int x = i / a.g, j = i - x * a.g;
    Up[(size_t)x * a.m + j] = U[(size_t)x * a.m + cols[j]];
  }
}

__global__ void k_chain_start(float* start, int B, float* one, const float* weight, float weight_value) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < B; i += gridDim.x * blockDim.x)
    start[i] = weight ? *weight : weight_value;
  if (blockIdx.x == 0 && threadIdx.x == 0) *one = 1.f;
}

void launch_chain_start(hipStream_t st, float* start, int B, float* one, const float* weight, float weight_value) {
  hipLaunchKernelGGL(k_chain_start, dim3((unsigned)(B + 255) / 256), dim3(256), 0, st, start, B, one, weight, weight_value);
}

void launch_raise(dim3 grid, size_t lds, hipStream_t st, const RaiseArgs& a) {
#define SLOS_RAISE(KM, SV, EX) hipLaunchKernelGGL((k_raise_rows<KM, SV, EX>), grid, dim3(256), lds, st, a)
  if (a.S < (1ull << 32)) {
    switch (a.K) {
      case 1: SLOS_RAISE(1, SpaceView32, true); return;
      case 2: SLOS_RAISE(2, SpaceView32, true); return;
      case 3: SLOS_RAISE(3, SpaceView32, true); return;
      case 4: SLOS_RAISE(4, SpaceView32, true); return;
      case 5: SLOS_RAISE(5, SpaceView32, true); return;
      case 6: SLOS_RAISE(6, SpaceView32, true); return;
      case 7: SLOS_RAISE(7, SpaceView32, true); return;
      case 8: SLOS_RAISE(8, SpaceView32, true); return;
      default: break;
    }
  }
  if (a.K <= 12) SLOS_RAISE(12, SpaceView, false);
  else SLOS_RAISE(kRaisePhotons, SpaceView, false);
#undef SLOS_RAISE
}

void launch_subsets(hipStream_t st, const SubsetArgs& a) {
  hipLaunchKernelGGL(k_subset_columns, dim3(a.rows, (unsigned)a.B), dim3(256), 0, st, a);
}

}  // namespace slos
