// The pulls over children: k_descend_insert and k_adjoint_insert (child_walk.hpp), k_descend_block
// (descend_block.hpp), k_adjoint_modes (adjoint_modes.hpp), k_descend_tail
// (descend_tail.hpp).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "adjoint_modes.hpp"
#include "block_launch.hpp"
#include "descend_tail.hpp"
#include "pull_index.hpp"

namespace slos {

namespace {

template <class F>
void with_prefix(int dp, F&& f) {
  switch (dp) {
    case 0: f(std::integral_constant<int, 0>()); break;
    case 1: f(std::integral_constant<int, 1>()); break;
    case 2: f(std::integral_constant<int, 2>()); break;
    case 3: f(std::integral_constant<int, 3>()); break;
    case 4: f(std::integral_constant<int, 4>()); break;
    case 5: f(std::integral_constant<int, 5>()); break;
    case 6: f(std::integral_constant<int, 6>()); break;
    case 7: f(std::integral_constant<int, 7>()); break;
    default: f(std::integral_constant<int, 8>()); break;
  }
}

}  // namespace

void launch_descend_block(int maxd, const BlockGrid& g, int K, const float* qk, uint64_t Sk, float* qout, uint64_t Sp,
                          uint64_t S_pre, uint64_t per_wave, float scale, uint32_t xcd_chunk) {
  const auto* tuples = static_cast<const TupleWord*>(g.tuples);
#define SLOS_DESC(D, E)                                                                                            \
  hipLaunchKernelGGL((k_descend_block<D, E>), g.grid, dim3(kBlockThreads), g.lds, g.st, g.cg, g.lo, tuples, g.me, \
                     g.me + 1, K, qk, Sk, qout, Sp, S_pre, per_wave, scale, xcd_chunk)
#define SLOS_DESC_E(D)               \
  do {                               \
    if (g.me <= 16) SLOS_DESC(D, 16); \
    else if (g.me <= 32) SLOS_DESC(D, 32); \
    else SLOS_DESC(D, 64);           \
  } while (0)
  if (maxd == 4) SLOS_DESC_E(4);
  else if (maxd == 6) SLOS_DESC_E(6);
  else SLOS_DESC_E(8);
#undef SLOS_DESC_E
#undef SLOS_DESC
}

void launch_descend_insert(int dp, const BlockGrid& g, const float* qk, uint64_t Sk, float* qout, uint64_t Sp,
                           uint64_t per_wave, float scale, uint32_t xcd_chunk, const uint32_t* ins) {
  with_prefix(dp, [&](auto d) {
    hipLaunchKernelGGL((k_descend_insert<decltype(d)::value>), g.grid, dim3(kBlockThreads), 0, g.st, g.cg, ins, g.me,
                       qk, Sk, qout, Sp, per_wave, scale, xcd_chunk);
  });
}

void launch_adjoint_insert(int dp, const BlockGrid& g, int m, int col, const float2* U, const float2* psi,
                           const float2* gk, uint64_t Sk, float2* gout, uint64_t Sp, uint64_t per_wave,
                           uint32_t xcd_chunk, double2* partial, const uint32_t* ins) {
#define SLOS_ADJ(E)                                                                                                     \
  hipLaunchKernelGGL((k_adjoint_insert<decltype(d)::value, E>), g.grid, dim3(kBlockThreads), 0, g.st, g.cg, ins, g.me, \
                     m, col, U, psi, gk, Sk, gout, Sp, per_wave, xcd_chunk, partial)
  with_prefix(dp, [&](auto d) {
    if (g.me <= 16) SLOS_ADJ(16);
    else SLOS_ADJ(32);
  });
#undef SLOS_ADJ
}

void launch_adjoint_modes(int P, dim3 grid, hipStream_t st, const AdjointModesArgs& a) {
#define SLOS_MODES(N)                                                                                                   \
  do {                                                                                                                  \
    if (a.me <= 32) {                                                                                                   \
      if (a.multiset) hipLaunchKernelGGL((k_adjoint_modes<N, 32, true>), grid, dim3(kModesThreads), 0, st, a);          \
      else hipLaunchKernelGGL((k_adjoint_modes<N, 32, false>), grid, dim3(kModesThreads), 0, st, a);                    \
    } else {                                                                                                            \
      if (a.multiset) hipLaunchKernelGGL((k_adjoint_modes<N, 64, true>), grid, dim3(kModesThreads), 0, st, a);          \
      else hipLaunchKernelGGL((k_adjoint_modes<N, 64, false>), grid, dim3(kModesThreads), 0, st, a);                    \
    }                                                                                                                   \
  } while (0)
  switch (P) {
    case 0: SLOS_MODES(0); break;
    case 1: SLOS_MODES(1); break;
    case 2: SLOS_MODES(2); break;
    case 3: SLOS_MODES(3); break;
    case 4: SLOS_MODES(4); break;
    default: SLOS_MODES(5); break;
  }
#undef SLOS_MODES
}

__global__ __launch_bounds__(kTailThreads) void k_descend_tail(TailArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int stride = a.me + 1;
  const int ncg = (a.top + 1) * stride;
  float* bufs = reinterpret_cast<float*>(smem);  // the even layers, then the odd ones
  uint32_t* cg = reinterpret_cast<uint32_t*>(bufs + 2 * kTailStates);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  const size_t b = blockIdx.y;
  for (int i = threadIdx.x; i < ncg; i += kTailThreads) cg[i] = (uint32_t)a.cg[i];
  for (int i = threadIdx.x; i < a.me; i += kTailThreads) lo[i] = a.lo[i];
  const SpaceView32 sv{cg, lo, a.me, stride};
  auto layer = [&](auto km, int k) {
    constexpr int KM = decltype(km)::value;
    const int P = k - 1;
    const float* q = k == a.top ? a.q + b * a.S[a.top] : bufs + (k & 1) * kTailStates;
    float* keep = bufs + (P & 1) * kTailStates;
    float* out = a.out[P] + b * a.S[P];
    const float invk = 1.f / (float)k, scale = a.scale[P];
    for (uint32_t t = threadIdx.x; t < a.S[P]; t += kTailThreads) {
      int p[KM];
      if (KM <= 4 && a.tuples && P == KM && (a.multiset || KM == 4)) {
        const TupleWord w = a.tuples[t];
#pragma unroll
        for (int i = 0; i < KM; ++i) p[i] = (int)(tw_byte(w, (4 - KM + i) & 3) & 63u);
      } else {
        unrank_fixed<KM>(sv, t, P, p);
      }
      const float acc = children_sum<KM>(sv, a.multiset, k, p, q);
      const float v = (acc * invk) * scale;
      keep[t] = v;
      out[t] = v;
    }
  };
  for (int k = a.top; k >= 1; --k) {
    __syncthreads();
    switch (k - 1) {
      case 0:
      case 1: layer(std::integral_constant<int, 1>{}, k); break;
      case 2: layer(std::integral_constant<int, 2>{}, k); break;
      case 3: layer(std::integral_constant<int, 3>{}, k); break;
      case 4: layer(std::integral_constant<int, 4>{}, k); break;
      case 5:
      case 6:
      case 7:
      case 8: layer(std::integral_constant<int, 8>{}, k); break;
      default: layer(std::integral_constant<int, kTailTop>{}, k); break;
    }
  }
}

void launch_descend_tail(dim3 grid, size_t lds, hipStream_t st, const TailArgs& a) {
  hipLaunchKernelGGL(k_descend_tail, grid, dim3(kTailThreads), lds, st, a);
}

}  // namespace slos
