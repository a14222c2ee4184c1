// complex128 form of the thread-per-state layer kernel (layer_simple.hpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "block_index.hpp"
#include "pull_index.hpp"
#include "space.hpp"

namespace slos {

struct LayerArgsF64 {
  const uint64_t* cg;
  const int* lo;
  const uint64_t* words;  // 5-position suffix words (or null)
  int me, multiset, K, m, col;
  const double2* U;    // [B][m][m]
  MatrixStride us;        // U's strides
  const double2* par;  // [B][S_par]
  uint64_t S_par;
  void* out;           // [B][S]: complex128 (kinds 0, 2) or float64 (kind 1)
  uint64_t S;
  int64_t B;
  double scale;
  unsigned immediate;  // kind 2: amplitudes times sqrt(prod t!)
};

// the counting table and lo of layer K into LDS (the first bytes of dynamic LDS)
// (SV: SpaceView, or SpaceView32 where the layer has fewer than 2^32 states)
template <class SV = SpaceView>
__device__ __forceinline__ SV load_space_f64(unsigned char* smem, const uint64_t* cg_g, const int* lo_g, int me, int K) {
  const int stride = me + 1;
  const int ncg = (K + 1) * stride;
  RankT<SV>* cg = reinterpret_cast<RankT<SV>*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = (RankT<SV>)cg_g[i];
  for (int i = threadIdx.x; i < me; i += blockDim.x) lo[i] = lo_g[i];
  return SV{cg, lo, me, stride};
}

// byte offset of the first free 16-byte slot of dynamic LDS after the table of load_space_f64
__host__ __device__ inline size_t space_lds_f64(int K, int me) {
  return ((size_t)(K + 1) * (me + 1) * 8 + (size_t)me * 4 + 15) & ~(size_t)15;
}

// layer K from layer K-1 (K <= KM; EXACT: K = KM): KIND 0 raw complex128, 1 float64 probabilities
// |amp s|^2 prod t!, 2 scaled complex128 amplitudes
template <int KIND, int KM, class SV, bool EXACT>
__global__ __launch_bounds__(256) void k_layer_f64(LayerArgsF64 a) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef RankT<SV> R;
  const int K = EXACT ? KM : a.K;
  const SV sv = load_space_f64<SV>(smem, a.cg, a.lo, a.me, K);
  double2* ucol = reinterpret_cast<double2*>(smem + space_lds_f64(K, a.me));
  for (int64_t b = blockIdx.y; b < a.B; b += gridDim.y) {
    __syncthreads();
    for (int j = threadIdx.x; j < a.m; j += blockDim.x) ucol[j] = a.U[b * a.us.B + j * a.us.R + a.col * a.us.C];
    __syncthreads();
    const double2* pb = a.par + (size_t)b * a.S_par;
    for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < a.S; g += (uint64_t)gridDim.x * blockDim.x) {
      int p[KM];
      unrank_words<KM>(sv, a.words, (R)g, K, p);
      double re = 0.0, im = 0.0;
      parents_fixed<KM>(sv, a.multiset, K, p, [&](R pr, int mode, int) {
        const double2 u = ucol[mode], v = pb[pr];
        re = fma(u.x, v.x, re);
        re = fma(-u.y, v.y, re);
        im = fma(u.x, v.y, im);
        im = fma(u.y, v.x, im);
      });
      if constexpr (KIND == 0) {
        static_cast<double2*>(a.out)[(size_t)b * a.S + g] = make_double2(re, im);
      } else {
        const double f = run_factorial_f64<KM>(p, K, a.multiset);
        re *= a.scale;
        im *= a.scale;
        if constexpr (KIND == 1) {
          static_cast<double*>(a.out)[(size_t)b * a.S + g] = (re * re + im * im) * f;
        } else {
          const double s = a.immediate ? sqrt(f) : 1.0;
          static_cast<double2*>(a.out)[(size_t)b * a.S + g] = make_double2(re * s, im * s);
        }
      }
    }
  }
}

}  // namespace slos
