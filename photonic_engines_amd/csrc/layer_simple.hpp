// Thread-per-state layer kernel: one thread a child; its positions, the ranks of its parents, gather
// and multiply-add.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "block_index.hpp"
#include "layer_block.hpp"
#include "pull_index.hpp"

namespace slos {

struct LayerArgs {
  const uint64_t* cg;
  const int* lo;
  int me, multiset, K, m, col;
  const float2* U;        // [B][m][m]
  MatrixStride us;        // U's strides
  const uint64_t* words;  // 5-position suffix words (or null)
  const float2* par;      // [B][S_par]
  uint64_t S_par;
  void* out;              // [B][S]
  uint64_t S;
  int64_t B;
  float scale;
  unsigned flags;
  int64_t par_lo, out_lo;  // compensated sums: element offsets of the low-order parts (0: none)
  const float* gp = nullptr;  // KIND 4: dL/dp [B][S]
};

// KIND 0: intermediate layer (complex64), 1: probabilities (float32), 2: scaled amplitudes, 4: the
// readout's adjoint (readout_gradient)
// (K <= KM: the per-state position arrays stay in registers; SV: 32-bit counts where the layer has
// fewer than 2^32 states; EXACT: K = KM). Bound by VALU instructions, most of them index arithmetic: with
// K known the compiler drops the guards and selects of the unrolled loops, the ranks take two table
// entries a position (parents_fixed) and the search ends with the prefix (unrank_words). n = 8, m = 24,
// layer 8 175 -> 94 us; collision-free n = 9, m = 26, layer 9 97 -> 55 us. Loading all parents before the
// first sum measured slower (149 against 135 us at n = 8, m = 24: registers for waves).
template <int KIND, bool COMP, int KM, class SV, bool EXACT>
__global__ __launch_bounds__(256) void k_layer_simple(LayerArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  typedef RankT<SV> R;
  const int K = EXACT ? KM : a.K;
  const int stride = a.me + 1;
  const int ncg = (K + 1) * stride;
  R* cg = reinterpret_cast<R*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  float2* ucol = reinterpret_cast<float2*>(smem + ((ncg * 8 + a.me * 4 + 15) & ~15));
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = (R)a.cg[i];
  for (int i = threadIdx.x; i < a.me; i += blockDim.x) lo[i] = a.lo[i];
  const SV sv{cg, lo, a.me, stride};
  for (int64_t b = blockIdx.y; b < a.B; b += gridDim.y) {
    __syncthreads();
    for (int j = threadIdx.x; j < a.m; j += blockDim.x)
      ucol[j] = a.U[b * a.us.B + j * a.us.R + a.col * a.us.C];
    __syncthreads();
    const float2* pb = a.par + (size_t)b * a.S_par;
    for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < a.S;
         g += (uint64_t)gridDim.x * blockDim.x) {
      int p[KM];
      unrank_words<KM>(sv, a.words, (R)g, K, p);
      BlockAcc<COMP> acc;
      parents_fixed<KM>(sv, a.multiset, K, p, [&](R pr, int mode, int) { bk_cmac(acc, ucol[mode], pb[pr]); });
      if constexpr (COMP) {
        if (a.par_lo)  // the parents' low-order parts
          parents_fixed<KM>(sv, a.multiset, K, p, [&](R pr, int mode, int) { bk_lo_mac(acc, ucol[mode], pb[a.par_lo + pr]); });
      }
      const float2 sum = acc.value();
      float re = sum.x, im = sum.y;
      if constexpr (KIND == 0) {
        reinterpret_cast<float2*>(a.out)[(size_t)b * a.S + g] = make_float2(re, im);
        if constexpr (COMP) {
          if (a.out_lo) reinterpret_cast<float2*>(a.out)[a.out_lo + (size_t)b * a.S + g] = acc.rest(sum);
        }
      } else if constexpr (KIND == 4) {
        const uint64_t c = (uint64_t)b * a.S + g;
        reinterpret_cast<float2*>(a.out)[c] =
            readout_gradient(re, im, a.scale, run_factorial_fixed<KM>(p, K, a.multiset), a.gp[c]);
      } else {
        const float f = run_factorial_fixed<KM>(p, K, a.multiset);
        re *= a.scale;
        im *= a.scale;
        if constexpr (KIND == 1) {
          reinterpret_cast<float*>(a.out)[(size_t)b * a.S + g] = prob_readout(re, im, f);
        } else {
          const float s = (a.flags & 2u) ? sqrtf(f) : 1.f;
          reinterpret_cast<float2*>(a.out)[(size_t)b * a.S + g] = make_float2(re * s, im * s);
        }
      }
    }
  }
}

}  // namespace slos
