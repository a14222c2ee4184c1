// The last steps of the loss recurrence in one launch, from layer `top` to the vacuum: layers of a few
// thousand states, each of which was a launch that mostly waited on its own set-up. One work group a
// row keeps two layers in LDS and writes each to memory; children and sums as in the thread-per-state
// descent (bit-identical). Only layers of a few hundred states: one work group takes 56 us for the 2,600
// of layer 3 at 24 modes and those below with its gathers one at a time, 40 us with eight at a time
// (children_sum), and 19 us (from layer 3 on, all launches of 5 us or more before) as it is.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "block_index.hpp"
#include "pull_index.hpp"

namespace slos {

constexpr int kTailThreads = 1024;
constexpr uint64_t kTailStates = 4096;      // states of a layer kept in LDS
constexpr uint64_t kTailEdges = 1u << 13;   // states times modes of one layer
constexpr int kTailTop = 32;

struct TailArgs {
  const uint64_t* cg;
  const int* lo;
  const TupleWord* tuples;     // 4-position tuple words (or null)
  int me, multiset, top;
  const float* q;              // layer `top` [B][S[top]]
  uint32_t S[kTailTop + 1];
  float* out[kTailTop];        // layer k [B][S[k]], k < top
  float scale[kTailTop];       // of layer k
};

#if defined(__HIPCC__)

// sum of q(child) times the child's copies of the mode over the children of the (k-1)-tuple p (k - 1 <= KM),
// modes ascending, eight gathers at a time. A mode's child in the telescoped ranks of pull_index.hpp
// (e(r, x) = cg[r][x+1], cg[1][x] for r = 1; i = the number of p_l <= j):
//   cg[k][0] - sum_{p_l <= j} e(k-l, p_l) - e(k-i, j) - sum_{p_l > j} e(k-1-l, p_l)
template <int KM>
__device__ __forceinline__ float children_sum(const SpaceView32& sv, int multiset, int k, const int (&p)[KM], const float* q) {
  const int P = k - 1;
  uint32_t le[KM], gt[KM];
#pragma unroll
  for (int l = 0; l < KM; ++l) {
    le[l] = l < P ? sv.C(k - l, p[l] + 1) : 0u;
    gt[l] = l >= P ? 0u : l == P - 1 ? sv.C(1, p[l]) : sv.C(k - 1 - l, p[l] + 1);
  }
  const uint32_t top = sv.C(k, 0);
  float acc = 0.f;
  for (int j0 = 0; j0 < sv.me; j0 += 8) {
    float v[8], copies[8];
    bool child[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int j = j0 + u < sv.me ? j0 + u : sv.me - 1;
      uint32_t c = top;
      int i = 0, n = 1, before = 0, after = 1 << 30;
#pragma unroll
      for (int l = KM - 1; l >= 0; --l)
        if (l < P) {
          const bool b = p[l] <= j;
          c -= b ? le[l] : gt[l];
          i += b ? 1 : 0;
          n += p[l] == j ? 1 : 0;
          after = b ? after : p[l];
          before = b && p[l] > before ? p[l] : before;
        }
      c -= i == P ? sv.C(1, j) : sv.C(k - i, j + 1);
      // (a set mask takes no mode up to the last position's block, nor one of the next position's)
      child[u] = j0 + u < sv.me && (multiset || ((i == 0 || sv.lo[before] <= j) && sv.lo[j] <= after));
      v[u] = q[child[u] ? c : 0u];
      copies[u] = (float)n;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = child[u] ? fmaf(v[u], copies[u], acc) : acc;
  }
  return acc;
}

#endif

inline size_t tail_lds(int top, int me) {
  return ((size_t)(top + 1) * (me + 1) + me) * 4 + 2 * kTailStates * sizeof(float);
}

// (descend_kernels.hip)
void launch_descend_tail(dim3 grid, size_t lds, hipStream_t st, const TailArgs& a);

}  // namespace slos
