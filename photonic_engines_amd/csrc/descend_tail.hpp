// The last steps of the loss recurrence in one launch, from layer `top` to the vacuum: layers of a few
// thousand states, each of which was a launch that mostly waited on its own set-up. One work group a
// row keeps two layers in LDS and writes each to memory; children and sums as in the thread-per-state
// descent (bit-identical).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "block_index.hpp"

namespace slos {

constexpr int kTailThreads = 1024;
constexpr uint64_t kTailStates = 4096;      // states of a layer kept in LDS
constexpr uint64_t kTailEdges = 1u << 16;   // states times modes of one layer
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

inline size_t tail_lds(int top, int me) {
  return ((size_t)(top + 1) * (me + 1) + me) * 4 + 2 * kTailStates * sizeof(float);
}

// (descend_kernels.hip)
void launch_descend_tail(dim3 grid, size_t lds, hipStream_t st, const TailArgs& a);

}  // namespace slos
