// The first layers of a forward in one launch.
//
// A layer of a few thousand states is a launch of 5 us whose kernel waits on its own set-up, and a
// forward begins with four or five of them (and a fill of layer 0). Here a work group computes the
// layers 1 .. kf-1 for itself, in LDS, and then its own 1,024 states of layer kf: the same parent sums
// in the same order (bit-identical), computed again by every work group, which costs less than the
// launches as long as layer kf-1 has at most kFrontStates states and the work groups of all rows
// together do not fill the chip (see front_layers in slos.hip). A launch takes about 10 us (where the
// tuple words do not give the positions they are searched for, see k_front); it replaces the fill and 3 to 6
// launches of 5 us or more: probs(U) at n = 4, m = 12 34.8 -> 21.5 us, n = 6, m = 18 42.6 -> 24.3 us,
// n = 8, m = 24 126 -> 107 us (with the host's part of then, 20 us of the first two).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layer_block.hpp"
#include "pull_index.hpp"
#include "space.hpp"

namespace slos {

constexpr int kFrontThreads = 1024;
constexpr int kFrontMax = 16;            // layers of one launch
constexpr uint64_t kFrontStates = 6144;  // states of a layer kept in LDS

struct FrontArgs {
  const uint64_t* cg;
  const int* lo;
  const TupleWord* tuples;   // 4- and 5-position tuple words (or null: positions by unranking)
  const uint64_t* tuples5;
  int me, multiset, m, kf;
  int kind;                  // of layer kf: 0 raw, 1 probabilities, 2 scaled amplitudes
  const void* U;             // [B][m][m]
  MatrixStride us;           // U's strides
  int cols[kFrontMax];       // input column of layer k at cols[k - 1]
  uint32_t S[kFrontMax + 1];
  uint32_t buf;              // LDS elements of one ping-pong buffer
  void* out;                 // [B][S_kf]
  double scale;
  unsigned immediate;
  int64_t out_lo;            // compensated sums: offset of layer kf's low-order parts (0: none)
  void* below[kFrontMax];    // layers 0..kf-1 in memory [B][S_k] too, for a backward pass (null: not)
};

// LDS: cg rows 0..kf (32-bit), lo, the input columns, two layers (twice with low-order parts)
inline size_t front_table_bytes(int kf, int me) {
  return (((size_t)(kf + 1) * (me + 1) + me) * 4 + 15) & ~(size_t)15;
}
inline size_t front_lds(int kf, int me, int m, size_t elem, uint64_t buf, bool comp) {
  return front_table_bytes(kf, me) + (size_t)kf * m * elem + 2 * buf * elem * (comp ? 2 : 1);
}

// (front_kernels.hip)
void launch_front(bool f64, bool comp, dim3 grid, size_t lds, hipStream_t st, const FrontArgs& a);

}  // namespace slos
