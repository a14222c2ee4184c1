// The x-model's raises (photonic_engines/slos/species.py:37-56,123-146), all rows of a level in one
// launch. The rows of level L are the sets T of L distinguishable photons, on layer n - L; each is
// raised by its smallest photon into the row T minus it. In the order used here (level by level: for
// every t of level L - 1, the sets (j, t), j below t's smallest photon) the sources of a target lie one
// after another, photon 0 first.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layer_block.hpp"
#include "pull_index.hpp"
#include "space.hpp"

namespace slos {

constexpr int kRaisePhotons = 24;  // photons of a native x-model

struct RaiseArgs {
  const uint64_t* cg;
  const int* lo;
  const uint64_t* words;   // 5-position suffix words (or null)
  int me, multiset, m;
  int K;                   // photons of the targets
  int B;
  uint64_t S_par, S;
  const float* q;          // [sources][B][S_par]
  float* out;              // [targets][B][S]
  uint32_t targets, rows_per;  // in all, and of a work group (grid z)
  const uint32_t* off;     // sources of target r: off[r] .. off[r + 1] - 1, photons 0, 1, ..; null: one
  int photon;              // source, one target, this photon
  int photons;             // photons the launch raises by (weights in LDS)
  const float* row_scale;  // out holds the targets' own terms, to be scaled by these (null: nothing) ..
  const float* weight;     // .. and by this (device, or null: weight_value)
  float weight_value;
  const float2* U;         // [B][m][m]
  int cols[kRaisePhotons]; // input column of each photon
};

// One subset-forward's unitaries: row r's interfering photons' columns, in order, as columns 0..g-1 of
// Up[r - r0][b]; and row_scale[r] = 1 / prod s_i! of its input.
struct SubsetArgs {
  const float2* U;         // [B][m][m]
  float2* Up;              // [rows][B][m][m]
  const uint32_t* masks;   // distinguishable photons of every row
  uint32_t r0, rows;
  int B, m, n, g;
  float* row_scale;
  int cols[kRaisePhotons];
};

// (raise_kernels.hip)
void launch_raise(dim3 grid, size_t lds, hipStream_t st, const RaiseArgs& a);
void launch_subsets(hipStream_t st, const SubsetArgs& a);
// start[0..B-1] = the weight (device, or the value); one = 1
void launch_chain_start(hipStream_t st, float* start, int B, float* one, const float* weight, float weight_value);
inline size_t raise_lds(int K, int me, int photons) { return ((size_t)(K + 1) * (me + 1) * 8 + (size_t)me * 4 + 15) / 16 * 16 + (size_t)photons * me * 4; }

}  // namespace slos
