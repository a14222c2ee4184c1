// Launches of the block-structured kernels (layer_block.hpp, descend_block.hpp). Each family of
// instantiations is a translation unit of its own, so that they compile in parallel.
#pragma once
#include "child_walk.hpp"
#include "descend_block.hpp"
#include "layer_block.hpp"
#include "layer_block_f64.hpp"

namespace slos {

struct LayerArgs;
struct LayerArgsF64;

// k_layer_simple and its complex128 form (simple_kernels.hip)
void launch_layer_simple(int kind, bool comp, dim3 grid, size_t lds, hipStream_t st, const LayerArgs& a);
void launch_layer_f64_simple(int kind, dim3 grid, size_t lds, hipStream_t st, const LayerArgsF64& a);

// grid, LDS, stream and the plan's device tables of one launch
struct BlockGrid {
  dim3 grid;
  size_t lds;
  hipStream_t st;
  const uint64_t* cg;
  const int* lo;
  const void* tuples;
  int me, multiset;
};

// the stream-slot count instantiated for prefix width d (exact where the big layers live)
inline int block_maxd(int d) { return d <= 4 ? 4 : d <= 8 ? d : 16; }
// the same for the complex128 block kernel (d <= 8)
inline int block_maxd_f64(int d) { return d <= 4 ? 4 : d <= 6 ? 6 : 8; }

// k_layer_block for prefix width d = K - suf (block_kernels.hip, one object per KIND)
template <int KIND>
void launch_layer_block(bool comp, int d, int suf, const BlockGrid& g, const float2* par, void* out, const BlockLayer& L);

// k_layer_group for prefix width d = K - 5 in 2..6, kind 0, 1 or 4 (group_kernels.hip)
void launch_layer_group(int d, int kind, bool comp, const BlockGrid& g, const float2* par, void* out, const BlockLayer& L,
                        const uint4* items, uint32_t n_items);

// the complex128 forms (f64_kernels.hip); the block kernel for prefixes of at most 8 positions
void launch_layer_block_f64(int kind, int d, int suf, const BlockGrid& g, const double2* par, void* out,
                            const BlockLayerF64& L);
void launch_layer_group_f64(int d, int kind, const BlockGrid& g, const double2* par, void* out, const BlockLayerF64& L,
                            const uint4* items, uint32_t n_items);

// k_layer_block_group for prefix width d = K - 4 (uneven_kernels.hip)
void launch_layer_block_group(bool comp, int d, uint32_t grid, size_t lds, hipStream_t st, const GroupLaunch& gl);

// k_descend_block with maxd (4, 6 or 8) prefix slots (descend_kernels.hip)
void launch_descend_block(int maxd, const BlockGrid& g, int K, const float* qk, uint64_t Sk, float* qout, uint64_t Sp,
                          uint64_t S_pre, uint64_t per_wave, float scale, uint32_t xcd_chunk);
// the insert-table form for a prefix of dp (0 to 8) positions
void launch_descend_insert(int dp, const BlockGrid& g, const float* qk, uint64_t Sk, float* qout, uint64_t Sp,
                           uint64_t per_wave, float scale, uint32_t xcd_chunk, const uint32_t* ins);
// the adjoint of one layer, at most 32 modes
void launch_adjoint_insert(int dp, const BlockGrid& g, int m, int col, const float2* U, const float2* psi,
                           const float2* gk, uint64_t Sk, float2* gout, uint64_t Sp, uint64_t per_wave,
                           uint32_t xcd_chunk, double2* partial, const uint32_t* ins);

}  // namespace slos
