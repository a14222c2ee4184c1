// k_descend_block and k_adjoint_block (descend_block.hpp).
#include <hip/hip_runtime.h>

#include "block_launch.hpp"

namespace slos {

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

void launch_adjoint_block(int maxd, const BlockGrid& g, int K, int m, int col, const float2* U, const float2* psi,
                          const float2* gk, uint64_t Sk, float2* gout, uint64_t Sp, uint64_t S_pre, uint64_t per_wave,
                          uint32_t xcd_chunk, double2* partial) {
  const auto* tuples = static_cast<const TupleWord*>(g.tuples);
#define SLOS_ADJ(D, E)                                                                                             \
  hipLaunchKernelGGL((k_adjoint_block<D, E>), g.grid, dim3(kBlockThreads), g.lds, g.st, g.cg, g.lo, tuples, g.me, \
                     g.me + 1, K, m, col, U, psi, gk, Sk, gout, Sp, S_pre, per_wave, xcd_chunk, partial)
#define SLOS_ADJ_E(D)                \
  do {                               \
    if (g.me <= 16) SLOS_ADJ(D, 16); \
    else SLOS_ADJ(D, 32);            \
  } while (0)
  if (maxd == 4) SLOS_ADJ_E(4);
  else if (maxd == 6) SLOS_ADJ_E(6);
  else SLOS_ADJ_E(8);
#undef SLOS_ADJ_E
#undef SLOS_ADJ
}

}  // namespace slos
