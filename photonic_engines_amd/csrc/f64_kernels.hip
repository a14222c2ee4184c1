// k_layer_block_f64 and k_layer_group_f64 (layer_block_f64.hpp).
#include <hip/hip_runtime.h>

#include "block_launch.hpp"

namespace slos {

void launch_layer_block_f64(int kind, int d, int suf, const BlockGrid& g, const double2* par, void* out,
                            const BlockLayerF64& L) {
#define SLOS_BLK(KIND, D, S)                                                                                       \
  hipLaunchKernelGGL((k_layer_block_f64<KIND, D, S>), g.grid, dim3(kBlockThreads), g.lds, g.st, g.cg, g.lo,        \
                     g.tuples, g.me, g.me + 1, g.multiset, par, out, L)
#define SLOS_BLK_S(D, S)                      \
  do {                                        \
    if (kind == 0) SLOS_BLK(0, D, S);         \
    else if (kind == 1) SLOS_BLK(1, D, S);    \
    else SLOS_BLK(2, D, S);                   \
  } while (0)
#define SLOS_BLK_D(D)                         \
  do {                                        \
    if (suf == 5) SLOS_BLK_S(D, 5);           \
    else SLOS_BLK_S(D, 4);                    \
  } while (0)
  if (d <= 4) SLOS_BLK_D(4);
  else if (d <= 6) SLOS_BLK_D(6);
  else SLOS_BLK_D(8);
#undef SLOS_BLK_D
#undef SLOS_BLK_S
#undef SLOS_BLK
}

void launch_layer_group_f64(int d, int kind, const BlockGrid& g, const double2* par, void* out, const BlockLayerF64& L,
                            const uint4* items, uint32_t n_items) {
  const auto* t5 = static_cast<const uint64_t*>(g.tuples);
#define SLOS_GRP(D, KIND)                                                                                        \
  hipLaunchKernelGGL((k_layer_group_f64<D, KIND>), g.grid, dim3(kBlockThreads), g.lds, g.st, g.cg, g.lo, t5,     \
                     g.me, g.me + 1, par, out, L, items, n_items)
#define SLOS_GRP_D(D)                         \
  do {                                        \
    if (kind == 1) SLOS_GRP(D, 1);            \
    else SLOS_GRP(D, 0);                      \
  } while (0)
  if (d <= 2) SLOS_GRP_D(2);
  else if (d == 3) SLOS_GRP_D(3);
  else if (d == 4) SLOS_GRP_D(4);
  else if (d == 5) SLOS_GRP_D(5);
  else SLOS_GRP_D(6);
#undef SLOS_GRP_D
#undef SLOS_GRP
}

}  // namespace slos
