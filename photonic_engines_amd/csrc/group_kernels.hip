// k_layer_group: the layers of multiset spaces in group order.
#include <hip/hip_runtime.h>

#include "block_launch.hpp"

namespace slos {

void launch_layer_group(int d, int kind, bool comp, const BlockGrid& g, const float2* par, void* out, const BlockLayer& L,
                        const uint4* items, uint32_t n_items) {
  const auto* t5 = static_cast<const uint64_t*>(g.tuples);
#define SLOS_GRP(D, KIND, C)                                                                                          \
  hipLaunchKernelGGL((k_layer_group<D, KIND, C>), g.grid, dim3(kBlockThreads), g.lds, g.st, g.cg, g.lo, t5, g.me,     \
                     g.me + 1, par, out, L, items, n_items)
#define SLOS_GRP_D(D)                                                   \
  do {                                                                  \
    if (kind == 4) {                                                    \
      SLOS_GRP(D, 4, false);                                            \
    } else if (kind == 1) {                                             \
      if (comp) SLOS_GRP(D, 1, true);                                   \
      else SLOS_GRP(D, 1, false);                                       \
    } else {                                                            \
      if (comp) SLOS_GRP(D, 0, true);                                   \
      else SLOS_GRP(D, 0, false);                                       \
    }                                                                   \
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
