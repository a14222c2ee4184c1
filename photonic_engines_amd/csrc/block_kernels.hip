// k_layer_block for one KIND (SLOS_BLOCK_KIND, given by the Makefile): 0 raw, 1 probabilities, 2 amplitudes, 4 readout's adjoint.
#include <hip/hip_runtime.h>

#include "block_launch.hpp"

namespace slos {

template <int KIND>
void launch_layer_block(bool comp, int d, int suf, const BlockGrid& g, const float2* par, void* out, const BlockLayer& L) {
  // one stream slot per prefix position: exact widths where the big layers live (d = K - suf)
#define SLOS_BLK(D, S)                                                                                                \
  do {                                                                                                                \
    if (comp && KIND != 4)                                                                                            \
      hipLaunchKernelGGL((k_layer_block<KIND == 4 ? 0 : KIND, true, D, S>), g.grid, dim3(kBlockThreads), g.lds, g.st, g.cg, g.lo,     \
                         g.tuples, g.me, g.me + 1, g.multiset, par, out, L);                                          \
    else                                                                                                              \
      hipLaunchKernelGGL((k_layer_block<KIND, false, D, S>), g.grid, dim3(kBlockThreads), g.lds, g.st, g.cg, g.lo,    \
                         g.tuples, g.me, g.me + 1, g.multiset, par, out, L);                                          \
  } while (0)
  if (suf == 5) {
    if (d <= 4) SLOS_BLK(4, 5);
    else if (d == 5) SLOS_BLK(5, 5);
    else if (d == 6) SLOS_BLK(6, 5);
    else if (d == 7) SLOS_BLK(7, 5);
    else SLOS_BLK(8, 5);
  } else {
    if (d <= 4) SLOS_BLK(4, 4);
    else if (d == 5) SLOS_BLK(5, 4);
    else if (d == 6) SLOS_BLK(6, 4);
    else if (d == 7) SLOS_BLK(7, 4);
    else if (d == 8) SLOS_BLK(8, 4);
    else SLOS_BLK(16, 4);
  }
#undef SLOS_BLK
}

template void launch_layer_block<SLOS_BLOCK_KIND>(bool, int, int, const BlockGrid&, const float2*, void*, const BlockLayer&);

}  // namespace slos
