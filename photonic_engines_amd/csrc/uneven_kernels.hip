// k_layer_block_group: one launch over several plans (uneven batches).
#include <hip/hip_runtime.h>

#include "block_launch.hpp"

namespace slos {

void launch_layer_block_group(bool comp, int d, uint32_t grid, size_t lds, hipStream_t st, const GroupLaunch& gl) {
#define SLOS_BLKG(D)                                                                                             \
  do {                                                                                                           \
    if (comp) hipLaunchKernelGGL((k_layer_block_group<true, D>), dim3(grid), dim3(kBlockThreads), lds, st, gl);  \
    else hipLaunchKernelGGL((k_layer_block_group<false, D>), dim3(grid), dim3(kBlockThreads), lds, st, gl);      \
  } while (0)
  if (d <= 4) SLOS_BLKG(4);
  else if (d == 5) SLOS_BLKG(5);
  else if (d == 6) SLOS_BLKG(6);
  else if (d == 7) SLOS_BLKG(7);
  else if (d == 8) SLOS_BLKG(8);
  else SLOS_BLKG(16);
#undef SLOS_BLKG
}

}  // namespace slos
