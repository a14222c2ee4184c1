// k_layer_simple and k_layer_f64 (layer_simple.hpp, layer_simple_f64.hpp).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "block_launch.hpp"
#include "layer_simple.hpp"
#include "layer_simple_f64.hpp"

namespace slos {

namespace {

// f(KM, view, exact): the photon count itself for 1..12 photons (with 32-bit counts), else the
// smallest bound 8, 16 or 32 that holds it. (Below 5 photons the 8-photon bound's guards and selects are
// most of the instructions: 60,000 rows of n = 2, m = 4 218 us with it, 84 so; 20,000 of n = 3, m = 6 121 and 55.)
template <class F>
void with_photons(int K, bool narrow, F&& f) {
  if (narrow) {
    switch (K) {
#define SLOS_EXACT(N) \
  case N: f(std::integral_constant<int, N>{}, SpaceView32{}, std::true_type{}); return
      SLOS_EXACT(1);
      SLOS_EXACT(2);
      SLOS_EXACT(3);
      SLOS_EXACT(4);
      SLOS_EXACT(5);
      SLOS_EXACT(6);
      SLOS_EXACT(7);
      SLOS_EXACT(8);
      SLOS_EXACT(9);
      SLOS_EXACT(10);
      SLOS_EXACT(11);
      SLOS_EXACT(12);
#undef SLOS_EXACT
    }
  }
  auto bound = [&](auto km) {
    if (narrow) f(km, SpaceView32{}, std::false_type{});
    else f(km, SpaceView{}, std::false_type{});
  };
  if (K <= 8) bound(std::integral_constant<int, 8>{});
  else if (K <= 16) bound(std::integral_constant<int, 16>{});
  else bound(std::integral_constant<int, 32>{});
}

}  // namespace

void launch_layer_simple(int kind, bool comp, dim3 grid, size_t lds, hipStream_t st, const LayerArgs& a) {
  with_photons(a.K, a.S < (1ull << 32), [&](auto km, auto view, auto exact) {
    constexpr int KM = decltype(km)::value;
    constexpr bool EX = decltype(exact)::value;
    typedef decltype(view) SV;
    if (!comp) {
      if (kind == 0) hipLaunchKernelGGL((k_layer_simple<0, false, KM, SV, EX>), grid, dim3(256), lds, st, a);
      else if (kind == 1) hipLaunchKernelGGL((k_layer_simple<1, false, KM, SV, EX>), grid, dim3(256), lds, st, a);
      else if (kind == 4) hipLaunchKernelGGL((k_layer_simple<4, false, KM, SV, EX>), grid, dim3(256), lds, st, a);
      else hipLaunchKernelGGL((k_layer_simple<2, false, KM, SV, EX>), grid, dim3(256), lds, st, a);
    } else {
      if (kind == 0) hipLaunchKernelGGL((k_layer_simple<0, true, KM, SV, EX>), grid, dim3(256), lds, st, a);
      else if (kind == 1) hipLaunchKernelGGL((k_layer_simple<1, true, KM, SV, EX>), grid, dim3(256), lds, st, a);
      else hipLaunchKernelGGL((k_layer_simple<2, true, KM, SV, EX>), grid, dim3(256), lds, st, a);
    }
  });
}

void launch_layer_f64_simple(int kind, dim3 grid, size_t lds, hipStream_t st, const LayerArgsF64& a) {
  with_photons(a.K, a.S < (1ull << 32), [&](auto km, auto view, auto exact) {
    constexpr int KM = decltype(km)::value;
    constexpr bool EX = decltype(exact)::value;
    typedef decltype(view) SV;
    if (kind == 0) hipLaunchKernelGGL((k_layer_f64<0, KM, SV, EX>), grid, dim3(256), lds, st, a);
    else if (kind == 1) hipLaunchKernelGGL((k_layer_f64<1, KM, SV, EX>), grid, dim3(256), lds, st, a);
    else hipLaunchKernelGGL((k_layer_f64<2, KM, SV, EX>), grid, dim3(256), lds, st, a);
  });
}

}  // namespace slos
