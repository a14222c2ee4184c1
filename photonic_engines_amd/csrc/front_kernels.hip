// k_front: the first layers of a forward in one launch (front.hpp).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "front.hpp"

namespace slos {

namespace {

template <class T>
struct Pair;
template <>
struct Pair<float> {
  typedef float2 type;
};
template <>
struct Pair<double> {
  typedef double2 type;
};

// one complex sum: plain (float, double) or compensated (float), as the layer kernels add it
template <class T, bool COMP>
struct Sum {
  T re = 0, im = 0;
  BlockAcc<COMP> c;
  __device__ __forceinline__ void add(typename Pair<T>::type u, typename Pair<T>::type v) {
    if constexpr (std::is_same<T, float>::value) {
      bk_cmac(c, u, v);
    } else {
      re = fma(u.x, v.x, re);
      re = fma(-u.y, v.y, re);
      im = fma(u.x, v.y, im);
      im = fma(u.y, v.x, im);
    }
  }
};

}  // namespace

template <class T, bool COMP>
__global__ __launch_bounds__(kFrontThreads) void k_front(FrontArgs a) {
  typedef typename Pair<T>::type T2;
  extern __shared__ __align__(16) unsigned char smem[];
  const int stride = a.me + 1;
  const int ncg = (a.kf + 1) * stride;
  uint32_t* cg = reinterpret_cast<uint32_t*>(smem);
  int* lo = reinterpret_cast<int*>(cg + ncg);
  T2* ucols = reinterpret_cast<T2*>(smem + (((ncg + a.me) * 4 + 15) & ~15));
  T2* bufs[2] = {ucols + a.kf * a.m, ucols + a.kf * a.m + (COMP ? 2 : 1) * a.buf};
  const int64_t b = blockIdx.y;
  const T2* U = static_cast<const T2*>(a.U) + b * a.us.B;
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg[i] = (uint32_t)a.cg[i];
  for (int i = threadIdx.x; i < a.me; i += blockDim.x) lo[i] = a.lo[i];
  for (int i = threadIdx.x; i < a.kf * a.m; i += blockDim.x) {
    const int k = i / a.m, j = i - k * a.m;
    ucols[i] = U[j * a.us.R + a.cols[k] * a.us.C];
  }
  if (threadIdx.x == 0) {
    bufs[0][0] = T2{1, 0};
    if constexpr (COMP) bufs[0][a.buf] = T2{0, 0};
  }
  const bool keep = a.below[0] && blockIdx.x == 0;  // one work group a row writes the layers below kf
  if (keep && threadIdx.x == 0) static_cast<T2*>(a.below[0])[b] = T2{1, 0};
  const SpaceView32 sv{cg, lo, a.me, stride};
  auto layer = [&](auto km, int K, bool last) {
    constexpr int KM = decltype(km)::value;
    const T2* par = bufs[(K - 1) & 1];
    T2* dst = bufs[K & 1];
    const T2* ucol = ucols + (K - 1) * a.m;
    const uint32_t S = a.S[K];
    const uint32_t first = last ? blockIdx.x * kFrontThreads : 0u;
    const uint32_t end = last ? (first + kFrontThreads < S ? first + kFrontThreads : S) : S;
    for (uint32_t g = first + threadIdx.x; g < end; g += blockDim.x) {
      int p[KM];
      // positions: in a multiset space the k-tuple g, k <= 4, is the 4-tuple g without its leading
      // zeros; a 4- or 5-tuple is its own word
      if (KM <= 4 && a.tuples && (a.multiset || KM == 4)) {
        const TupleWord w = a.tuples[g];
#pragma unroll
        for (int i = 0; i < KM; ++i) p[i] = (int)(tw_byte(w, (4 - KM + i) & 3) & 63u);
      } else if (KM == 5 && a.tuples5) {
        const uint64_t w = a.tuples5[g];
#pragma unroll
        for (int i = 0; i < KM; ++i) p[i] = (int)(tw_byte(w, i) & 63u);
      } else if (a.me >= 3 * KM) {
        // one search of log2(me) reads a position where a walk over the modes is long: us a forward against the
        // walk, n = 3, m = 64 11.5 / 27.3, n = 4, m = 32 20.5 / 30.3, n = 4, m = 24 14.6 / 19.4, n = 4, m = 12
        // 10.8 / 11.9, n = 6, m = 18 17.1 / 17.2. Below 3 modes a position the walk takes few more reads than
        // the searches do.
        unrank_search<KM>(sv, g, K, p);
      } else {
        unrank_fixed<KM>(sv, g, K, p);
      }
      Sum<T, COMP> s;
      parents_fixed<KM>(sv, a.multiset, K, p, [&](uint32_t pr, int mode, int) { s.add(ucol[mode], par[pr]); });
      if constexpr (COMP) {
        if (K > 1)  // the parents' low-order parts
          parents_fixed<KM>(sv, a.multiset, K, p,
                            [&](uint32_t pr, int mode, int) { bk_lo_mac(s.c, ucol[mode], par[a.buf + pr]); });
      }
      T re, im;
      if constexpr (std::is_same<T, float>::value) {
        const float2 sum = s.c.value();
        re = sum.x;
        im = sum.y;
      } else {
        re = s.re;
        im = s.im;
      }
      if (!last) {
        dst[g] = T2{re, im};
        if (keep) (static_cast<T2*>(a.below[K]) + (size_t)b * S)[g] = T2{re, im};
        if constexpr (COMP) dst[a.buf + g] = s.c.rest(T2{re, im});
      } else if (a.kind == 0) {
        T2* out = static_cast<T2*>(a.out) + (size_t)b * S;
        out[g] = T2{re, im};
        if constexpr (COMP)
          if (a.out_lo) out[a.out_lo + g] = s.c.rest(T2{re, im});
      } else {
        T f;
        if constexpr (std::is_same<T, float>::value) f = run_factorial_fixed<KM>(p, K, a.multiset);
        else f = run_factorial_f64<KM>(p, K, a.multiset);
        re *= (T)a.scale;
        im *= (T)a.scale;
        if (a.kind == 1) {
          T* out = static_cast<T*>(a.out) + (size_t)b * S;
          if constexpr (std::is_same<T, float>::value) out[g] = prob_readout(re, im, f);
          else out[g] = (re * re + im * im) * f;
        } else {
          const T q = a.immediate ? sqrt(f) : T(1);
          (static_cast<T2*>(a.out) + (size_t)b * S)[g] = T2{re * q, im * q};
        }
      }
    }
  };
  for (int K = 1; K <= a.kf; ++K) {
    __syncthreads();
    const bool last = K == a.kf;
    switch (K) {
      case 1: layer(std::integral_constant<int, 1>{}, K, last); break;
      case 2: layer(std::integral_constant<int, 2>{}, K, last); break;
      case 3: layer(std::integral_constant<int, 3>{}, K, last); break;
      case 4: layer(std::integral_constant<int, 4>{}, K, last); break;
      case 5: layer(std::integral_constant<int, 5>{}, K, last); break;
      case 6: layer(std::integral_constant<int, 6>{}, K, last); break;
      case 7:
      case 8: layer(std::integral_constant<int, 8>{}, K, last); break;
      default: layer(std::integral_constant<int, kFrontMax>{}, K, last); break;
    }
  }
}

void launch_front(bool f64, bool comp, dim3 grid, size_t lds, hipStream_t st, const FrontArgs& a) {
  if (f64) hipLaunchKernelGGL((k_front<double, false>), grid, dim3(kFrontThreads), lds, st, a);
  else if (comp) hipLaunchKernelGGL((k_front<float, true>), grid, dim3(kFrontThreads), lds, st, a);
  else hipLaunchKernelGGL((k_front<float, false>), grid, dim3(kFrontThreads), lds, st, a);
}

}  // namespace slos
