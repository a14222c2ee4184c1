// The layer adjoint on small layers, a lane a mode (see k_adjoint_insert for what it computes).
//
// A group of 32 lanes (64 with more than 32 modes) takes a parent: lane j gathers the child with mode j,
// so that dL/dU needs no sum over lanes and grad_prev one. The child's rank is the telescoped sum of
// pull_index.hpp: with e(r, x) = cg[r][x+1] (cg[1][x] for r = 1), i = the number of p_l <= j,
//   cg[k][0] - sum_{p_l <= j} e(k-l, p_l) - e(k-i, j) - sum_{p_l > j} e(k-1-l, p_l),
// of which the sums' terms are the group's and e(k-i, j), i = 0..P, the lane's own for all parents.
// The thread-per-state kernel took 10 to 26 us for such a layer, whatever its size: one wave a work group,
// a thread's modes one after another, and its sums of dL/dU added up by a loop over 64 rows. Here a
// parent is one gather; a launch takes 5 to 8 us, its own latency (us with the sum over work groups
// and the host's part, at n = 8, m = 24, layers 6 to 1: 35 / 38 / 37 / 32 / 31 / 25 -> 31 / 24 / 23 / 23 / 23 / 23).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layer_block.hpp"
#include "pull_index.hpp"
#include "space.hpp"

namespace slos {

constexpr int kModesThreads = 256;
constexpr int kModesPhotons = 5;  // parents of at most this many photons

struct AdjointModesArgs {
  const uint64_t* cg;
  const int* lo;
  const TupleWord* tuples;   // 4- and 5-position tuple words (or null)
  const uint64_t* tuples5;
  int me, multiset, m, col;
  const float2* U;           // [B][m][m]
  const float2* psi;         // [B][Sp]
  const float2* gk;          // [B][Sk]
  float2* gout;              // [B][Sp] or null
  uint32_t Sp, Sk;
  uint32_t turns;            // parents a group takes, one after another
  double2* partial;          // [B][work groups][me]
};

inline int modes_lanes(int me) { return me <= 32 ? 32 : 64; }
inline uint32_t modes_groups(int me) { return (uint32_t)(kModesThreads / modes_lanes(me)); }

// parents of P <= kModesPhotons photons (descend_kernels.hip)
void launch_adjoint_modes(int P, dim3 grid, hipStream_t st, const AdjointModesArgs& a);

#if defined(__HIPCC__)

// v plus that of the lanes a DPP control names (zero where it names none, or the row mask is off)
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROWS, 0xf, false));
}
// the sum over each group of G lanes, in its last lane
template <int G>
__device__ __forceinline__ float group_sum(float v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  if (G == 64) v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}

template <int P, int G, bool MULTISET>
__global__ __launch_bounds__(kModesThreads) void k_adjoint_modes(AdjointModesArgs a) {
  constexpr int K = P + 1;
  constexpr int kRow = 65;
  constexpr int kGroups = kModesThreads / G;
  __shared__ uint32_t cg[(K + 1) * kRow];
  __shared__ int lo[64];
  __shared__ double2 sum[kGroups][G];
  const int stride = a.me + 1;
  for (int i = threadIdx.x; i < (K + 1) * stride; i += kModesThreads) cg[i] = (uint32_t)a.cg[i];
  for (int i = threadIdx.x; i < a.me; i += kModesThreads) lo[i] = a.lo[i];
  __syncthreads();
  const SpaceView32 sv{cg, lo, a.me, stride};
  const int64_t b = blockIdx.y;
  const int j = (int)(threadIdx.x % G);
  const uint32_t group = threadIdx.x / G;
  const bool mode = j < a.me;
  const int jj = mode ? j : 0;
  const int lo_j = MULTISET ? 0 : lo[jj];
  uint32_t own[P + 1];  // e(K - i, j)
#pragma unroll
  for (int i = 0; i <= P; ++i) own[i] = i == P ? sv.C(1, jj) : sv.C(K - i, jj + 1);
  const float2 u = mode ? a.U[(size_t)b * a.m * a.m + (size_t)j * a.m + a.col] : make_float2(0.f, 0.f);
  const float2* psi = a.psi + (size_t)b * a.Sp;
  const float2* gk = a.gk + (size_t)b * a.Sk;
  float2* gout = a.gout ? a.gout + (size_t)b * a.Sp : nullptr;
  const uint32_t top = sv.C(K, 0);
  double2 acc = make_double2(0.0, 0.0);
  for (uint32_t turn = 0; turn < a.turns; ++turn) {
    const uint32_t t = (blockIdx.x * a.turns + turn) * kGroups + group;
    const bool in = t < a.Sp;
    const uint32_t tt = in ? t : a.Sp - 1u;
    int p[P ? P : 1] = {};
    if constexpr (P > 0) {
      if (P <= 4 && a.tuples && (MULTISET || P == 4)) {
        const TupleWord w = a.tuples[tt];
#pragma unroll
        for (int i = 0; i < P; ++i) p[i] = (int)(tw_byte(w, (4 - P + i) & 3) & 63u);
      } else if (P == 5 && a.tuples5) {
        const uint64_t w = a.tuples5[tt];
#pragma unroll
        for (int i = 0; i < P; ++i) p[i] = (int)(tw_byte(w, i) & 63u);
      } else {
        unrank_fixed<P>(sv, tt, P, p);
      }
    }
    uint32_t idx = top, mine = own[0];
    int before = 0, after = P ? p[0] : 64;
    bool first = true;
#pragma unroll
    for (int l = 0; l < P; ++l) {
      const bool le = p[l] <= jj;
      idx -= le ? sv.C(K - l, p[l] + 1) : (l == P - 1 ? sv.C(1, p[l]) : sv.C(K - 1 - l, p[l] + 1));
      mine = le ? own[l + 1] : mine;
      if (!MULTISET && le) {
        before = lo[p[l]];
        after = l + 1 < P ? p[in_range<P ? P : 1>(l + 1)] : 64;
        first = false;
      }
    }
    idx -= mine;
    bool child = mode && in;
    if (!MULTISET) child = child && (first || before <= jj) && lo_j <= after;
    const float2 ps = psi[tt];
    const float2 g = child ? gk[idx] : make_float2(0.f, 0.f);
    // (the products are selected, not g alone: where there is no child, an infinite or NaN psi or U adds nothing)
    acc.x += child ? (double)fmaf(ps.y, g.y, ps.x * g.x) : 0.0;  // conj(psi) * g
    acc.y += child ? (double)fmaf(-ps.y, g.x, ps.x * g.y) : 0.0;
    if (gout) {
      const float gr = group_sum<G>(child ? fmaf(u.y, g.y, u.x * g.x) : 0.f);   // conj(u) * g
      const float gi = group_sum<G>(child ? fmaf(-u.y, g.x, u.x * g.y) : 0.f);
      if (in && j == G - 1) gout[t] = make_float2(gr, gi);
    }
  }
  sum[group][j] = acc;
  __syncthreads();
  if (threadIdx.x < a.me) {
    double sr = 0.0, si = 0.0;
#pragma unroll
    for (int i = 0; i < kGroups; ++i) {
      sr += sum[i][threadIdx.x].x;
      si += sum[i][threadIdx.x].y;
    }
    a.partial[((size_t)b * gridDim.x + blockIdx.x) * a.me + threadIdx.x] = make_double2(sr, si);
  }
}

#endif

}  // namespace slos
