// Pulls over children through the insert table (block_index.hpp: insert_word), for multiset spaces of
// at most 41 modes and parent layers D = K - 1 = DP + 4, DP = 1..8: one step of the uniform-loss
// recurrence (photonic_engines/imperfections.py:254-276), q_{K-1}(t) = sum_a q_K(t + e_a) (t_a + 1) / K.
//
// A wave owns a contiguous range of parents and takes it block by block (a block: the parents (P, u)
// of one DP-position prefix P, u their last four positions). The block's data stay in registers:
// lane a holds the base of mode a's child stream and the copies of a, computed for all modes at once
// from lane tables of the counting rows (lane x of row l: cg[K - l][x + 1]):
//   a < last(P): the children of the block's parents lie one after another, from
//     cg[K][0] - sum_{p_l <= a} cg[K-l][p_l+1] - cg[K-i][a+1] - sum_{p_l > a} cg[K-1-l][p_l+1] - cg[4][last(P)]
//     (i = the number of p_l <= a);
//   a >= last(P): index of the insert table past cg[K][0] - sum_l cg[K-l][p_l+1] - N5.
// The lanes hold adjacent parents (64 at a time, up to four such groups a step), so that streams,
// table words and stores are coalesced and the children above last(P) nearly so.
// The sums run over ascending modes with the fused multiply-adds of the thread-per-state kernel: the
// two give bit-identical results.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layer_block.hpp"

namespace slos {

// a block's children, for one wave (wave-uniform but for the lane-held tables)
struct ChildBlock {
  uint64_t CBp;     // first parent of the block
  uint64_t sb;      // lane a < last(P): base of mode a's child stream, at u = 0
  uint64_t tail;    // child of index 0 of the insert table
  uint32_t cnt;     // lane a: 1 + copies of a in P
  uint32_t toff;    // the block's first 4-tuple
  int lastP;
};

// sweep(block, u0, u_stop) for each block of the parents [g, g + per_wave) of layer DP + 4
template <int DP, class Sweep>
__device__ __forceinline__ void child_walk(const uint64_t* __restrict__ cg, int me, uint64_t Sp, uint64_t per_wave,
                                           uint64_t g, Sweep&& sweep) {
  constexpr int K = DP + 5;
  const int W = me + 1;
  const int lane = threadIdx.x & 63;
  if (g >= Sp) return;
  const uint64_t g_end = g + per_wave < Sp ? g + per_wave : Sp;
  uint64_t row[DP + 1];  // lane x: cg[K - l][x + 1]
#pragma unroll
  for (int l = 0; l <= DP; ++l) row[l] = lane < me ? cg[(K - l) * W + lane + 1] : 0u;
  const uint32_t c4 = lane < me ? (uint32_t)cg[4 * W + lane] : 0u;
  const uint64_t cK = cg[K * W], n5 = cg[5 * W];
  const uint32_t n4 = (uint32_t)cg[4 * W];
  // the prefix of parent g: position l is the number of modes x >= its predecessor that g's rank
  // among the tuples from there on has passed
  int p[DP];
  uint64_t u0 = g;
  {
    uint64_t top = Sp;
    int lo = 0;
#pragma unroll
    for (int l = 0; l < DP; ++l) {
      const uint64_t passed = __builtin_amdgcn_ballot_w64(lane >= lo && lane < me - 1 && top - row[l + 1] <= u0);
      p[l] = lo + __builtin_popcountll(passed);
      const uint64_t at = p[l] == lo ? top : rl64(row[l + 1], p[l] - 1);
      u0 -= top - at;
      top = at - rl64(row[l + 1], p[l]);
      lo = p[l];
    }
  }
  while (g < g_end) {
    ChildBlock b;
    b.lastP = p[DP - 1];
    const uint32_t L = rl(c4, b.lastP);
    b.CBp = g - u0;
    b.toff = n4 - L;
    uint64_t lower = cK, own = row[0];  // lane a: lower - own = its stream's base
    uint64_t tail = cK - n5;
    b.cnt = 1u;
#pragma unroll
    for (int l = 0; l < DP; ++l) {
      const uint64_t s_le = rl64(row[l], p[l]), s_gt = rl64(row[l + 1], p[l]);
      const bool le = p[l] <= lane;
      lower -= le ? s_le : s_gt;
      own = le ? row[l + 1] : own;
      b.cnt += p[l] == lane ? 1u : 0u;
      tail -= s_le;
    }
    b.sb = lower - own - (uint64_t)L;
    b.tail = tail;
    const uint64_t left = g_end - g;
    const uint32_t u_stop = (uint64_t)L - u0 < left ? L : (uint32_t)(u0 + left);
    sweep(b, (uint32_t)u0, u_stop);
    g += u_stop - u0;
    u0 = 0;
    // the next prefix: the last position below me - 1 steps up, those after it follow
    int up = 0;
    bool found = false;
#pragma unroll
    for (int l = DP - 1; l >= 0; --l)
      if (!found && p[l] < me - 1) {
        found = true;
        up = p[l] + 1;
#pragma unroll
        for (int j = l; j < DP; ++j) p[j] = up;
      }
  }
}

// V groups of 64 parents from uc (all but the last group whole)
template <int V>
struct LaneParents {
  uint32_t first, last;  // the lane's parent in groups 0 and V - 1
  bool in;               // its parent in the last group is one of the sweep's
  __device__ __forceinline__ LaneParents(uint32_t uc, uint32_t u_stop) {
    first = uc + (threadIdx.x & 63u);
    const uint32_t l = first + 64u * (V - 1);
    in = l < u_stop;
    last = in ? l : u_stop - 1u;
  }
  __device__ __forceinline__ uint32_t u(int i) const { return i < V - 1 ? first + 64u * i : last; }
};

struct DescendArgs {
  const float* qk;
  float* qout;
  const uint32_t* ins;
  uint32_t n4;
  int me;
  float invk, scale;
};

template <int V, int NA>
__device__ __forceinline__ void descend_streams(const DescendArgs& x, const ChildBlock& b, const LaneParents<V>& lp, int a0,
                                                float (&acc)[V]) {
  float q[NA][V];
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    const float* s = x.qk + rl64(b.sb, a0 + k);
#pragma unroll
    for (int i = 0; i < V; ++i) q[k][i] = at_bytes(s, lp.u(i) * 4u);
  }
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    const float c = (float)rl(b.cnt, a0 + k);
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = fmaf(q[k][i], c, acc[i]);
  }
}

// FIRST: a0 is last(P), of which the children hold P's copies too
template <int V, int NA, bool FIRST>
__device__ __forceinline__ void descend_tail(const DescendArgs& x, const ChildBlock& b, const LaneParents<V>& lp, int a0,
                                             float (&acc)[V]) {
  uint32_t w[NA][V];
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    const uint32_t* t = x.ins + (size_t)((uint32_t)(a0 + k) * x.n4 + b.toff);
#pragma unroll
    for (int i = 0; i < V; ++i) w[k][i] = at_bytes(t, lp.u(i) * 4u);
  }
  const float* qt = x.qk + b.tail;
  float q[NA][V];
#pragma unroll
  for (int k = 0; k < NA; ++k)
#pragma unroll
    for (int i = 0; i < V; ++i) q[k][i] = at_bytes(qt, w[k][i] & kInsertMask);
#pragma unroll
  for (int k = 0; k < NA; ++k)
#pragma unroll
    for (int i = 0; i < V; ++i) {
      uint32_t c = w[k][i] >> kInsertShift;
      if (FIRST && k == 0) c += rl(b.cnt, a0) - 1u;
      acc[i] = fmaf(q[k][i], (float)c, acc[i]);
    }
}

template <int V>
__device__ __forceinline__ void descend_groups(const DescendArgs& x, const ChildBlock& b, uint32_t uc, uint32_t u_stop) {
  const LaneParents<V> lp(uc, u_stop);
  float acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = 0.f;
  constexpr int kS = V == 4 ? 4 : 8;   // modes whose loads are issued together
  constexpr int kT = V == 4 ? 4 : 8;
  int a = 0;
  for (; a + kS <= b.lastP; a += kS) descend_streams<V, kS>(x, b, lp, a, acc);
  if (kS > 4 && a + 4 <= b.lastP) { descend_streams<V, 4>(x, b, lp, a, acc); a += 4; }
  if (a + 2 <= b.lastP) { descend_streams<V, 2>(x, b, lp, a, acc); a += 2; }
  if (a < b.lastP) { descend_streams<V, 1>(x, b, lp, a, acc); ++a; }
  if (a + kT <= x.me) { descend_tail<V, kT, true>(x, b, lp, a, acc); a += kT; }
  else { descend_tail<V, 1, true>(x, b, lp, a, acc); ++a; }
  for (; a + kT <= x.me; a += kT) descend_tail<V, kT, false>(x, b, lp, a, acc);
  if (kT > 4 && a + 4 <= x.me) { descend_tail<V, 4, false>(x, b, lp, a, acc); a += 4; }
  if (a + 2 <= x.me) { descend_tail<V, 2, false>(x, b, lp, a, acc); a += 2; }
  if (a < x.me) descend_tail<V, 1, false>(x, b, lp, a, acc);
  float* o = x.qout + b.CBp;
#pragma unroll
  for (int i = 0; i < V; ++i)
    if (i < V - 1 || lp.in)
      *reinterpret_cast<float*>(reinterpret_cast<char*>(o) + lp.u(i) * 4u) = (acc[i] * x.invk) * x.scale;
}

// What bounds it: the block walk with offsets computed per lane and mode (descend_block.hpp) spent 42 %
// of the VALU cycles and 74 % of the L1's, most of the former on blocks set up 64 at a time of which a
// wave used few, and on ~25 instructions per mode above last(P); 8-byte loads of two parents a lane
// cost the L1 as much as 16-byte ones. Here a block costs ~15 instructions a prefix position, a mode
// and 64 parents two to four, and every load is 4 bytes a lane. n=10 m=24: 1198 -> 463 us (10 -> 9) and
// 462 -> 149 (9 -> 8); n=11 m=32: 32.6 -> 19.1 ms (11 -> 10). What is left at those sizes is the L1's
// rate (three 4-byte accesses an edge) and, at n=11, reads beyond the L2.
template <int DP>
__global__ __launch_bounds__(kBlockThreads) void k_descend_insert(const uint64_t* __restrict__ cg,
                                                                  const uint32_t* __restrict__ ins, int me,
                                                                  const float* __restrict__ qk_all, uint64_t Sk,
                                                                  float* __restrict__ qout_all, uint64_t Sp,
                                                                  uint64_t per_wave, float scale, uint32_t xcd_chunk) {
  const int64_t row = blockIdx.y;
  const int wv = (int)rfl(threadIdx.x >> 6);
  const uint64_t g = uniform_u64(((uint64_t)xcd_chunk_index(blockIdx.x, xcd_chunk, gridDim.x) * kWaves + wv) * per_wave);
  const DescendArgs x{qk_all + (size_t)row * Sk, qout_all + (size_t)row * Sp, ins, (uint32_t)cg[4 * (me + 1)], me,
                      1.f / (float)(DP + 5), scale};
  child_walk<DP>(cg, me, Sp, per_wave, g, [&](const ChildBlock& b, uint32_t uc, uint32_t u_stop) {
    for (; uc + 192u < u_stop; uc += 256u) descend_groups<4>(x, b, uc, u_stop);
    if (uc + 64u < u_stop) {
      descend_groups<2>(x, b, uc, u_stop);
      uc += 128u;
    }
    if (uc < u_stop) descend_groups<1>(x, b, uc, u_stop);
  });
}

}  // namespace slos
