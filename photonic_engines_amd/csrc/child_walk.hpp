// Pulls over children through the insert table (block_index.hpp: insert_word), for multiset spaces of
// at most 41 modes and parent layers D = K - 1 = DP + 4, DP = 0..8: one step of the uniform-loss
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
// The blocks of the last eight modes (last(P) >= X) would hold 1 to 330 parents, and they are the most:
// those of one shorter prefix P' make one block, whose suffixes are the 5-tuples from
// max(X, last(P')) on (up to 792 parents), with the same formulas for a prefix one shorter.
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
  uint64_t sb;      // lane a < x0: base of mode a's child stream, at u = 0
  uint64_t tail;    // child of index 0 of the insert table
  uint32_t cnt;     // lane a: 1 + copies of a in the prefix
  uint32_t tab;     // insert-table word of mode 0 and the block's first suffix (modulo 2^32), and the
  uint32_t pitch;   // words from mode to mode
  int x0;           // smallest mode of the suffixes: modes from here on go through the table
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
  if constexpr (DP == 0) {  // no prefix: one block, every mode through the table
    sweep(ChildBlock{0, 0, 0, 1u, 0u, (uint32_t)Sp, 0}, (uint32_t)g, (uint32_t)g_end);
    return;
  }
  constexpr int D1 = DP > 0 ? DP : 1;
  uint64_t row[DP + 1];  // lane x: cg[K - l][x + 1]
#pragma unroll
  for (int l = 0; l <= DP; ++l) row[l] = lane < me ? cg[(K - l) * W + lane + 1] : 0u;
  const uint32_t c4 = lane < me ? (uint32_t)cg[4 * W + lane] : 0u;
  const uint32_t c5 = lane < me ? (uint32_t)cg[5 * W + lane] : 0u;
  const int X = insert_from(me);
  const uint64_t cK = cg[K * W], n5 = cg[5 * W], n6X = cg[6 * W + X];
  const uint32_t n4 = (uint32_t)cg[4 * W], n5X = rl(c5, X);
  // the prefix of parent g: position l is the number of modes x >= its predecessor that g's rank
  // among the tuples from there on has passed
  int p[D1];
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
      if (l == DP - 1 && p[l] >= X) {  // inside a merged block: from its first suffix
        const int x0 = lo > X ? lo : X;
        u0 += rl(c5, x0) - rl(c5, p[l]);
        p[l] = x0;
      }
      top = at - rl64(row[l + 1], p[l]);
      lo = p[l];
    }
  }
  while (g < g_end) {
    ChildBlock b;
    // suffixes of 5 positions from X on, else of 4 (p[D1 - 1] >= X: the first of the run it begins)
    const bool merged = p[D1 - 1] >= X;
    b.x0 = p[D1 - 1];
    const uint32_t L = rl(merged ? c5 : c4, b.x0);
    b.CBp = g - u0;
    uint64_t lower = cK, own = row[0];  // lane a: lower - own = its stream's base
    uint64_t tail = cK;
    b.cnt = 1u;
#pragma unroll
    for (int l = 0; l < DP; ++l) {
      if (l == DP - 1 && merged) break;
      const uint64_t s_le = rl64(row[l], p[l]), s_gt = rl64(row[l + 1], p[l]);
      const bool le = p[l] <= lane;
      lower -= le ? s_le : s_gt;
      own = le ? row[l + 1] : own;
      b.cnt += p[l] == lane ? 1u : 0u;
      tail -= s_le;
    }
    b.sb = lower - own - (uint64_t)L;
    b.tail = tail - (merged ? n6X : n5);
    b.pitch = merged ? n5X : n4;
    b.tab = merged ? n4 * (uint32_t)me - (uint32_t)X * n5X + (n5X - L) : n4 - L;
    const uint64_t left = g_end - g;
    const uint32_t u_stop = (uint64_t)L - u0 < left ? L : (uint32_t)(u0 + left);
    sweep(b, (uint32_t)u0, u_stop);
    g += u_stop - u0;
    u0 = 0;
    // the next prefix: the last position below me - 1 steps up, those after it follow
    bool found = false;
#pragma unroll
    for (int l = DP - 1; l >= 0; --l) {
      if (!found && p[l] < me - 1 && !(l == DP - 1 && merged)) {
        found = true;
        const int up = p[l] + 1;
#pragma unroll
        for (int j = l; j < DP; ++j) p[j] = up;
      }
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
    const uint32_t* t = x.ins + (size_t)((uint32_t)(a0 + k) * b.pitch + b.tab);
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
  for (; a + kS <= b.x0; a += kS) descend_streams<V, kS>(x, b, lp, a, acc);
  if (kS > 4 && a + 4 <= b.x0) { descend_streams<V, 4>(x, b, lp, a, acc); a += 4; }
  if (a + 2 <= b.x0) { descend_streams<V, 2>(x, b, lp, a, acc); a += 2; }
  if (a < b.x0) { descend_streams<V, 1>(x, b, lp, a, acc); ++a; }
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
// and 64 parents two to four, and every load is 4 bytes a lane. n=10 m=24: 1198 -> 413 us (10 -> 9) and
// 462 -> 127 (9 -> 8); n=11 m=32: 32.6 -> 18.9 ms (11 -> 10). What is left at those sizes is the L1's
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
  const DescendArgs x{qk_all + (size_t)row * Sk, qout_all + (size_t)row * Sp, ins, me,
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

// ------------------------------------------------------------------------------------------
// Adjoint of one forward layer (the backward of the recurrence, photonic_engines/slos/kernel.py:63-80,
// as a pull over children): for every parent t of layer K-1 and every mode a, the child t + e_a is an
// edge with coefficient U[a, col], so
//   grad_prev[t] = sum_a conj(U[a, col]) g_K[t + e_a]          (ascending a)
//   dL/dU[a, col] += sum_t conj(psi_{K-1}[t]) g_K[t + e_a].
// The U-gradient is kept per lane and mode in registers (the mode loop is unrolled to ME), summed over
// a wave's lanes and the work group's waves in FP64 and written as one FP64 partial per work group and
// mode (k_reduce_gu sums those). No atomics.
// ------------------------------------------------------------------------------------------
struct AdjointArgs {
  const float2* gk;    // g_K (child layer)
  const float2* psi;   // psi_{K-1} (parent layer)
  float2* gout;        // grad_prev (parent layer), or nullptr
  const uint32_t* ins;
  int me;
  uint32_t ure, uim;   // lane a: U[a, col]
};

template <int V, int ME>
__device__ __forceinline__ void adjoint_groups(const AdjointArgs& x, const ChildBlock& b, uint32_t uc, uint32_t u_stop,
                                               float2 (&gacc)[ME]) {
  const LaneParents<V> lp(uc, u_stop);
  const float2* pb = x.psi + b.CBp;
  float2 ps[V];
#pragma unroll
  for (int i = 0; i < V; ++i) ps[i] = at_bytes(pb, lp.u(i) * 8u);
  if (!lp.in) ps[V - 1] = make_float2(0.f, 0.f);  // lanes past the block add nothing
  float gr[V], gi[V];
#pragma unroll
  for (int i = 0; i < V; ++i) gr[i] = gi[i] = 0.f;
  const float2* gt = x.gk + b.tail;
  constexpr int kStep = V == 1 ? 8 : 4;  // modes whose loads are issued together
#pragma unroll
  for (int a0 = 0; a0 < ME; a0 += kStep) {
    if (a0 >= x.me) break;
    // (opaque here: else the compiler reads all modes' coefficients and bases into scalar registers
    // ahead of the loop over the block's parents, and spills them)
    uint32_t ure = x.ure, uim = x.uim, tab = b.tab;
    int x0 = b.x0, me = x.me;
    uint32_t slo = (uint32_t)b.sb, shi = (uint32_t)(b.sb >> 32);
    asm volatile("" : "+v"(ure), "+v"(uim), "+v"(slo), "+v"(shi), "+s"(tab), "+s"(x0), "+s"(me));
    __builtin_amdgcn_sched_barrier(0);
    uint32_t w[kStep][V];
#pragma unroll
    for (int k = 0; k < kStep; ++k)
      if (a0 + k >= x0 && a0 + k < me) {
        const uint32_t* t = x.ins + (size_t)((uint32_t)(a0 + k) * b.pitch + tab);
#pragma unroll
        for (int i = 0; i < V; ++i) w[k][i] = at_bytes(t, lp.u(i) * 4u);
      }
    float2 gv[kStep][V];
#pragma unroll
    for (int k = 0; k < kStep; ++k) {
      if (a0 + k < x0) {
        const float2* s = x.gk + (((uint64_t)rl(shi, a0 + k) << 32) | rl(slo, a0 + k));
#pragma unroll
        for (int i = 0; i < V; ++i) gv[k][i] = at_bytes(s, lp.u(i) * 8u);
      } else if (a0 + k < me) {
#pragma unroll
        for (int i = 0; i < V; ++i) gv[k][i] = at_bytes(gt, (w[k][i] & kInsertMask) * 2u);
      }
    }
#pragma unroll
    for (int k = 0; k < kStep; ++k) {
      const int a = a0 + k;
      if (a < me) {
        const float ur = __builtin_bit_cast(float, rl(ure, a)), ui = __builtin_bit_cast(float, rl(uim, a));
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float2 v = gv[k][i];
          gr[i] = fmaf(ur, v.x, gr[i]);  // conj(u) * g
          gr[i] = fmaf(ui, v.y, gr[i]);
          gi[i] = fmaf(ur, v.y, gi[i]);
          gi[i] = fmaf(-ui, v.x, gi[i]);
          gacc[a].x = fmaf(ps[i].x, v.x, gacc[a].x);  // conj(psi) * g
          gacc[a].x = fmaf(ps[i].y, v.y, gacc[a].x);
          gacc[a].y = fmaf(ps[i].x, v.y, gacc[a].y);
          gacc[a].y = fmaf(-ps[i].y, v.x, gacc[a].y);
        }
      }
    }
  }
  if (x.gout) {
    float2* o = x.gout + b.CBp;
#pragma unroll
    for (int i = 0; i < V; ++i)
      if (i < V - 1 || lp.in)
        *reinterpret_cast<float2*>(reinterpret_cast<char*>(o) + lp.u(i) * 8u) = make_float2(gr[i], gi[i]);
  }
}

// The lanes' sums of ME modes, added in FP64 to wsum (the work group's waves in order); rows of 65
// floats in LDS, two lanes a row. `tr`: 32 rows a wave.
constexpr int kAdjRows = 32, kAdjPitch = 65;
// parents a wave takes at a time, the work group's waves in turn (a stretch of short blocks, which
// costs a wave many walk steps, is shared by the four)
constexpr uint32_t kAdjChunk = 128;

template <int ME>
__device__ __forceinline__ void adjoint_reduce(const float2 (&gacc)[ME], float* tr, double* wsum) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int a0 = 0; a0 < ME; a0 += kAdjRows / 2) {
    wave_sync();
#pragma unroll
    for (int a = 0; a < kAdjRows / 2; ++a) {
      tr[(2 * a) * kAdjPitch + lane] = gacc[a0 + a].x;
      tr[(2 * a + 1) * kAdjPitch + lane] = gacc[a0 + a].y;
    }
    wave_sync();
    const float* r = tr + (lane >> 1) * kAdjPitch + (lane & 1) * 32;
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < 32; ++j) s += (double)r[j];
    s += __shfl_xor(s, 1, 64);
    if (!(lane & 1)) wsum[2 * a0 + (lane >> 1)] = s;
  }
}

// What bounds it: the earlier form (offsets computed, 64 blocks set up at a time in LDS) issued 768 FP64
// shuffles a wave for the sums over its lanes and spilled 153 scalars; a wave that met a stretch of
// one-parent blocks ran several times as long as the others. Here the sums go through LDS rows
// (adjoint_reduce), short blocks are merged (child_walk) and shared by the work group's waves, and the
// stretch in question (the last parents) is launched first. 8 -> 7 at n=8 m=24 (2.0M parents) 255 ->
// 119 us with its reduction, 7 -> 6 100 -> 55; 200k parents of n=11 m=8 264 -> 130. What is left is the
// latency of two dependent loads per four modes, at four waves a SIMD.
template <int DP, int ME>
__global__ __launch_bounds__(kBlockThreads, 4) void k_adjoint_insert(const uint64_t* __restrict__ cg,
                                                                  const uint32_t* __restrict__ ins, int me, int m,
                                                                  int col, const float2* __restrict__ U,
                                                                  const float2* __restrict__ psi_all,
                                                                  const float2* __restrict__ gk_all, uint64_t Sk,
                                                                  float2* __restrict__ gout_all, uint64_t Sp,
                                                                  uint64_t per_wave, uint32_t xcd_chunk,
                                                                  double2* __restrict__ partial) {
  __shared__ float tr[kWaves][kAdjRows * kAdjPitch];
  __shared__ double wsum[kWaves][2 * ME];
  const int64_t row = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wv = (int)rfl(threadIdx.x >> 6);
  const uint64_t g = uniform_u64((uint64_t)(gridDim.x - 1u - xcd_chunk_index(blockIdx.x, xcd_chunk, gridDim.x)) * kWaves * per_wave);
  const float2 ua = lane < me ? U[(size_t)row * m * m + (size_t)lane * m + col] : make_float2(0.f, 0.f);
  const AdjointArgs x{gk_all + (size_t)row * Sk, psi_all + (size_t)row * Sp, gout_all ? gout_all + (size_t)row * Sp : nullptr,
                      ins, me, __builtin_bit_cast(uint32_t, ua.x),
                      __builtin_bit_cast(uint32_t, ua.y)};
  float2 gacc[ME];
#pragma unroll
  for (int a = 0; a < ME; ++a) gacc[a] = make_float2(0.f, 0.f);
  for (uint32_t c = (uint32_t)wv * kAdjChunk; c < kWaves * per_wave; c += kWaves * kAdjChunk)
    child_walk<DP>(cg, me, Sp, kAdjChunk, g + c, [&](const ChildBlock& b, uint32_t uc, uint32_t u_stop) {
      for (; uc + 64u < u_stop; uc += 128u) adjoint_groups<2>(x, b, uc, u_stop, gacc);
      if (uc < u_stop) adjoint_groups<1>(x, b, uc, u_stop, gacc);
    });
  adjoint_reduce<ME>(gacc, tr[wv], wsum[wv]);
  __syncthreads();
  for (int a = threadIdx.x; a < 2 * me; a += blockDim.x) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s += wsum[w][a];
    reinterpret_cast<double*>(partial + ((size_t)row * gridDim.x + blockIdx.x) * me)[a] = s;
  }
}

}  // namespace slos
