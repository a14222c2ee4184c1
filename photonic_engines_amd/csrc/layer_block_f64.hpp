// complex128 forms of the block kernel and of the group-order kernel (layer_block.hpp): the same
// blocks, prefix streams, suffix tables and work items, with complex128 layers and FP64 sums in the
// same order.
//
// What bounds them: the loads. A lane takes one child, whose parents are 16-byte values, so every
// stream and every suffix parent is one full-rate 16-byte load a lane (17 clocks of a CU's cache for a
// wave), 8 to 10 of them a child; the FP64 multiply-adds (40) run at the rate of FP32 ones. The
// thread-per-state kernel, which they replace on layers of 2M states or more (use_blocks in slos.hip),
// spends its time on each state's unrank and rank arithmetic: layer 10 of n = 10, m = 20 took 643 us
// there, 194 us here, layer 11 of n = 11, m = 22 4.48 and 1.46 ms.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layer_block.hpp"

namespace slos {

// a row of the suffix table (SufRow) with an FP64 coefficient, 32 bytes
struct __attribute__((aligned(16))) SufRow64 {
  double re, im;
  uint32_t t0, t1, pad0, pad1;
};
constexpr size_t kBlockStaticLds64 = kSufRows * sizeof(SufRow64) + kNormRows * kNormCodes * sizeof(float);

__device__ __forceinline__ void cmac64(double2& a, double2 u, double2 v) {
  a.x = fma(u.x, v.x, a.x);
  a.x = fma(-u.y, v.y, a.x);
  a.y = fma(u.x, v.y, a.y);
  a.y = fma(u.y, v.x, a.y);
}

// KIND 0: raw complex128, 1: float64 probabilities, 2: scaled complex128 amplitudes; f: prod t_j!, which
// divides K!. Up to 13 photons every such number and every product on the way to it is exact in float: the odd
// part of 13! is 6,081,075 < 2^24 (that of 14! is not below it).
constexpr int kExactFactorials = 13;
template <int KIND>
__device__ __forceinline__ void store64(void* out, uint64_t i, double2 v, float f, double scale, unsigned flags) {
  if constexpr (KIND == 0) {
    static_cast<double2*>(out)[i] = v;
  } else {
    const double re = v.x * scale, im = v.y * scale;
    if constexpr (KIND == 1) {
      static_cast<double*>(out)[i] = (re * re + im * im) * (double)f;
    } else {
      const double s = (flags & 2u) ? sqrt((double)f) : 1.0;
      static_cast<double2*>(out)[i] = make_double2(re * s, im * s);
    }
  }
}

struct BlockLayerF64 {
  BlockLayer l;       // (U and scale unused)
  const double2* U;   // [B][m][m]
  double scale;
};

// Children [u0, u_stop) of one block with its first NS stream slots, 64 a step
template <int KIND, int MAXD, int NS, int SUF>
__device__ __forceinline__ void block_children64(const uint32_t* bj, const double2* par, const double2* lp,
                                                 const TupleWordT<SUF>* tb, void* out, uint64_t CB, const SufRow64* rows,
                                                 const float* rn, uint32_t C0, uint32_t u0, uint32_t u_stop, int lane,
                                                 float fQ, int lastrun, int skip0, int lo, int multiset, double scale,
                                                 unsigned flags) {
  constexpr int kBaseW = 8 + (MAXD + 3) / 4;
  auto word = [&](int f) { return rfl(bj[f * kBlockBatch]); };
  const double2* sp[NS];
  double2 coef[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const SufRow64 r = rows[(word(8 + s / 4) >> (8 * (s % 4))) & 0xffu];
    coef[s] = make_double2(r.re, r.im);
    sp[s] = par + ((uint64_t)word(kBaseW + 2 * s) | ((uint64_t)word(kBaseW + 2 * s + 1) << 32));
  }
  for (uint32_t uc = u0; uc < u_stop; uc += 64u) {
    const uint32_t ur = uc + (uint32_t)lane;
    const bool in = ur < u_stop;
    const uint32_t u = in ? ur : u_stop - 1u;
    const TupleWordT<SUF> w = tb[u];
    double2 sv[NS], lv[SUF], lc[SUF];
#pragma unroll
    for (int s = 0; s < NS; ++s) sv[s] = at_bytes(sp[s], u * 16u);
    uint32_t off[SUF];
    suffix_edges_of<SUF>(rows, C0, skip0, lo, w, lc, off);
#pragma unroll
    for (int j = 0; j < SUF; ++j) lv[j] = at_bytes(lp, off[j]);
    double2 acc = make_double2(0.0, 0.0);
#pragma unroll
    for (int s = 0; s < NS; ++s) cmac64(acc, coef[s], sv[s]);
#pragma unroll
    for (int j = 0; j < SUF; ++j) cmac64(acc, lc[j], lv[j]);
    float f = 1.f;
    if (KIND != 0 && multiset) {
      const uint32_t row = (skip0 && (int)((uint32_t)w & 0xffu) == lo) ? (uint32_t)lastrun + 1u : 0u;
      f = fQ * rn[row * (1u << (SUF - 1)) + tuple_code<SUF>(w)];
    }
    if (in) store64<KIND>(out, CB + u, acc, f, scale, flags);
  }
}

// a wave's children [g, g + per_wave), block by block (block_wave of layer_block.hpp)
template <int KIND, int MAXD, int SUF>
__global__ __launch_bounds__(kBlockThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_layer_block_f64(
    const uint64_t* __restrict__ cg_t, const int* __restrict__ lo_t, const void* __restrict__ tuples, int me, int stride,
    int multiset, const double2* __restrict__ par_all, void* __restrict__ out_all, BlockLayerF64 p) {
  static_assert(MAXD + SUF <= kExactFactorials, "store64 takes prod t_j! in float");
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ SufRow64 rows[kSufRows];
  __shared__ float rn[kNormRows * kNormCodes];
  const BlockLayer& a = p.l;
  const int K = a.K, d = K - SUF;
  const int ncg = (K + 1) * stride;
  uint64_t* cg_l = reinterpret_cast<uint64_t*>(smem);
  int* lo_l = reinterpret_cast<int*>(cg_l + ncg);
  int64_t b;
  const uint32_t bid = batch_item(a.rows, a.row_wgs, a.xcd_chunk, &b);
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg_l[i] = cg_t[i];
  for (int i = threadIdx.x; i < me; i += blockDim.x) lo_l[i] = lo_t[i];
  fill_suffix_rows<SUF>(rows, p.U + b * a.us.B + a.col * a.us.C, a.us.R, a.m, cg_t, stride, me);
  fill_norm_rows<SUF>(rn);
  __syncthreads();
  const BlockTables tg{cg_t, lo_t, tuples, me, stride, multiset};  // global: scalar loads
  const BlockTables tl{cg_l, lo_l, tuples, me, stride, multiset};  // LDS: per-lane lookups
  const int lane = threadIdx.x & 63;
  const int wv = (int)rfl(threadIdx.x >> 6);
  uint64_t g = uniform_u64(((uint64_t)bid * kWaves + wv) * a.per_wave);
  if (g >= a.S) return;
  const uint64_t g_end = (g + a.per_wave < a.S) ? g + a.per_wave : a.S;
  uint32_t* tbl = reinterpret_cast<uint32_t*>(smem + block_table_offset(K, me)) +
                  (size_t)wv * kBlockBatch * block_words(MAXD);
  const double2* par = par_all + (size_t)b * a.S_par;
  void* out = static_cast<char*>(out_all) + (size_t)b * a.S * (KIND == 1 ? 8 : 16);
  const auto* words = static_cast<const TupleWordT<SUF>*>(tuples);
  const uint32_t C0 = (uint32_t)cg_t[(SUF - 1) * stride];
  uint64_t r = 0, u0 = 0;
  bool seek = true;
  while (g < g_end) {
    if (seek) {
      int q[MAXD];
      u0 = unrank_prefix<MAXD>(tg, K, d, g, q);
      r = prefix_rank<MAXD>(tg, d, q);
    }
    const uint64_t g0 = g;
    if (r >= a.S_pre) break;  // cannot happen while g < S; keeps the loop bounded regardless
    fill_block_table<MAXD, SUF>(tl, K, d, r, a.S_pre, tbl, lane);
    const int nb = (int)((a.S_pre - r < kBlockBatch) ? a.S_pre - r : kBlockBatch);
    for (int j = 0; j < nb && g < g_end; ++j) {
      const uint32_t* bj = tbl + j;
      auto word = [&](int f) { return rfl(bj[f * kBlockBatch]); };
      const uint32_t L = word(4);
      if (L == 0) continue;  // empty block (set masks only)
      const uint64_t CB = (uint64_t)word(0) | ((uint64_t)word(1) << 32);
      const uint64_t LBp = (uint64_t)word(2) | ((uint64_t)word(3) << 32);
      const uint32_t w6 = word(6);
      const int nact = (int)(w6 >> 24);
      const float fQ = __builtin_bit_cast(float, word(7));
      const uint64_t avail = g_end - g;
      const uint32_t u_stop = (uint32_t)(((uint64_t)L - u0 < avail) ? (uint64_t)L : u0 + avail);
      auto children = [&](auto ns) {
        block_children64<KIND, MAXD, decltype(ns)::value, SUF>(
            bj, par, par + LBp, words + word(5), out, CB, rows, rn, C0, (uint32_t)u0, u_stop, lane, fQ,
            (int)((w6 >> 16) & 0xffu), (int)((w6 >> 8) & 1u), (int)(w6 & 0xffu), multiset, p.scale, a.flags);
      };
      group_dispatch<MAXD>((uint32_t)nact, children);
      g += u_stop - u0;
      u0 = 0;
    }
    r += kBlockBatch;
    // 64 prefixes without a child: a set mask's, whose runs of them are thousands long. On to the next child's
    // block.
    seek = g == g0;
  }
}

// ------------------------------------------------------------------------------------------
// group order (k_layer_group): a wave takes a group R and a range of suffix positions; each 64-child
// step reads the shared first stream, the tuple words and the local-parent offsets once for all of
// the group's blocks. Group table: CB(2) LBp(2) w6 fQ, base and mode of 6 slots (3 each), toff
// ------------------------------------------------------------------------------------------
constexpr int kGroupWords64 = 28;
__host__ __device__ inline size_t group_dyn_lds64(int K, int me) {
  return group_table_offset(K, me) + (size_t)kWaves * me * kGroupWords64 * 4;
}

template <int NS, int KIND>
__device__ __forceinline__ void group_block64(const uint32_t* bw, const double2* par, double2 v0, const double2 (&lc)[5],
                                              const uint32_t (&off)[5], uint32_t u, bool in, uint32_t code, bool lead,
                                              const SufRow64* rows, const float* rn, double scale, void* out) {
  const uint64_t CB = (uint64_t)rfl(bw[0]) | ((uint64_t)rfl(bw[1]) << 32);
  const uint64_t LBp = (uint64_t)rfl(bw[2]) | ((uint64_t)rfl(bw[3]) << 32);
  const uint32_t w6 = bw[4];
  double2 sv[NS], coef[NS], lv[5];
  sv[0] = v0;
#pragma unroll
  for (int s = 1; s < NS; ++s) {
    const uint64_t base = (uint64_t)rfl(bw[6 + 3 * s]) | ((uint64_t)rfl(bw[7 + 3 * s]) << 32);
    sv[s] = at_bytes(par + base, u * 16u);
  }
  const double2* lp = par + LBp;
#pragma unroll
  for (int j = 0; j < 5; ++j) lv[j] = at_bytes(lp, off[j]);
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const SufRow64 r = rows[bw[8 + 3 * s]];
    coef[s] = make_double2(r.re, r.im);
  }
  double2 acc = make_double2(0.0, 0.0);
#pragma unroll
  for (int s = 0; s < NS; ++s) cmac64(acc, coef[s], sv[s]);
#pragma unroll
  for (int j = 0; j < 5; ++j) cmac64(acc, lc[j], lv[j]);
  float f = 1.f;
  if constexpr (KIND != 0)
    f = __builtin_bit_cast(float, bw[5]) * rn[(lead ? ((w6 >> 16) & 0xffu) + 1u : 0u) * 16u + code];
  if (in) store64<KIND>(out, CB + u, acc, f, scale, 0u);
}

template <int MAXD, int KIND>
__global__ __launch_bounds__(kBlockThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_layer_group_f64(
    const uint64_t* __restrict__ cg_t, const int* __restrict__ lo_t, const uint64_t* __restrict__ tuples5, int me,
    int stride, const double2* __restrict__ par_all, void* __restrict__ out_all, BlockLayerF64 p,
    const uint4* __restrict__ items, uint32_t n_items) {
  static_assert(MAXD >= 2 && MAXD <= 6, "group table holds 6 stream slots");
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ SufRow64 rows[kSufRows];
  __shared__ float rn[kNormRows * kNormCodes];
  const BlockLayer& a = p.l;
  const int K = a.K, d = K - 5;
  const int ncg = (K + 1) * stride;
  uint64_t* cg_l = reinterpret_cast<uint64_t*>(smem);
  int* lo_l = reinterpret_cast<int*>(cg_l + ncg);
  int64_t b;
  const uint32_t bid = batch_item(a.rows, a.row_wgs, a.xcd_chunk, &b);
  for (int i = threadIdx.x; i < ncg; i += blockDim.x) cg_l[i] = cg_t[i];
  for (int i = threadIdx.x; i < me; i += blockDim.x) lo_l[i] = lo_t[i];
  fill_suffix_rows<5>(rows, p.U + b * a.us.B + a.col * a.us.C, a.us.R, a.m, cg_t, stride, me);
  fill_norm_rows<5>(rn);
  __syncthreads();
  const int wv = (int)rfl(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const uint32_t item = bid * kWaves + (uint32_t)wv;
  if (item >= n_items) return;
  const uint4 it = items[item];
  const uint32_t r = rfl(it.x), u_b = rfl(it.y), u_e = rfl(it.z);
  const BlockTables tl{cg_l, lo_l, tuples5, me, stride, 1};
  const SpaceView sv{cg_l, lo_l, me, stride};
  int R[MAXD];
  sv.unrank(r, d - 1, R);
  const int G = (int)rfl((uint32_t)R[0]) + 1;  // blocks (a, R), a = 0..R_0 (lo[x] = x)
  uint32_t* tbl = reinterpret_cast<uint32_t*>(smem + group_table_offset(K, me)) + (size_t)wv * me * kGroupWords64;
  const double2* par = par_all + (size_t)b * a.S_par;
  void* out = static_cast<char*>(out_all) + (size_t)b * a.S * (KIND == 0 ? 16 : 8);
  if (lane < G) {
    int q[MAXD];
    q[0] = lane;
#pragma unroll
    for (int i = 1; i < MAXD; ++i) q[i] = i < d ? R[i - 1] : 0;
    BlockInfo bi;
    Streams<MAXD> st;
    block_info<MAXD, 5>(tl, K, d, q, bi, st);
    uint32_t* col = tbl + lane * kGroupWords64;
    col[0] = (uint32_t)bi.CB;
    col[1] = (uint32_t)(bi.CB >> 32);
    col[2] = (uint32_t)bi.LBp;
    col[3] = (uint32_t)(bi.LBp >> 32);
    col[5] = __builtin_bit_cast(uint32_t, bi.fQ);
    // slot 0, then the other active streams in ascending position, then slot 0's base, no edge
#pragma unroll
    for (int t = 0; t < 6; ++t) {
      col[6 + 3 * t] = (uint32_t)st.base[0];
      col[7 + 3 * t] = (uint32_t)(st.base[0] >> 32);
      col[8 + 3 * t] = t == 0 ? (uint32_t)st.mode[0] : (uint32_t)kNoEdgeRow;
    }
    uint32_t nact = 1;
#pragma unroll
    for (int s = 1; s < MAXD; ++s)
      if (st.active[s]) {
        col[6 + 3 * nact] = (uint32_t)st.base[s];
        col[7 + 3 * nact] = (uint32_t)(st.base[s] >> 32);
        col[8 + 3 * nact] = (uint32_t)st.mode[s];
        ++nact;
      }
    col[4] = (uint32_t)bi.lo | ((uint32_t)bi.skip0 << 8) | ((uint32_t)bi.lastrun << 16) | (nact << 24);
    col[24] = bi.toff;
  }
  wave_sync();
  // shared by the group: the parent block R (slot 0's base), the tuple range, lo, skip0
  const uint64_t base0 = (uint64_t)rfl(tbl[6]) | ((uint64_t)rfl(tbl[7]) << 32);
  const uint32_t toff = rfl(tbl[24]);
  const uint32_t w60 = rfl(tbl[4]);
  const int lo = (int)(w60 & 0xffu), skip0 = (int)((w60 >> 8) & 1u);
  const double2* sp0 = par + base0;
  const uint64_t* tb = tuples5 + toff;
  const uint32_t C0 = (uint32_t)cg_t[4 * stride];
  for (uint32_t uc = u_b; uc < u_e; uc += 64u) {
    const uint32_t ur = uc + (uint32_t)lane;
    const bool in = ur < u_e;
    const uint32_t u = in ? ur : u_e - 1u;
    const uint64_t w = tb[u];
    const double2 v0 = at_bytes(sp0, u * 16u);
    double2 lc[5];
    uint32_t off[5];
    suffix_edges_of<5>(rows, C0, skip0, lo, w, lc, off);
    const uint32_t code = tuple_code<5>(w);
    const bool lead = skip0 && (int)((uint32_t)w & 0xffu) == lo;
    for (int g = 0; g < G; ++g) {
      const uint32_t* bw = tbl + g * kGroupWords64;
      group_dispatch<MAXD>(rfl(bw[4]) >> 24, [&](auto ns) {
        group_block64<decltype(ns)::value, KIND>(bw, par, v0, lc, off, u, in, code, lead, rows, rn, p.scale, out);
      });
    }
  }
}

}  // namespace slos
