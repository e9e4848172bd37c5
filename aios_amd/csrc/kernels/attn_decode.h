// Split-K flash-decode attention core (device code of attention.hip's decode kernel).  See
// attention.hip for the design.
#pragma once
#include "../common.h"
#include "../ops.h"
#include "gemm_common.h"

#include <algorithm>
#include <cstdlib>

#ifndef AIOS_ATTN_PROBES
#define AIOS_ATTN_PROBES 0
#endif

namespace aios {

// the two values of a bf16 pair
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// ... each halved: one from the exponent, down to 0 (values below 2^-125 lose it, beside a largest of 1)
__device__ __forceinline__ uint32_t bf16x2_half(uint32_t w) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2, w), u16x2{0x80, 0x80}));
}

__device__ __forceinline__ void st_wt(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_wt(const float* p) {
  return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// op(v[lane], v[lane ^ OFF]) for OFF = 8, 16, 32
template <int OFF, typename Op>
__device__ __forceinline__ float xlane_op(float v, Op op) {
  if constexpr (OFF == 8) return op(v, lane_dpp<0x128>(v));  // row_ror:8 within 16 lanes = lane ^ 8
  else if constexpr (OFF == 16) return lane_xor16(v, op);
  else return lane_xor32(v, op);
}
// max / sum over the lanes that share (lane % LPK), i.e. across the 64/LPK key groups of a wave
template <int LPK>
__device__ __forceinline__ float keys_max(float v) {
  if constexpr (LPK <= 8) v = xlane_op<8>(v, LaneMax{});
  if constexpr (LPK <= 16) v = xlane_op<16>(v, LaneMax{});
  return xlane_op<32>(v, LaneMax{});
}
template <int LPK>
__device__ __forceinline__ float keys_sum(float v) {
  if constexpr (LPK <= 8) v = xlane_op<8>(v, LaneAdd{});
  if constexpr (LPK <= 16) v = xlane_op<16>(v, LaneAdd{});
  return xlane_op<32>(v, LaneAdd{});
}

// max / sum over the four 16-lane quarters of a wave (lanes of equal column)
template <typename Op>
__device__ __forceinline__ float quarters(float v, Op op) {
  return xlane_op<32>(xlane_op<16>(v, op), op);
}

constexpr float kLog2e = 1.4426950408889634f;
// masked-key score / empty-state max: finite, so exp2(kNeg - m) underflows to 0 and
// exp2(kNeg - kNeg) = 1 without -inf compares on the hot path
constexpr float kNeg = -1e30f;
// raw v_exp_f32 (denormal results flush to 0, which is all a softmax weight needs); ocml's exp2f
// adds a range-scaling compare + 2 selects per call
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

typedef short av4i16 __attribute__((ext_vector_type(4)));
typedef short av8i16 __attribute__((ext_vector_type(8)));

// fp8 KV (OCP e4m3): 8 codes -> 8 bf16 (exact)
__device__ __forceinline__ gu32x4 fp8x8_bf16x8(uint32_t w0, uint32_t w1) {
  gu32x4 o;
  o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.f, false));
  o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.f, true));
  o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.f, false));
  o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.f, true));
  return o;
}

__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(gbf16x2, a), __builtin_bit_cast(gbf16x2, b), c, false);
}

typedef unsigned int gu32x2 __attribute__((ext_vector_type(2)));
// fp8 KV (OCP e4m3): 2 codes (bytes 2*hi, 2*hi+1 of w) -> a bf16 pair (one v_cvt_scalef32_pk_bf16_fp8)
template <bool HI>
__device__ __forceinline__ uint32_t fp8x2_bf16x2(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, HI));
}
// ... -> an fp32 pair (v_cvt_pk_f32_fp8)
template <bool HI>
__device__ __forceinline__ gf32x2 fp8x2_f32x2(uint32_t w) {
  return __builtin_amdgcn_cvt_pk_f32_fp8((int)w, HI);
}

constexpr int AT_NW = 8;    // waves per workgroup
constexpr int ATTN_SPLIT_LEN = 512;  // keys of a short context
// descriptor of n raw bytes at p (both uniform over the wave)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniform_rsrc(const uint8_t* p, int n) {
  const uint64_t u = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), (short)0, n, 0x00020000);
}
// the lane's number, computed here and now (the asm has no inputs to be hoisted with)
__device__ __forceinline__ int lane_again() {
  int z = 0;
  asm volatile("" : "+s"(z));
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, z));
}
constexpr int AT_TK = 32;   // keys per tile: one wave's unit of work
// LDS row (bytes) of a wave's V tile: rows 32 B apart mod 256, so the 8 rows x 32 B that half a wave's
// transposed read takes fall on distinct banks
template <int HD>
constexpr int at_vrow() { return HD * 2 + 32; }
template <int HD>
constexpr int at_lds_bytes() { return AT_NW * AT_TK * at_vrow<HD>(); }

// A workgroup's last part: the 8 waves' states of its G heads (s_o unnormalised, s_m, s_l; ordered before) merged, and the
// output written (P == 1) or the partial published and, by the last of the P workgroups to arrive, all of them combined.
template <int HD, int G, bool F8, typename Stamp>
__device__ __forceinline__ void attn_meet(const AttnDecodeArgs& a, int h0, int sp, int nact, int tid, int wave, float (*s_o)[G][HD],
                                          float (*s_m)[G], float (*s_l)[G], Stamp stamp) {
  constexpr int NW = AT_NW, NT = NW * 64;
  __shared__ int s_last;
  const int b = blockIdx.z, mlane = tid & 63;
  const float vs = F8 ? a.kv_scale_v : 1.f;
  for (int idx = tid; idx < G * HD; idx += NT) {
    const int g = idx / HD, d = idx - g * HD;
    float M = s_m[0][g];
#pragma unroll
    for (int w = 1; w < NW; ++w) M = fmaxf(M, s_m[w][g]);
    float L = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float sw = fast_exp2(s_m[w][g] - M);
      L += sw * s_l[w][g];
      acc += sw * s_o[w][g][d];
    }
    const int h = h0 + g;
    if (F8) acc *= vs;
    if (nact == 1) {
      if (a.out16) a.out16[((size_t)b * a.n_heads + h) * HD + d] = f32_to_bf16(acc / L);
      else if (a.out_wt) st_wt(a.out + ((size_t)b * a.n_heads + h) * HD + d, acc / L);
      else a.out[((size_t)b * a.n_heads + h) * HD + d] = acc / L;
    } else {
      st_wt(a.o_part + (((size_t)b * a.n_heads + h) * a.n_chunks + sp) * HD + d, acc);
      if (d == 0) {
        float* ml = a.ml + (((size_t)b * a.n_heads + h) * a.n_chunks + sp) * 2;
        st_wt(ml, M);
        st_wt(ml + 1, L);
      }
    }
  }
  if (nact == 1) {
    stamp(6);
    return;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every storing wave drains its sc1 stores
  __syncthreads();
  int* cnt = a.counters + (size_t)b * a.n_heads + h0;
  if (tid == 0) {
    const int t = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = (t == nact - 1);
  }
  __syncthreads();
  stamp(4);
  if (!s_last) return;
  // ---- last arriver.  (1) one thread per (head, partial) loads that partial's (m, l);
  //      (measured: one batch of (m, l) + o loads per output thread -- one round trip but 2x the
  //      loads, the (m, l) ones redundant across a head's 128 threads -- was 1.3 us SLOWER at 1000
  //      keys, 10.09 vs 8.73 us; hoisting the block-table loads above the seq_len test, or
  //      issuing pass 0's K/V before seq_len is read, did not help either: 4.32-4.40 vs 4.18 us
  //      at 153 keys, tools/attn_probe.py -- the short-context launch is the 1.7 us launch chain
  //      plus one K/V round trip plus the merge, not the table lookups)
  //      (2) wave g reduces head g's max M and total L and turns them into normalised weights
  //      w_p = exp2(m_p - M) / L in LDS; (3) every output sums w_p * o_p with 16 loads in flight.
  //      Two memory round trips for up to 64 partials (was one per 8 partials).
  __shared__ float s_pm[G][64], s_pl[G][64];
  // one memory round trip (round 4): when every output has one thread and the partials fit one
  // register batch, each thread issues its output's nact partial loads TOGETHER with the (m, l)
  // sweep and folds them after the weights are ready -- same order of sums as the two-trip path
  auto one_trip = [&](auto ob) __attribute__((always_inline)) {
    constexpr int OB = decltype(ob)::value;
    const int idx = tid;
    const bool act = idx < G * HD;
    const int g = act ? idx / HD : 0, d = act ? idx - g * HD : 0;
    const float* op = a.o_part + ((size_t)b * a.n_heads + h0 + g) * a.n_chunks * HD + d;
    float ov[OB];
#pragma unroll
    for (int j = 0; j < OB; ++j) ov[j] = ld_wt(op + (size_t)min(j, nact - 1) * HD);  // clamped: in bounds
    for (int i = tid; i < G * nact; i += NT) {
      const int gg = i / nact, p = i - gg * nact;
      const float* mlp = a.ml + (((size_t)b * a.n_heads + h0 + gg) * a.n_chunks + p) * 2;
      s_pm[gg][p] = ld_wt(mlp);
      s_pl[gg][p] = ld_wt(mlp + 1);
    }
    __syncthreads();
    if (wave < G) {
      const float mv = mlane < nact ? s_pm[wave][mlane] : kNeg;
      const float lv = mlane < nact ? s_pl[wave][mlane] : 0.f;
      const float M = wave_max(mv);
      const float e = fast_exp2(mv - M);
      const float L = lanes_sum<64>(e * lv);
      if (mlane < nact) s_pm[wave][mlane] = e / L;
    }
    __syncthreads();
    stamp(5);
    if (act) {
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < OB; ++j)
        if (j < nact) acc = fmaf(s_pm[g][j], ov[j], acc);
      const int h = h0 + g;
      if (a.out16) a.out16[((size_t)b * a.n_heads + h) * HD + d] = f32_to_bf16(acc);
      else if (a.out_wt) st_wt(a.out + ((size_t)b * a.n_heads + h) * HD + d, acc);
      else a.out[((size_t)b * a.n_heads + h) * HD + d] = acc;
    }
  };
  if (G * HD <= NT && nact <= 32 && a.combine_trips != 2) {
    if (nact <= 8) one_trip(std::integral_constant<int, 8>{});
    else if (nact <= 16) one_trip(std::integral_constant<int, 16>{});
    else one_trip(std::integral_constant<int, 32>{});
    if (tid == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-arm
    stamp(6);
    return;
  }
  for (int i = tid; i < G * nact; i += NT) {
    const int g = i / nact, p = i - g * nact;
    const float* mlp = a.ml + (((size_t)b * a.n_heads + h0 + g) * a.n_chunks + p) * 2;
    s_pm[g][p] = ld_wt(mlp);
    s_pl[g][p] = ld_wt(mlp + 1);
  }
  __syncthreads();
  if (wave < G) {
    const int g = wave;
    const float mv = mlane < nact ? s_pm[g][mlane] : kNeg;
    const float lv = mlane < nact ? s_pl[g][mlane] : 0.f;
    const float M = wave_max(mv);
    const float e = fast_exp2(mv - M);
    const float L = lanes_sum<64>(e * lv);
    if (mlane < nact) s_pm[g][mlane] = e / L;
  }
  __syncthreads();
  stamp(5);
  for (int idx = tid; idx < G * HD; idx += NT) {
    const int g = idx / HD, d = idx - g * HD;
    const int h = h0 + g;
    const float* op = a.o_part + ((size_t)b * a.n_heads + h) * a.n_chunks * HD + d;
    float acc = 0.f;
    for (int c = 0; c < nact; c += 16) {
      float ov[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) ov[j] = ld_wt(op + (size_t)min(c + j, nact - 1) * HD);
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (c + j < nact) acc = fmaf(s_pm[g][c + j], ov[j], acc);
    }
    if (a.out16) a.out16[((size_t)b * a.n_heads + h) * HD + d] = f32_to_bf16(acc);
    else if (a.out_wt) st_wt(a.out + ((size_t)b * a.n_heads + h) * HD + d, acc);
      else a.out[((size_t)b * a.n_heads + h) * HD + d] = acc;
  }
  if (tid == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-arm
  stamp(6);
}

// One workgroup's share: the G query heads of KV head kvh over the 32-key tiles of P workgroups x 8 waves,
// dealt wave by wave (tile t to wave t mod 8 P: 32 keys is also the granularity of the balance).
//
// Per tile, on the matrix cores:
//   S^T[key][c] = K Q^T   (16x16x32; K comes in whole lines and takes the A operand's order through the wave's own LDS tile: asked
//                         for in that order, 16 lanes at 16 keys, each lane is an address of its own to the address unit: 16000 fp8 keys
//                         15.0 -> 13.4 us, 16 rows of 1000 bf16 ones 16.3 -> 15.0, 32 / 8 heads of 128).  Column
//                         c holds head c mod GP (GP = 4 or 8 >= G): every head's scores, and with them its
//                         probabilities in fp32, stand in 16 / GP columns.
//   O^T[dim][c] += V^T P^T   Each of a head's columns multiplies another bf16 part of the same probability (p's
//                         leading 8 bits, the next 8, the last 8): the three products' sum has p in all its
//                         24 bits, at no matrix instruction more for GP = 4 (two passes for GP = 8: half of the
//                         leading part in each, the middle and the last one beside it).  A leading part stands alone
//                         in its columns' sums, so an infinite value's product is what its probability makes it;
//                         the other parts can be 0 and their sums, 0 x Inf, are left out then.  P^T comes
//                         from the S^T registers, its k order with it; V goes through a wave's own LDS tile
//                         (row-major in, ds_read_b64_tr_b16 out: no barrier, a wave's LDS operations are in order).
// The arithmetic of a tile is then ~100 VALU instructions a wave where dots and P.V on the VALU took ~900:
// at 16000 fp8 keys a workgroup spent 10 us on 512 keys, against 3 us for its bytes.  Loads: two tiles per wave
// in flight (registers), so 512 keys of a workgroup cost one memory round trip.
// q is rounded to bf16 (scaled; fp8: by the layer's K scale too, V's scale on the output); scores, max, sum and
// O in fp32.
template <int HD, int G, bool F8 = false>
__device__ __forceinline__ void attn_core(const AttnDecodeArgs& a, int sp, int kvh, int P_max) {
  constexpr int GP = G <= 4 ? 4 : 8;
  constexpr int NR = GP == 4 ? 1 : 2;       // passes over P's bf16 parts
  constexpr int ES = F8 ? 1 : 2;            // bytes per cached element
  constexpr int EL = 16 / ES;               // elements per 16-B load
  constexpr int KL = HD / (4 * EL);         // K loads per lane and 16 keys
  constexpr int VL = AT_TK * HD / EL / 64;  // K or V loads per lane and tile
  constexpr int VPR = HD / EL;              // 16-B pieces of a row
  constexpr int KROW = HD * ES + 16;        // LDS row of K as cached: 16 rows' reads of one piece on distinct banks
  static_assert(KROW <= at_vrow<HD>());
  constexpr int DT = HD / 16;               // O^T tiles
  constexpr int VROW = at_vrow<HD>();
  constexpr int NW = AT_NW;
  extern __shared__ __attribute__((aligned(16))) uint8_t at_smem[];
  float (*s_o)[G][HD] = (float (*)[G][HD])at_smem;  // (the merge; after the V tiles)
  static_assert(sizeof(float) * NW * G * HD <= at_lds_bytes<HD>(), "merge buffer");
  __shared__ float s_m[NW][G], s_l[NW][G];

  const int b = blockIdx.z, h0 = kvh * G;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 15, q4 = lane >> 4;
  // probe stamps (a.ts; probe builds only, -DAIOS_ATTN_PROBES=1): 0 entry, 1 seq_len known, 2 first tile
  // computed (its K/V landed), 3 waves merged, 4 partial published + ticket, 5 (m, l) weights ready (last
  // arriver), 6 done
  auto stamp = [&](int k) __attribute__((always_inline)) {
    if (AIOS_ATTN_PROBES && a.ts && threadIdx.x == 0)
      a.ts[((size_t)blockIdx.z * gridDim.x + blockIdx.x) * 8 + k] = __builtin_amdgcn_s_memrealtime();
  };
  stamp(0);
  // q first: everything after waits for older loads only, and the tiles below are the youngest
  constexpr int KS = HD / 32;
  float4 qr[KS][2];
  {
    const float* qp = a.q + ((size_t)b * a.n_heads + h0 + min(col & (GP - 1), G - 1)) * HD;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      // bf16: element 32 s + 8 q4; fp8: a 16-element K piece serves two steps
      const float* x = qp + (F8 ? 64 * (s >> 1) + 16 * q4 + 8 * (s & 1) : 32 * s + 8 * q4);
      qr[s][0] = *(const float4*)x;
      qr[s][1] = *(const float4*)(x + 4);
    }
  }
  // the row's numbers through the scalar cache (uniform addresses; written by earlier launches), requested together
  using cint = const __attribute__((address_space(4))) int*;
  // paged KV: tile t lies in block bt[t / 4]
  static_assert(KV_BLOCK == 4 * AT_TK, "four tiles per paged KV block");
  const int maxb = a.max_ctx / KV_BLOCK;
  const size_t blk_stride = (size_t)a.n_kv_heads * KV_BLOCK * HD;
  const int len = ((cint)a.seq_len)[b];
  const int slot = ((cint)(a.slot ? a.slot : a.seq_len))[b];  // (no slots: row b; the value read is not used)
  const int row = a.slot ? slot : b;
  const bool paged = a.block_table != nullptr;
  const cint btr = (cint)(a.block_table + (size_t)(a.bt_rows ? b : row) * maxb);
  const int ntile = (len + AT_TK - 1) / AT_TK;
  // tiles go to the P workgroups in turn, and in a workgroup to its waves.  From 9 tiles up as many workgroups as have
  // 4 tiles: what a CU alone can draw from memory (~40 B/ns) bounds a short launch more than the combine does
  const int P = ntile <= NW ? 1 : max(1, min((ntile + 3) / 4, P_max));
  if (sp >= P) return;  // uniform: this workgroup has no tile, issues no K/V traffic
  stamp(1);

  struct Tile {
    gu32x4 k[VL], v[VL];
    size_t base;  // of the tile in its pool, bytes
    int bytes;    // of its live keys
  };
  Tile tA, tB;
  const uint32_t voff = (uint32_t)lane * 16;  // this lane's 16-B pieces: lane + 64 i, row-major
  const size_t hoff = (size_t)kvh * KV_BLOCK * HD * ES;
  // A tile is a buffer of its live keys' bytes: dead keys of the last tile, and all keys past it, read as zeros without
  // a memory access.  So every path issues the same loads, and the wait for one tile's leaves the next one's in
  // flight (a skipped issue made it wait for both); P = 0 meets no stale V either.
  auto block_of = [&](int tile) __attribute__((always_inline)) { return paged ? btr[min(tile >> 2, maxb - 1)] : 0; };
  auto place = [&](Tile& t, int tile, int blk) __attribute__((always_inline)) {
    const int live = min(max(len - tile * AT_TK, 0), AT_TK);
    t.bytes = __builtin_amdgcn_readfirstlane(live * HD * ES);
    t.base = hoff + (live ? (size_t)(paged ? blk : row * maxb + (tile >> 2)) * blk_stride + (size_t)(tile & 3) * AT_TK * HD : 0) * ES;
  };
  // (streaming loads, aux 2: every K/V line is read once per launch)
  auto issue_k = [&](Tile& t) __attribute__((always_inline)) {
    const auto r = uniform_rsrc((const uint8_t*)a.k_cache + t.base, t.bytes);
#pragma unroll
    for (int i = 0; i < VL; ++i) t.k[i] = __builtin_amdgcn_raw_buffer_load_b128(r, voff + 1024 * i, 0, 2);
  };
  auto issue_v = [&](Tile& t) __attribute__((always_inline)) {
    const auto r = uniform_rsrc((const uint8_t*)a.v_cache + t.base, t.bytes);
#pragma unroll
    for (int i = 0; i < VL; ++i) t.v[i] = __builtin_amdgcn_raw_buffer_load_b128(r, voff + 1024 * i, 0, 2);
  };
  const int step = P * NW, t0 = sp + P * wave;
  place(tA, t0, block_of(t0));
  issue_k(tA);
  issue_v(tA);
  place(tB, t0 + step, block_of(t0 + step));
  issue_k(tB);

  // Q^T (B operand): lane (col, q4) holds head col mod GP's elements of the K pieces' order
  gbf16x8 qf[KS];
  {
    const float qs = a.scale * kLog2e * (F8 ? a.kv_scale_k : 1.f);  // scores in the log2 domain: exp2 below
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float4 x0 = qr[s][0], x1 = qr[s][1];
      const uint4 u = make_uint4(pk_bf16(x0.x * qs, x0.y * qs), pk_bf16(x0.z * qs, x0.w * qs),
                                 pk_bf16(x1.x * qs, x1.y * qs), pk_bf16(x1.z * qs, x1.w * qs));
      __builtin_memcpy(&qf[s], &u, 16);
    }
  }
  float m = kNeg, l = 0.f;  // column's running max; this lane's part of its sum
  gf32x4 o[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i) o[i] = gf32x4{0.f, 0.f, 0.f, 0.f};
  uint8_t* vt = at_smem + wave * (AT_TK * VROW);
  // which part of P this lane's column multiplies (GP = 8: 0 the leading one, 1 the middle and then the last one)
  const int term0 = GP == 4 ? col >> 2 : col >> 3;
  const uint32_t sel0 = term0 == 0 ? ~0u : 0u, sel1 = term0 == 1 ? ~0u : 0u, sel2 = term0 == 2 ? ~0u : 0u;

  // (after_s: what to issue once the K registers are free)
  auto math = [&](Tile& t, int tile, auto after_s) __attribute__((always_inline)) {
    const bool part = (tile + 1) * AT_TK > len;  // the context's last, partly filled tile
    const int live = len - tile * AT_TK;
    // ---- K through the wave's LDS tile: this lane's pieces of key 16 j + col are elements 4 EL i + EL q4 ..
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int p = lane + 64 * i;
      *(gu32x4*)(vt + p / VPR * KROW + p % VPR * 16) = t.k[i];
    }
    gu32x4 kw[2][KL];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < KL; ++i) kw[j][i] = *(const gu32x4*)(vt + (16 * j + col) * KROW + (4 * i + q4) * 16);
    // ---- S^T: keys 16 j + 4 q4 + e of column col
    gf32x4 st[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      st[j] = gf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        gu32x4 w;
        if constexpr (F8) w = fp8x8_bf16x8(kw[j][s >> 1][2 * (s & 1)], kw[j][s >> 1][2 * (s & 1) + 1]);
        else w = kw[j][s];
        st[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gbf16x8, w), qf[s], st[j], 0, 0, 0);
      }
    }
    after_s();
    // ---- online softmax of the tile's 32 keys per column
    if (part) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (16 * j + 4 * q4 + e >= live) st[j][e] = kNeg;
    }
    float mx = st[0][0];
#pragma unroll
    for (int i = 1; i < 8; ++i) mx = fmaxf(mx, st[i >> 2][i & 3]);
    const float mn = fmaxf(m, quarters(mx, LaneMax{}));
    // O is rescaled only when some column's max grew (wave-uniform)
    if (__builtin_amdgcn_ballot_w64(mn > m)) {
      const float alpha = fast_exp2(m - mn);
      l *= alpha;
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[i][e] *= alpha;
      m = mn;
    }
    float p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p[i] = fast_exp2(st[i >> 2][i & 3] - m);
      l += p[i];
    }
    // ---- P^T's bf16 parts
    gbf16x8 pf[NR];
    {
      uint32_t w[NR][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t hi = pk_bf16(p[2 * i], p[2 * i + 1]);
        const float r0 = p[2 * i] - bf16_lo(hi), r1 = p[2 * i + 1] - bf16_hi(hi);  // (exact)
        const uint32_t mid = pk_bf16(r0, r1);
        const uint32_t lo = pk_bf16(r0 - bf16_lo(mid), r1 - bf16_hi(mid));          // (exact: 8 bits left)
        if constexpr (GP == 8) hi = bf16x2_half(hi);
        w[0][i] = (hi & sel0) | (mid & sel1);
        if constexpr (GP == 4) w[0][i] |= lo & sel2;
        else w[1][i] = (hi & sel0) | (lo & sel1);
      }
#pragma unroll
      for (int r = 0; r < NR; ++r) __builtin_memcpy(&pf[r], w[r], 16);
    }
    // ---- V to the wave's LDS tile, row-major
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int p = lane + 64 * i, key = p / VPR, c = p % VPR;
      if constexpr (F8) {
        *(gu32x4*)(vt + key * VROW + c * 32) = fp8x8_bf16x8(t.v[i][0], t.v[i][1]);
        *(gu32x4*)(vt + key * VROW + c * 32 + 16) = fp8x8_bf16x8(t.v[i][2], t.v[i][3]);
      } else {
        *(gu32x4*)(vt + key * VROW + c * 16) = t.v[i];
      }
    }
    // ---- O^T += V^T P^T: k slots of quarter q4 are keys 4 q4 .. + 3 and 16 + 4 q4 .. + 3 (P^T's registers)
    const uint8_t* va = vt + (4 * q4 + (col >> 2)) * VROW + (col & 3) * 8;
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      using tp = __attribute__((address_space(3))) av4i16*;
      const av4i16 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tp)(va + 32 * i));
      const av4i16 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tp)(va + 16 * VROW + 32 * i));
      const av8i16 xv = __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
      const gbf16x8 vf = __builtin_bit_cast(gbf16x8, xv);
#pragma unroll
      for (int r = 0; r < NR; ++r) o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[r], o[i], 0, 0, 0);
    }
  };
  // a wave's registers hold one and a half tiles in flight: the next tile's V is requested when this one's K is used (K of the tile after the next
  // as soon as this one's lies in LDS: no faster, and at head_dim 64 the registers spill)
  for (int t = t0; t < ntile; t += 2 * step) {
    math(tA, t, [&]() __attribute__((always_inline)) { issue_v(tB); });
    if (t == t0) stamp(2);
    place(tA, t + 2 * step, block_of(t + 2 * step));
    issue_k(tA);
    if (t + step >= ntile) break;
    math(tB, t + step, [&]() __attribute__((always_inline)) { issue_v(tA); });
    place(tB, t + 3 * step, block_of(t + 3 * step));
    issue_k(tB);
  }
  // ---- a head's columns summed (row rotates within 16 lanes), then the 8 waves merged in LDS
  l = quarters(l, LaneAdd{});
  gf32x4 z = gf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) z[e] = fmaf(o[i][e], 0.f, z[e]);
  if (__builtin_amdgcn_ballot_w64((z[0] + z[1]) + (z[2] + z[3]) != 0.f)) {  // some Inf or NaN: the leading part's columns have it
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[i][e] = term0 && !__builtin_isfinite(o[i][e]) ? 0.f : o[i][e];
  }
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[i][e] += lane_dpp<0x128>(o[i][e]);                                // row_ror:8
      if constexpr (GP == 4) o[i][e] += lane_dpp<0x124>(o[i][e]);         // row_ror:4
    }
  __syncthreads();  // every wave is done with its V tile: the LDS is the merge's
  // (the thread's number read again, opaque to the compiler: kept through the loop it costs registers that spill)
  const int tid = wave * 64 + lane_again();
  const int mlane = tid & 63, mc = tid & 15, mq = mlane >> 4;
  if (mc < G) {
#pragma unroll
    for (int i = 0; i < DT; ++i) *(float4*)&s_o[wave][mc][16 * i + 4 * mq] = make_float4(o[i][0], o[i][1], o[i][2], o[i][3]);
    if (mq == 0) {
      s_m[wave][mc] = m;
      s_l[wave][mc] = l;
    }
  }
  __syncthreads();
  stamp(3);
  attn_meet<HD, G, F8>(a, h0, sp, P, tid, wave, s_o, s_m, s_l, stamp);
}

// A workgroup per QUERY head, P of them to a head's 128-key passes in turn.  Two uses.
// Contexts up to ATTN_SPLIT_LEN keys of a launch that leaves CUs idle (P = 1): one workgroup walks all (<= 4) passes,
// without a combine.  The G workgroups of a KV head read the same K and V (from L2 after the first, see the roles
// below), so a launch this short is one memory round trip of 64 KB on each of n_heads CUs and little else; attn_core's
// one workgroup per KV head then waits for a longer chain: 130 keys, 32 / 8 heads of 128: 5.2 us
// here, 7.5 us there (4.0 and 4.9 us for 32 / 4 heads of 64); 500 keys of three rows: equal.
// One head of 128 per KV head, every context (attn_lanes_only): attn_core's matrix columns are 4 heads wide, and of its
// workgroups one fits a CU, of these two.
// VALU: q . k on v_dot2_f32_bf16 (q rounded to bf16 pairs), P . V in fp32.  Every lane loads 16 B (fp8 at head_dim 64:
// 8 B) of a key; two passes in flight.
// (LONG: the second use; the first is P = 1)
template <int HD, bool F8, bool LONG>
__device__ __forceinline__ void attn_lanes(const AttnDecodeArgs& a, int kvh, int h, int sp, int P_max) {
  constexpr int DPL = (F8 && HD == 128) ? 16 : 8;  // dims per lane
  using KVT = typename std::conditional<F8 && DPL == 8, uint2, uint4>::type;
  constexpr int ES = F8 ? 1 : 2;  // bytes per cached element
  constexpr int NP = DPL / 2;     // bf16 / fp32 pairs per lane
  constexpr int NW = AT_NW;
  constexpr int LPK = HD / DPL;        // lanes per key
  constexpr int KPS = 64 / LPK;        // keys per wave-instruction
  constexpr int CH = 128;              // keys per pass
  constexpr int KPW = CH / NW;         // keys per wave per pass
  constexpr int STEPS = KPW / KPS;     // loads per lane per pass (each of K and V)
  extern __shared__ __attribute__((aligned(16))) uint8_t at_smem[];
  float (*s_o)[1][HD] = (float (*)[1][HD])at_smem;
  __shared__ float s_m[NW][1], s_l[NW][1];

  const int b = blockIdx.z;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int ksub = lane / LPK, dsl = lane % LPK;
  static_assert(CH == KV_BLOCK, "one pass = one paged KV block");
  const int slot = a.slot ? a.slot[b] : b;
  const int maxb = a.max_ctx / KV_BLOCK;
  const int* btr = a.block_table ? a.block_table + (size_t)(a.bt_rows ? b : slot) * maxb : nullptr;
  const size_t blk_stride = (size_t)a.n_kv_heads * KV_BLOCK * HD;
  const int koff = wave * KPW + ksub;  // this lane's key within a pass (+ s * KPS)
  const uint8_t* kc = (const uint8_t*)a.k_cache + ((size_t)kvh * KV_BLOCK * HD + (size_t)koff * HD + dsl * DPL) * ES;
  const uint8_t* vc = (const uint8_t*)a.v_cache + ((size_t)kvh * KV_BLOCK * HD + (size_t)koff * HD + dsl * DPL) * ES;
  const int len = a.seq_len[b];
  const int nchunk = (len + CH - 1) / CH;
  const int P = !LONG || nchunk <= 2 ? 1 : min(nchunk, P_max);  // (two passes are in flight at once)
  if (LONG && sp >= P) return;  // (uniform)

  KVT kA[STEPS], vA[STEPS], kB[STEPS], vB[STEPS];
  auto ld = [&](const uint8_t* p) __attribute__((always_inline)) {
    if constexpr (LONG) {  // (read once per launch)
      typedef uint32_t vec __attribute__((ext_vector_type(sizeof(KVT) / 4)));
      const vec v = __builtin_nontemporal_load((const vec*)p);
      KVT r;
      __builtin_memcpy(&r, &v, sizeof(r));
      return r;
    } else {
      return *(const KVT*)p;
    }
  };
  auto issue = [&](KVT (&kr)[STEPS], KVT (&vr)[STEPS], int c) __attribute__((always_inline)) {
    const size_t base = (size_t)(btr ? btr[c] : slot * maxb + c) * blk_stride * ES;  // (bytes)
    if ((c + 1) * CH > len) {
      // the context's last, partly filled block: only the lanes of live keys load (a 153-key context
      // fetched 2 x 64 KB for 25 keys of its second block); dead keys hold zeros (scores masked, V x 0)
      const int k0 = c * CH + koff;
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        kr[s] = KVT{};
        vr[s] = KVT{};
        if (k0 + s * KPS < len) {
          kr[s] = ld(kc + base + (size_t)s * KPS * HD * ES);
          vr[s] = ld(vc + base + (size_t)s * KPS * HD * ES);
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < STEPS; ++s) kr[s] = ld(kc + base + (size_t)s * KPS * HD * ES);
#pragma unroll
      for (int s = 0; s < STEPS; ++s) vr[s] = ld(vc + base + (size_t)s * KPS * HD * ES);
    }
  };
  issue(kA, vA, sp);
  if (sp + P < nchunk) issue(kB, vB, sp + P);
  const float qs = a.scale * kLog2e * (F8 ? a.kv_scale_k : 1.f);  // scores in the log2 domain: exp2 below
  uint32_t q2[NP];                 // q * scale as bf16 pairs
  {
    const float* qp = a.q + ((size_t)b * a.n_heads + h) * HD + dsl * DPL;
#pragma unroll
    for (int j = 0; j < DPL / 4; ++j) {
      const float4 q0 = *(const float4*)(qp + 4 * j);
      q2[2 * j] = pk_bf16(q0.x * qs, q0.y * qs);
      q2[2 * j + 1] = pk_bf16(q0.z * qs, q0.w * qs);
    }
  }
  float m = kNeg, l = 0.f;  // per key group: the LPK lanes of a key share its score
  gf32x2 o[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) o[i] = gf32x2{0.f, 0.f};
  auto pass = [&](const KVT (&kr)[STEPS], const KVT (&vr)[STEPS], int c) __attribute__((always_inline)) {
    float sc[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const bool valid = c * CH + koff + s * KPS < len;
      uint32_t kb[NP];
      if constexpr (F8 && DPL == 16) {
        const uint32_t w4[4] = {kr[s].x, kr[s].y, kr[s].z, kr[s].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) { kb[2 * i] = fp8x2_bf16x2<false>(w4[i]); kb[2 * i + 1] = fp8x2_bf16x2<true>(w4[i]); }
      } else if constexpr (F8) {
        kb[0] = fp8x2_bf16x2<false>(kr[s].x); kb[1] = fp8x2_bf16x2<true>(kr[s].x);
        kb[2] = fp8x2_bf16x2<false>(kr[s].y); kb[3] = fp8x2_bf16x2<true>(kr[s].y);
      } else {
        kb[0] = kr[s].x; kb[1] = kr[s].y; kb[2] = kr[s].z; kb[3] = kr[s].w;
      }
      float d = dot2_bf16(kb[0], q2[0], 0.f);
#pragma unroll
      for (int i = 1; i < NP; ++i) d = dot2_bf16(kb[i], q2[i], d);
      d = lanes_sum<LPK>(d);
      sc[s] = valid ? d : kNeg;
    }
    float mx = sc[0];
#pragma unroll
    for (int s = 1; s < STEPS; ++s) mx = fmaxf(mx, sc[s]);
    const float mn = fmaxf(m, mx);
    float ps = 0.f;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      sc[s] = fast_exp2(sc[s] - mn);
      ps += sc[s];
    }
    if (__builtin_amdgcn_ballot_w64(mn > m)) {  // (wave-uniform: some lane's max grew)
      const float alpha = fast_exp2(m - mn);
      l *= alpha;
#pragma unroll
      for (int i = 0; i < NP; ++i) o[i] *= alpha;
    }
    l += ps;
    m = mn;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      gf32x2 vf[NP];
      if constexpr (F8 && DPL == 16) {
        const uint32_t w4[4] = {vr[s].x, vr[s].y, vr[s].z, vr[s].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) { vf[2 * i] = fp8x2_f32x2<false>(w4[i]); vf[2 * i + 1] = fp8x2_f32x2<true>(w4[i]); }
      } else if constexpr (F8) {
        vf[0] = fp8x2_f32x2<false>(vr[s].x); vf[1] = fp8x2_f32x2<true>(vr[s].x);
        vf[2] = fp8x2_f32x2<false>(vr[s].y); vf[3] = fp8x2_f32x2<true>(vr[s].y);
      } else {
        const uint32_t w[4] = {vr[s].x, vr[s].y, vr[s].z, vr[s].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) vf[i] = gf32x2{__uint_as_float(w[i] << 16), __uint_as_float(w[i] & 0xffff0000u)};
      }
      const gf32x2 pp = gf32x2{sc[s], sc[s]};
#pragma unroll
      for (int i = 0; i < NP; ++i) o[i] = __builtin_elementwise_fma(pp, vf[i], o[i]);
    }
  };
  for (int c = sp; c < nchunk; c += 2 * P) {
    pass(kA, vA, c);
    if (c + 2 * P < nchunk) issue(kA, vA, c + 2 * P);
    if (c + P < nchunk) {
      pass(kB, vB, c + P);
      if (c + 3 * P < nchunk) issue(kB, vB, c + 3 * P);
    }
  }
  // ---- merge the key groups of a wave (their (m, l, o) rescaled to the wave's max), then the 8 waves in LDS
  const float M = keys_max<LPK>(m), w = fast_exp2(m - M);
  l = keys_sum<LPK>(l * w);
  float of[DPL];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    of[2 * i] = keys_sum<LPK>(o[i].x * w);
    of[2 * i + 1] = keys_sum<LPK>(o[i].y * w);
  }
  if (ksub == 0) {
    float4* dst = (float4*)&s_o[wave][0][dsl * DPL];
#pragma unroll
    for (int j = 0; j < DPL / 4; ++j) dst[j] = make_float4(of[4 * j], of[4 * j + 1], of[4 * j + 2], of[4 * j + 3]);
  }
  if (lane == 0) {
    s_m[wave][0] = M;
    s_l[wave][0] = l;
  }
  __syncthreads();
  if constexpr (LONG) {
    attn_meet<HD, 1, F8>(a, h, sp, P, threadIdx.x, wave, s_o, s_m, s_l, [](int) {});
    return;
  }
  const int d = threadIdx.x;
  if (d >= HD) return;
  float W = s_m[0][0];
#pragma unroll
  for (int v = 1; v < NW; ++v) W = fmaxf(W, s_m[v][0]);
  float L = 0.f, acc = 0.f;
#pragma unroll
  for (int v = 0; v < NW; ++v) {
    const float sw = fast_exp2(s_m[v][0] - W);
    L += sw * s_l[v][0];
    acc += sw * s_o[v][0][d];
  }
  if (F8) acc *= a.kv_scale_v;
  const size_t oi = ((size_t)b * a.n_heads + h) * HD + d;
  if (a.out16) a.out16[oi] = f32_to_bf16(acc / L);
  else if (a.out_wt) st_wt(a.out + oi, acc / L);
  else a.out[oi] = acc / L;
}

// The grid is flat (one x-slot per role of the larger form) and each workgroup derives its role from seq_len, so a
// launch captured for max_ctx serves every context; workgroups without keys return at once.
struct AttnSplit {
  int p;           // workgroups per (row, KV head) of attn_core
  int turn, most;  // where the grid has more x-slots: rows take other ones of them (row >> turn, at most `most`)
};

template <int HD, int G, bool F8 = false>
__device__ __forceinline__ void attn_role(const AttnDecodeArgs& a, const AttnSplit& s, int wg) {
  if ((G > 1 || a.short_len > 0) && a.seq_len[blockIdx.z] <= a.short_len) {
    // workgroups are dealt round-robin over the 8 XCDs (blockIdx % 8), so workgroup wg takes query head
    // (wg % 8) * (H / 8) + wg / 8: the G query heads of a KV head then run on one XCD and read its K/V from that
    // XCD's L2 after the first miss (the plain mapping put them on G different XCDs)
    if (wg >= a.n_heads) return;
    const int h = (a.n_heads & 7) == 0 ? (wg & 7) * (a.n_heads >> 3) + (wg >> 3) : wg;
    attn_lanes<HD, F8, false>(a, h / G, h, 0, 1);
  } else {
    // (the same slots in every row put two workgroups on some CUs and none on others: 16 rows of 1500 keys, 32 / 16 heads of
    // 64 30 -> 21 us)
    if (s.most) {
      wg -= min((int)blockIdx.z >> s.turn, s.most) * (a.n_kv_heads * s.p);
      if (wg < 0) wg += gridDim.x;
    }
    if (wg >= a.n_kv_heads * s.p) return;
    attn_core<HD, G, F8>(a, wg % s.p, wg / s.p, s.p);
  }
}

inline int attn_env_int(const char* k, int dflt) {
  const char* e = std::getenv(k);
  return e ? std::atoi(e) : dflt;
}

int attn_decode_split(int max_ctx, int B, int n_kv_heads);
// the launcher's defaults filled in (split, combine)
inline AttnDecodeArgs attn_resolve(const AttnDecodeArgs& a) {
  AttnDecodeArgs b = a;
  if (b.split <= 0) b.split = attn_decode_split(a.max_ctx, a.B, a.n_kv_heads);
  if (b.combine_trips == 0) b.combine_trips = attn_env_int("AIOS_ATTN_COMBINE", 1);
  // The short form as long as its workgroups (a row's query heads) are resident at once, two to a CU at head_dim 64
  // and one at 128 (registers); beyond, attn_core's (a row's KV heads): 12 rows of 450 keys, 32 / 8 heads of 128:
  // 14.6 us short, 11.5 us core; 16 rows, 32 / 4 heads of 64: 7.5 and 8.1 us.  One head of 64 per KV head, where
  // either form has a workgroup a head: up to half of the CUs (8 rows of 400 keys, 16 heads 6.2 and 7.9 us, 16 rows of 500
  // 9.8 and 8.9).  AIOS_ATTN_GROUPED_MIN=n: attn_core from n such workgroups up.
  if (b.short_len < 0) {
    const int grouped_min = attn_env_int("AIOS_ATTN_GROUPED_MIN", 0), cus = device_cu_count(), wgs = a.B * a.n_heads;
    const int most = a.head_dim != 64 ? cus : a.n_heads == a.n_kv_heads ? cus / 2 : 2 * cus;
    b.short_len = (grouped_min > 0 ? a.B * a.n_kv_heads >= grouped_min : wgs > most) ? 0 : ATTN_SPLIT_LEN;
  }
  return b;
}

// Whether every context takes attn_lanes: one query head of 128 per KV head, bf16, or fp8 where the heads alone are more
// than the CUs.  us, lanes / core, 32 heads: bf16 16 rows of 130 keys 9.5 / 13.1, of 600 27.7 / 30.9, one row of 600 8.6 / 9.5; fp8
// 16 rows of 600 18.4 / 20.4, 4 of 4000 32 / 29.
inline bool attn_lanes_only(const AttnDecodeArgs& a, int G) {
  return G == 1 && a.head_dim == 128 && (!a.kv_fp8 || a.B * a.n_heads > device_cu_count());
}

// the launch shape for AttnDecodeArgs a (split already resolved): fills the split and returns the flat
// workgroup count (one x-slot per role of the larger form)
inline int attn_plan(const AttnDecodeArgs& a, int G, AttnSplit& sp) {
  const int nch = std::max(1, a.max_ctx / 128);
  sp.p = std::max(1, std::min(nch, a.split / ATTN_CHUNK));
  if (sp.p > a.n_chunks || sp.p > 64)
    throw std::runtime_error("attn_decode: more splits than partial buffers / 64");
  const int core = a.n_kv_heads * sp.p, slots = std::max(core, a.short_len != 0 ? a.n_heads : 0);
  sp.most = slots / core - 1;
  for (sp.turn = 0; sp.most && (2 << sp.turn) * (sp.most + 1) <= a.B;) ++sp.turn;
  return slots;
}
}  // namespace aios
