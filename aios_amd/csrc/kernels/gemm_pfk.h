// Prefill GEMM, K over the waves (Q4_K / Q6_K weights, 33 rows and more):
//   C[M][N] (epilogue) = A[M][K] (bf16) x W[N][K]^T
//
// Four waves (eight: two groups, half of the columns each) share the k of a tile of 32 MT x 32 CT.  X goes through LDS in slots
// of 128 k, and a wave reads the 32 k of a slot that are its own, where each wave of the column-split tiles (gemm_pf.h) reads the
// whole slot; weights are decoded once a workgroup, by the wave whose k they are.  The partial tiles meet in LDS at the end.
// What a wave does not read it need not wait for: slots of 128 k make half the barriers of the 64-k ones.
//
// Weights come 256 k at a time, whole 128-byte lines of codes: 64 lanes that ask for 64 pieces of 32 bytes cost the address unit
// as much as 4 KB of lines do (X from L2 in 16- and 32-byte pieces 15 bytes a clock and CU, in lines 50).
// Bounds, 160 x 128 tile, per slot at 1.9 GHz: matrix instructions 1280 cycles, the loop 1900 (1500 without the requests and the decode: two
// waves a SIMD meet at one barrier); beside the loop ~3 us to the first data and 5 us in which four partial tiles
// meet.  Weights and X from memory, us, column-split tiles -> this:
//   28672 x 4096 Q4_K SwiGLU, 64 / 130 / 300 rows  40 -> 29, 68 -> 46, 131 -> 91     6144 x 4096, 130 / 711 rows  40 -> 18, 78 -> 48
//   4096 x 4096 Q4_K, 130 / 300 / 700 rows  22 -> 15, 37 -> 20, 53 -> 33             4096 x 14336 Q4_K, 130 / 300 rows  40 -> 30, 102 -> 46
//   4096 x 14336 Q6_K, 130 rows  47 -> 35    2048 x 5632 Q4_K, 64 rows  37 -> 10     11264 x 2048 Q4_K SwiGLU, 64 rows  20 -> 11
// 256 x 256 tiles (gemm_pf.h) stay the faster ones for wide products from ~700 rows (28672 x 4096, 2048 rows: 444 / 533).
//
// Not better: one wave a SIMD (320 accumulators do not fit beside AGPRs; 128 rows 58 us); requests in one burst behind the barrier
// (they hold each wave until the address unit has taken them: 48 to 49 us of 46); slices of a tile on different XCDs (4096 x 14336 33 of 31).
#pragma once
#include "gemm_pf.h"
#include "skinny_epi.h"

namespace aios {

constexpr int PFK_LDS = 160 * 1024 - 64;  // dynamic LDS of these kernels at most: their last_flag lies beside it

// The fused RMSNorm's consumer: the scales of the tile's rows from the producer's sums of squares (at most 64 parts a row: one per 64
// columns).  A wave has its rows' parts brought into its own share of an X slot that is not in use yet, so they travel with the first
// requests (read into registers they were waited for together with all of those), and adds them up in a fixed order, eight lanes a row.
template <int BM, int NW>
struct PfkRows {
  static constexpr int RW = BM / NW, NP = RW / 4, KI = (RW + 7) / 8;  // rows of a wave, its requests (4 rows each), rows of a lane's eighth
  float inv[KI];
  __device__ __forceinline__ void request(const GemmQArgs& a, int m0, int wave, int lane, uint32_t slot);
  __device__ __forceinline__ void done(const GemmQArgs& a, int wave, int lane, const uint8_t* slot) {
    const uint8_t* own = slot + wave * (RW * 256);
#pragma unroll
    for (int k = 0; k < KI; ++k) {
      const int r = min(8 * k + (lane >> 3), RW - 1);
      gf32x4 t = gf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const gf32x4 u = *(const gf32x4*)(own + r * 256 + 128 * j + 16 * (lane & 7));
        if (32 * j + 4 * (lane & 7) < a.nrm_parts) t += u;
      }
      float s = (t[0] + t[1]) + (t[2] + t[3]);
      inv[k] = rsqrtf(lanes_sum<8>(s) / (float)a.K + a.nrm_eps);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the slot's own requests follow)
  }
  __device__ __forceinline__ void put(int wave, int lane, float* inv_s) const {
#pragma unroll
    for (int k = 0; k < KI; ++k) {
      const int r = 8 * k + (lane >> 3);
      if ((lane & 7) == 0 && r < RW) inv_s[wave * RW + r] = inv[k];
    }
  }
};

template <int QT, int MT, int CT, int NG>
struct PfkLayout {
  static constexpr bool Q6 = QT == QT_Q6_K;
  static constexpr int BM = 32 * MT, BN = 32 * CT;
  static constexpr int XS = BM * 256;  // an X slot: 128 k
  static constexpr int NSX = 3;
  // a W block (256 k): codes (128 B a column, units swizzled), high bits, records (Q6_K: int8 scales), dwords that hold d
  static constexpr int CODE = BN * 128, HB = Q6 ? BN * 64 : 0, REC = BN * 16, DW = Q6 ? (BN * 4 < 256 ? 256 : BN * 4) : 0;
  static constexpr int OFF_HB = CODE, OFF_REC = OFF_HB + HB, OFF_D = OFF_REC + REC, WB = OFF_D + DW;
  static constexpr int NWB = (PFK_LDS - NSX * XS) / WB < 4 ? (PFK_LDS - NSX * XS) / WB : 4;
  static constexpr int OFF_W = NSX * XS;
  static constexpr int NW = 4 * NG, NX = 2 * MT / NG;  // waves; DMA requests a wave, per X slot
  static constexpr int PC = 4 * CT, PR = 2 * CT;       // pieces of a W block: codes, records (high bits); a wave's (of few: some twice)
  static constexpr int NC = PC / NW, NR = PR > NW ? PR / NW : 1, NH = Q6 ? NR : 0, ND = Q6 ? 1 : 0, NWP = NC + NR + NH + ND;
  static constexpr int RED_BYTES = 2 * 4 * 32 * BN * 4 + BM * 4;  // two row tiles of four partial sums, the rows' scales
  // the rows' scales: behind the slots where there is room, else behind the partial sums once the loop is done
  static constexpr bool KEEP = OFF_W + NWB * WB + BM * 4 > PFK_LDS;
  static constexpr int USED = OFF_W + NWB * WB + (KEEP ? 0 : BM * 4), TOTAL = USED > RED_BYTES ? USED : RED_BYTES;
  static_assert(NWB < 2 || TOTAL <= PFK_LDS, "pfk LDS");
};

// a 1-KB (256-B) request to LDS bytes lds ..
__device__ __forceinline__ void pfk_dma1(const void* base, uint32_t off, uint32_t lds) {
  uint64_t from;
  asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 %0, %2\n\tglobal_load_lds_dwordx4 %1, %0"
               : "=&s"(from)
               : "v"(off), "s"(base), "s"(lds)
               : "memory", "m0");
}
__device__ __forceinline__ void pfk_dma4(const void* base, uint32_t off, uint32_t lds) {
  uint64_t from;
  asm volatile("s_mov_b32 m0, %3\n\ts_mov_b64 %0, %2\n\tglobal_load_lds_dword %1, %0"
               : "=&s"(from)
               : "v"(off), "s"(base), "s"(lds)
               : "memory", "m0");
}

template <int BM, int NW>
__device__ __forceinline__ void PfkRows<BM, NW>::request(const GemmQArgs& a, int m0, int wave, int lane, uint32_t slot) {
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int row = min(m0 + wave * RW + 4 * i + (lane >> 4), a.M - 1), u = 4 * (lane & 15) < a.nrm_parts ? lane & 15 : 0;
    pfk_dma1(a.nrm_in, ((uint32_t)row * (uint32_t)a.nrm_parts + 4u * u) * 4u, slot + wave * (RW * 256) + i * 1024);
  }
}

// host: whether the epilogue's operands fit the stores of these kernels (bn: columns of a tile).  16-byte stores to C, 8-byte ones to C16 and
// 4-byte ones of a gated product; a part of the split RMSNorm per 64 columns, on either side
inline bool pfk_epi_ok(const GemmQArgs& a, int bn) {
  auto off = [](const void* p, int n) { return ((uintptr_t)p & (n - 1)) != 0; };
  if (a.nrm_in && (a.K % 256 || a.K > 4096 || a.nrm_parts != a.K / 64 || off(a.nrm_in, 16))) return false;
  switch (a.epi) {
    case GEPI_STORE: case GEPI_ACCUM: return a.C && a.ldc % 4 == 0 && !off(a.C, 16);
    case GEPI_ACCUM_NORM:
      return a.C && a.ldc % 4 == 0 && !off(a.C, 16) && bn >= 64 && a.nrm_g && !off(a.nrm_g, 16) && a.nrm_out16 && !off(a.nrm_out16, 8) && a.nrm_part &&
             a.nrm_parts == a.N / 64 && !a.bias16;
    case GEPI_SWIGLU_BF16: return a.C16 && a.ldc % 2 == 0 && !off(a.C16, 4);
    case GEPI_STORE16: return a.C16 && a.ldc % 4 == 0 && !off(a.C16, 8);
    case GEPI_QKV:  // (a lane's four columns in one head, its stores whole)
      return a.q_out && a.k_cache && a.v_cache && !off(a.q_out, 16) && !off(a.k_cache, 8) && !off(a.v_cache, 8) && a.head_dim % 4 == 0 && a.q_dim % 4 == 0 && a.kv_dim % 4 == 0;
    default: return false;
  }
}

// host: f(MT, CT, NG) of a tile, false if there is none: 64 to 160 rows; 32 columns (four waves), 64 or 128 (eight)
template <typename F>
inline bool pfk_tile(int bm, int bn, F f) {
#define PFK_T(N) std::integral_constant<int, N> {}
  auto cols = [&](auto mt) {
    switch (bn) {
      case 32: return f(mt, PFK_T(1), PFK_T(1));
      case 64: return f(mt, PFK_T(2), PFK_T(2));
      case 128: return f(mt, PFK_T(4), PFK_T(2));
      default: return false;
    }
  };
  switch (bm) {
    case 64: return cols(PFK_T(2));
    case 96: return cols(PFK_T(3));
    case 128: return cols(PFK_T(4));
    case 160: return cols(PFK_T(5));
    default: return false;
  }
#undef PFK_T
}

// host: whether S slices of K have the workspace for their slabs and a ticket per tile
inline bool pfk_slabs_ok(const GemmQArgs& a, int bm, int bn, int S) {
  if (S == 1) return true;
  const size_t tiles = (size_t)(a.N / bn) * ((a.M + bm - 1) / bm), by = (size_t)S * tiles * bm * bn * 4;
  return a.ws && a.cnt && tiles <= (size_t)a.cnt_len && by <= a.ws_bytes && by < 0x7fffffff;
}

// ---- end of a tile: the four partial sums of every output, the slices of K, the epilogue
template <int MT, int CT, int NG, int EPI, bool KEEP, int TOTAL>
__device__ __forceinline__ void pfk_close(const GemmQArgs& a, const gf32x16 (&acc)[MT][CT / NG], int m0, int n0, int sp, int S, int tile,
                                          int ntile, int& last_flag, const PfkRows<32 * MT, 4 * NG>& rows) {
  constexpr int BM = 32 * MT, BN = 32 * CT, NW = 4 * NG, CW = CT / NG;
  extern __shared__ __attribute__((aligned(16))) uint8_t pf_smem0[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wv = wave & 3, cg = wave >> 2;
  const int r32 = lane & 31, h = lane >> 5;
  float* inv_s = (float*)(pf_smem0 + (KEEP ? 2 * 4 * 32 * BN * 4 : TOTAL - BM * 4));
  // ---- the four partial tiles meet, 32 rows at a time: [wave][row][columns], 16-B units swizzled by the row; a row tile is
  // written while the one before it is added up
  constexpr int QR = 8 * CT, RP = 64 * NW / QR, SRC = 32 * 32 * CT * 4;
  auto unit = [&](int row, int q) __attribute__((always_inline)) {
    return (uint32_t)(row * (32 * CT * 4) + ((q ^ (CT == 1 ? (row >> 1) & 7 : row & 15)) << 4));
  };
  const int q = tid % QR, n = n0 + 4 * q;
  const auto ws = __builtin_amdgcn_make_buffer_rsrc((void*)a.ws, (short)0, 0x7fffffff, 0x00020000);
  auto slab = [&](int k) __attribute__((always_inline)) {  // byte of slice k's partial sums of this tile
    return (uint32_t)(k * ntile + tile) * (uint32_t)(BM * BN * 4);
  };
  // What an output needs besides its sum is requested ahead: a load behind a store to what may be the same place would wait for it, row by
  // row.  us, residual so -> ahead: 4096 x 4096 Q4_K, 300 / 700 rows 22 -> 20, 40 -> 33; 4096 x 14336, 300 rows Q4_K 51 -> 46, Q6_K
  // 63 -> 56; 130 rows Q6_K 39 -> 35.  6144 x 4096 to q and the cache, 130 rows in two slices 27 -> 25.
  gf32x4 gain = {};
  if constexpr (EPI == GEPI_ACCUM_NORM) gain = *(const gf32x4*)(a.nrm_g + n);
  const int hd = EPI == GEPI_QKV ? a.head_dim : 4;
  const int sect = EPI != GEPI_QKV || n < a.q_dim ? 0 : (n < a.q_dim + a.kv_dim ? 1 : 2);  // q, k, v
  const int nr = sect == 0 ? n : n - (sect == 1 ? a.q_dim : a.q_dim + a.kv_dim), head = nr / hd, lr = nr - head * hd;
  struct Ahead {
    gf32x4 c;   // the residual | RoPE's (cos, sin) of the two pairs
    size_t to;  // QKV: where the row's four elements go
  };
  auto ahead = [&](int row) __attribute__((always_inline)) {
    Ahead h_;
    h_.c = gf32x4{1.f, 0.f, 1.f, 0.f};
    h_.to = 0;
    const int m = min(m0 + row, a.M - 1);
    if constexpr (EPI == GEPI_ACCUM || EPI == GEPI_ACCUM_NORM) {
      h_.c = *(const gf32x4*)(a.C + (size_t)m * a.ldc + n);
    } else if constexpr (EPI == GEPI_QKV) {
      const int pos = a.pos[m], slot = a.slot ? a.slot[m] : 0;
      if (sect < 2) {
        const float2* cs = a.rope_cs + (size_t)pos * (hd >> 1) + (lr >> 1);
        const float2 c0 = cs[0], c1 = cs[1];
        h_.c = gf32x4{c0.x, c0.y, c1.x, c1.y};
      }
      h_.to = sect == 0 ? (size_t)m * a.q_dim + n : kv_offset(a.block_table, a.max_ctx / KV_BLOCK, slot, a.n_kv_heads, head, pos, hd) + lr;
    }
    return h_;
  };
  auto finish = [&](int row, gf32x4 v, const Ahead& h_) __attribute__((always_inline)) {
    const int m = m0 + row;
    if (a.nrm_in) v *= inv_s[row];
    if constexpr (EPI == GEPI_ACCUM_NORM) {
      const gf32x4 x = h_.c + v;
      *(gf32x4*)(a.C + (size_t)m * a.ldc + n) = x;
      *(uint2*)(a.nrm_out16 + (size_t)m * a.ldc + n) = make_uint2(pk_bf16(x[0] * gain[0], x[1] * gain[1]), pk_bf16(x[2] * gain[2], x[3] * gain[3]));
      float ss = (x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]);
      ss = lanes_sum<16>(ss);  // 64 columns of a row lie on 16 successive lanes
      if ((q & 15) == 0) a.nrm_part[(size_t)m * a.nrm_parts + (n >> 6)] = ss;
    } else if constexpr (EPI == GEPI_QKV) {
      const gf32x4 t = h_.c;
      if (sect < 2)  // (v's (1, 0) would turn an infinite value's partner into NaN)
        v = gf32x4{v[0] * t[0] - v[1] * t[1], v[0] * t[1] + v[1] * t[0], v[2] * t[2] - v[3] * t[3], v[2] * t[3] + v[3] * t[2]};
      const float o0 = v[0], o1 = v[1], o2 = v[2], o3 = v[3];
      if (sect == 0) {
        *(gf32x4*)(a.q_out + h_.to) = gf32x4{o0, o1, o2, o3};
      } else {
        bf16_t* cache = sect == 1 ? a.k_cache : a.v_cache;
        const float inv = sect == 1 ? a.kv_inv_k : a.kv_inv_v;
        if (a.kv_fp8) *(uint32_t*)((uint8_t*)cache + h_.to) = f32x2_to_fp8x2(o0 * inv, o1 * inv) | f32x2_to_fp8x2(o2 * inv, o3 * inv) << 16;
        else *(uint2*)(cache + h_.to) = make_uint2(pk_bf16(o0, o1), pk_bf16(o2, o3));
      }
    } else {
      sk_finish<EPI>(a, nullptr, m, n, v, (const float4*)&h_.c);
    }
  };
  constexpr int AH = EPI == GEPI_QKV && RP < 32 ? 2 : MT;  // row tiles ahead (of 128 columns' QKV all do not fit beside the accumulators)
  Ahead now[MT][32 / RP];
  auto fetch = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 32 / RP; ++k) now[i][k] = ahead(32 * i + tid / QR + RP * k);
  };
  if (S == 1) {
#pragma unroll
    for (int i = 0; i < AH; ++i) fetch(i);
  }
#pragma unroll
  for (int i = 0; i <= MT; ++i) {
    pf_barrier();
    if (KEEP && i == 0 && a.nrm_in) rows.put(wave, lane, inv_s);
    if (S == 1 && i > 0 && i - 1 + AH < MT) fetch(i - 1 + AH);
    if (i < MT) {
#pragma unroll
      for (int c = 0; c < CW; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *(gf32x4*)(pf_smem0 + (i & 1) * (4 * SRC) + wv * SRC + unit(r32, 8 * (cg * CW + c) + 2 * e + h)) =
              gf32x4{acc[i][c][4 * e], acc[i][c][4 * e + 1], acc[i][c][4 * e + 2], acc[i][c][4 * e + 3]};
    }
    if (i > 0) {
      const uint8_t* src = pf_smem0 + ((i - 1) & 1) * (4 * SRC);
      gf32x4 v[32 / RP];
#pragma unroll
      for (int k = 0; k < 32 / RP; ++k) {
        const uint32_t at = unit(tid / QR + RP * k, q);
        v[k] = *(const gf32x4*)(src + at);
#pragma unroll
        for (int s = 1; s < 4; ++s) v[k] += *(const gf32x4*)(src + s * SRC + at);
      }
#pragma unroll
      for (int k = 0; k < 32 / RP; ++k) {
        const int row = 32 * (i - 1) + tid / QR + RP * k;
        if (m0 + row >= a.M) continue;
        if (S == 1) finish(row, v[k], now[i - 1][k]);
        else
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(gu32x4, v[k]), ws, slab(sp) + ((uint32_t)row * BN + 4 * q) * 4, 0, 16 /* sc1 */);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  if (S == 1) return;
  // ---- K split over workgroups: the slabs are written through; a tile's last arriver adds them up, in the order of the slices
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every storing wave drains its slab stores
  __syncthreads();
  if (tid == 0) {
    const int last = __hip_atomic_fetch_add(a.cnt + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == S - 1;
    if (last) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __hip_atomic_store(a.cnt + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-arm
    }
    last_flag = last;
  }
  __syncthreads();
  if (!last_flag) return;
  constexpr int NP = BM / RP, PB = EPI == GEPI_QKV ? (NP < 4 ? NP : 4) : (NP < 8 ? NP : 8);  // rows of a lane; so many at a time
#pragma unroll
  for (int p0_ = 0; p0_ < NP; p0_ += PB) {
    gf32x4 v[PB];
    Ahead c[PB];
#pragma unroll
    for (int p = 0; p < PB; ++p) {
      v[p] = gf32x4{0.f, 0.f, 0.f, 0.f};
      c[p] = ahead(tid / QR + RP * (p0_ + p));
    }
    for (int k0 = 0; k0 < S; k0 += 4) {  // four slabs' loads in flight
      gf32x4 t[PB][4];
#pragma unroll
      for (int p = 0; p < PB; ++p) {
        const int row = min(tid / QR + RP * min(p0_ + p, NP - 1), a.M - 1 - m0);
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k0 + k < S) t[p][k] = *(const gf32x4*)((const uint8_t*)a.ws + slab(k0 + k) + ((uint32_t)row * BN + 4 * q) * 4);
      }
#pragma unroll
      for (int p = 0; p < PB; ++p)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k0 + k < S) v[p] += t[p][k];
    }
#pragma unroll
    for (int p = 0; p < PB; ++p) {
      const int row = tid / QR + RP * (p0_ + p);
      if (p0_ + p < NP && m0 + row < a.M) finish(row, v[p], c[p]);
    }
  }
}

template <int QT, int MT, int CT, int NG, int EPI>
__device__ __forceinline__ void pfk_body(const GemmQArgs& a, int m0, int n0, int seg, int b0, int b1, int sp, int S, int tile, int ntile,
                                         int& last_flag) {
  using L = PfkLayout<QT, MT, CT, NG>;
  constexpr bool Q6 = L::Q6;
  constexpr int NX = L::NX, NWP = L::NWP, NWB = L::NWB, NW = L::NW, CW = CT / NG;
  extern __shared__ __attribute__((aligned(16))) uint8_t pf_smem0[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wv = wave & 3, cg = wave >> 2;  // its quarter of K, column group
  const int r32 = lane & 31, h = lane >> 5;
  const uint8_t* p0 = seg == 0 ? a.seg[0].p0 : (seg == 1 ? a.seg[1].p0 : a.seg[2].p0);
  const uint8_t* p1 = seg == 0 ? a.seg[0].p1 : (seg == 1 ? a.seg[1].p1 : a.seg[2].p1);
  const uint8_t* p2 = seg == 0 ? a.seg[0].p2 : (seg == 1 ? a.seg[1].p2 : a.seg[2].p2);
  const uint8_t* p3 = seg == 0 ? a.seg[0].p3 : (seg == 1 ? a.seg[1].p3 : a.seg[2].p3);
  const int col0 = n0 - (seg == 0 ? a.seg_n0[0] : (seg == 1 ? a.seg_n0[1] : a.seg_n0[2]));  // first row of the segment's planes
  const uint32_t nbk = (uint32_t)a.K >> 8;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(pf_lds_addr(pf_smem0));

  // ---- requests: this wave's pieces of an X slot (4 rows x 256 B each) and of a W block
  uint32_t xo[NX], co[L::NC], ro[L::NR], ho[Q6 ? L::NH : 1], dcol = 0;
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int row = 4 * (wave * NX + i) + (lane >> 4), u = (lane & 15) ^ (row & 15);
    xo[i] = ((uint32_t)min(m0 + row, a.M - 1) * (uint32_t)a.lda + (uint32_t)u * 8u) * 2u;
  }
#pragma unroll
  for (int i = 0; i < L::NC; ++i) {
    const int col = 8 * (wave * L::NC + i) + (lane >> 3), u = (lane & 7) ^ ((col >> 1) & 7);
    co[i] = (uint32_t)(col0 + col) * nbk * 128u + u * 16u;
  }
#pragma unroll
  for (int i = 0; i < L::NR; ++i) {
    const int col = 16 * ((wave * L::NR + i) & (L::PR - 1)) + (lane >> 2), u = lane & 3;
    ro[i] = (uint32_t)(col0 + col) * nbk * 16u + u * 4u;
    if constexpr (Q6) ho[i] = (uint32_t)(col0 + col) * nbk * 64u + (u ^ ((col >> 2) & 3)) * 16u;
  }
  const int pd = CT == 4 ? wave & 1 : 0;  // its piece of the dwords with d: 64 columns (32 columns: twice)
  if constexpr (Q6) dcol = (uint32_t)(col0 + 64 * pd + (CT == 1 ? r32 : lane)) * nbk;

  const int t0 = 2 * b0, tlast = 2 * b1 - 1, blast = b1 - 1, nk = 2 * (b1 - b0);
  // request i of this wave's NX of slot t (absolute), of its NWP of block b
  auto req_x = [&](int i, int t, uint32_t dst) __attribute__((always_inline)) {
    pfk_dma1((const uint8_t*)a.A + (size_t)(uint32_t)min(t, tlast) * 256, xo[i], dst + (wave * NX + i) * 1024);
  };
  auto req_w = [&](int i, int b, uint32_t dst) __attribute__((always_inline)) {
    const uint32_t bb = (uint32_t)min(b, blast);
    if (i < L::NC) {
      pfk_dma1(p0 + (size_t)bb * 128, co[i], dst + (wave * L::NC + i) * 1024);
    } else if (i < L::NC + L::NR) {
      const int k = i - L::NC;
      pfk_dma4((Q6 ? p2 : p1) + bb * 16, ro[k], dst + L::OFF_REC + ((wave * L::NR + k) & (L::PR - 1)) * 256);
    } else if (i < L::NC + L::NR + L::NH) {
      const int k = i - L::NC - L::NR;
      pfk_dma1(p1 + bb * 64, ho[Q6 ? k : 0], dst + L::OFF_HB + ((wave * L::NR + k) & (L::PR - 1)) * 1024);
    } else {
      pfk_dma4(p3, ((dcol + bb) >> 1) << 2, dst + L::OFF_D + pd * 256);
    }
  };
  auto issue_x = [&](int t, uint32_t dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NX; ++i) req_x(i, t, dst);
  };
  auto issue_w = [&](int b, uint32_t dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NWP; ++i) req_w(i, b, dst);
  };

  gf32x16 acc[MT][CW];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][c][e] = 0.f;

  // ---- LDS reads and decode.  Lane (r32, h), part j: k 16 h + 8 j .. of the wave's 32
  gbf16x8 fa[MT], fb[MT], bf0[CW], bf1[CW];
  const uint32_t xa = r32 * 256 + (((4 * wv + 2 * h) ^ (r32 & 15)) << 4);
  auto ld_x = [&](gbf16x8(&f)[MT], uint32_t slot, int j, int i) __attribute__((always_inline)) {
    f[i] = *(const gbf16x8*)(pf_smem0 + slot + (xa ^ (16 * j)) + 8192 * i);
  };
  const int hi = wv & 1;
  const uint32_t mm = hi ? 0x00f000f0u : 0x000f000fu;
  const float up = hi ? 1048576.f : 16777216.f;  // (a masked code read as an fp16 denormal: pf_dq8)
  gu32x4 rq[CW], rm[CW];  // 16 code bytes; record (Q6_K: high bits, scale, d)
  float ds[CW], dm[CW];
  const int wcol = 32 * cg * CW + r32;
  const uint32_t qa = wcol * 128 + (((2 * (wv >> 1) + h) ^ ((wcol >> 1) & 7)) << 4);
  const uint32_t ha = L::OFF_HB + wcol * 64 + (((wv >> 1) ^ ((wcol >> 2) & 3)) << 4) + 8 * h + 4 * hi;
  // half J of the block in the buffer at w
  auto ld_q = [&](auto jc, uint32_t w, int c) __attribute__((always_inline)) {
    rq[c] = *(const gu32x4*)(pf_smem0 + w + (qa ^ (64 * decltype(jc)::value)) + 4096 * c);
  };
  auto ld_m = [&](auto jc, uint32_t w, int b, int c) __attribute__((always_inline)) {
    constexpr int J = decltype(jc)::value;
    const uint8_t* m = pf_smem0 + w + L::OFF_REC + wcol * 16 + 512 * c;
    if constexpr (Q6) {
      rm[c][0] = *(const uint32_t*)(pf_smem0 + w + (ha ^ (32 * J)) + 2048 * c);
      rm[c][1] = (uint32_t)*(const int8_t*)(m + 8 * J + 4 * (wv >> 1) + 2 * h + hi);
      const int par = (int)(((uint32_t)(col0 + wcol + 32 * c) * nbk + (uint32_t)min(b, blast)) & 1u);
      rm[c][2] = *(const uint16_t*)(pf_smem0 + w + L::OFF_D + wcol * 4 + 128 * c + 2 * par);
    } else {
      rm[c] = *(const gu32x4*)m;
    }
  };
  auto scale = [&](auto jc, int c) __attribute__((always_inline)) {
    constexpr int J = decltype(jc)::value;
    if constexpr (Q6) {
      ds[c] = h2f((uint16_t)rm[c][2]) * (float)(int)rm[c][1];
      dm[c] = 32.f * ds[c];
      ds[c] *= 16777216.f;
    } else {
      asm volatile("" ::"v"(rm[c]));  // (the whole record lives until here: what is not used of it would be an address before it has arrived)
      const uint64_t two = J == 0 ? ((uint64_t)rm[c][2] << 32 | rm[c][1]) : ((uint64_t)rm[c][3] << 32 | rm[c][2]);
      const uint32_t f = (uint32_t)(two >> ((J == 0 ? 0 : 16) + 24 * (wv >> 1)));
      ds[c] = h2f((uint16_t)(rm[c][0] & 0xffff)) * up * (float)__builtin_amdgcn_ubfe(f, 6 * hi, 6);
      dm[c] = h2f((uint16_t)(rm[c][0] >> 16)) * (float)__builtin_amdgcn_ubfe(f, 12 + 6 * hi, 6);
    }
    asm volatile("" : "+v"(ds[c]), "+v"(dm[c]));
  };
  // weights 4 P .. of fragment part J of column c
  auto dec = [&](gbf16x8(&bf)[CW], auto jc, int c, int P) __attribute__((always_inline)) {
    constexpr int J = decltype(jc)::value;
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    uint32_t w = rq[c][2 * J + P];
    if constexpr (Q6) w = ((w >> (4 * hi)) & 0x0f0f0f0fu) | (((rm[c][0] >> (4 * J + 2 * P)) & 0x03030303u) << 4);
    const h2 x = __builtin_bit_cast(h2, Q6 ? w & 0x003f003fu : w & mm), y = __builtin_bit_cast(h2, Q6 ? (w >> 8) & 0x003f003fu : (w >> 8) & mm);
    const float q0 = fmaf((float)x[0], ds[c], -dm[c]), q2 = fmaf((float)x[1], ds[c], -dm[c]);
    const float q1 = fmaf((float)y[0], ds[c], -dm[c]), q3 = fmaf((float)y[1], ds[c], -dm[c]);
    uint32_t p0_ = pk_bf16(q0, q1), p1_ = pk_bf16(q2, q3);
    asm volatile("" : "+v"(p0_), "+v"(p1_));  // decoded here, beside these matrix instructions (the compiler sinks it to its use)
    gu32x4 t = __builtin_bit_cast(gu32x4, bf[c]);
    t[2 * P] = p0_;
    t[2 * P + 1] = p1_;
    bf[c] = __builtin_bit_cast(gbf16x8, t);
  };
  constexpr int NM = MT * CW;
  auto mfma = [&](const gbf16x8(&bf)[CW], const gbf16x8(&f)[MT], int k) __attribute__((always_inline)) {
    acc[k % MT][k / MT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf[k / MT], f[k % MT], acc[k % MT][k / MT], 0, 0, 0);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;

  // ---- pipeline: X slots three deep, W blocks NWB deep; before the barrier B(t) a wave has waited for its own pieces of slot t
  // and read its last of slot t - 1, so behind it slot t is whole and the buffers of t - 1 are free
  PfkRows<L::BM, NW> rows;
  if (a.nrm_in) rows.request(a, m0, wave, lane, lds0 + 2 * L::XS);
  const uint32_t w0a = lds0 + L::OFF_W;
  issue_w(b0, w0a);
  issue_x(t0, lds0);
#pragma unroll
  for (int p = 1; p < NWB - 1; ++p) issue_w(b0 + p, w0a + p * L::WB);
  issue_x(t0 + 1, lds0 + L::XS);
  pf_vmcnt<(NWB - 2) * NWP + NX>();
  if (a.nrm_in) {
    rows.done(a, wave, lane, pf_smem0 + 2 * L::XS);
    if constexpr (!L::KEEP) rows.put(wave, lane, (float*)(pf_smem0 + L::TOTAL - L::BM * 4));
  }
  pf_barrier();
#pragma unroll
  for (int c = 0; c < CW; ++c) {
    ld_q(I0{}, L::OFF_W, c);
    ld_m(I0{}, L::OFF_W, b0, c);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) ld_x(fa, 0, 0, i);
#pragma unroll
  for (int c = 0; c < CW; ++c) {
    scale(I0{}, c);
    dec(bf0, I0{}, c, 0);
    dec(bf0, I0{}, c, 1);
  }

  // a slot: its first 16 k beside the decode of the second, its second beside the reads and decode of the next slot's first.
  // Matrix instructions, decode and requests are dealt out by hand, one by one: left to itself the compiler groups each kind.
  // The requests that B(t + 1) lets go (slot t + 3; W block b + NWB where t is block b's second slot) go out over the second half of slot t
  // and the first of slot t + 1: a burst of them holds the wave until the address unit has taken each, 16 cycles and more
  uint32_t cur = 0, wb = 0;   // byte offsets of slot t and of its W block
  uint32_t free_x = 2 * L::XS, free_w = (NWB - 1) * L::WB;  // of the buffers that were let go last
  auto reqs = [&](auto jc, int t, int from, int to) __attribute__((always_inline)) {  // J: of slot t; requests [from, to) of its NREQ
    constexpr int J = decltype(jc)::value;
#pragma unroll
    for (int i = from; i < to; ++i) {
      if (J == 1 && i < NWP) req_w(i, (t >> 1) + NWB, w0a + free_w);
      else req_x(i - (J == 1 ? NWP : 0), t + 3, lds0 + free_x);
    }
  };
  constexpr int UB = NM > 2 ? 6 * NM / 10 : 1, UM = NM > 2 ? UB + (NM - UB + 1) / 2 : NM, UF = NM > 4 ? NM / 4 : 1;
  // of n things over the units [from, to): how many come before unit u
  auto part = [](int n, int u, int from, int to) constexpr { return u <= from ? 0 : (u >= to ? n : n * (u - from) / (to - from)); };
  auto step = [&](auto jc, int t) __attribute__((always_inline)) {
    constexpr int J = decltype(jc)::value;
    using JN = std::integral_constant<int, 1 - J>;
    constexpr int RP = NX + (J == 0 ? NWP : 0), RN = NX + (J == 1 ? NWP : 0);  // requests let go by B(t), by B(t + 1)
    const uint32_t nxt = cur == 2 * L::XS ? 0 : cur + L::XS;
    const uint32_t wn = J == 0 ? wb : (wb == (NWB - 1) * L::WB ? 0 : wb + L::WB);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 2 * NM; ++u) {
      if (u == UB) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        pf_vmcnt<J == 1 ? NX : NX + NWP>();
        pf_barrier();
        free_x = cur;
        free_w = wb;
        __builtin_amdgcn_sched_barrier(0);
      }
      if (u < NM) mfma(bf0, fa, u);
      else mfma(bf1, fb, u - NM);
#pragma unroll
      for (int i = part(MT, u, 0, UF); i < part(MT, u + 1, 0, UF); ++i) ld_x(fb, cur, 1, i);
#pragma unroll
      for (int i = part(2 * CW, u, UB, UM); i < part(2 * CW, u + 1, UB, UM); ++i) {
        if (i < CW) ld_q(JN{}, L::OFF_W + wn, i);
        else ld_m(JN{}, L::OFF_W + wn, t + 1 >> 1, i - CW);
      }
#pragma unroll
      for (int i = part(MT, u, NM, NM + UF); i < part(MT, u + 1, NM, NM + UF); ++i) ld_x(fa, nxt, 0, i);
      if (u < UB) reqs(JN{}, t - 1, part(RP, u + 2 * NM, UB, UB + 2 * NM), part(RP, u + 1 + 2 * NM, UB, UB + 2 * NM));
      else reqs(jc, t, part(RN, u, UB, UB + 2 * NM), part(RN, u + 1, UB, UB + 2 * NM));
#pragma unroll
      for (int i = part(2 * CW, u, 0, UB); i < part(2 * CW, u + 1, 0, UB); ++i) dec(bf1, I1{}, i / 2, i % 2);
#pragma unroll
      for (int i = part(3 * CW, u, NM, 2 * NM); i < part(3 * CW, u + 1, NM, 2 * NM); ++i) {
        if (i % 3 == 0) scale(JN{}, i / 3);
        else dec(bf0, I0{}, i / 3, i % 3 - 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = nxt;
    wb = wn;
  };
  reqs(I1{}, t0 - 1, 0, part(NX + NWP, 2 * NM, UB, UB + 2 * NM));
  for (int t = t0; t < t0 + nk; t += 2) {
    step(I0{}, t);
    step(I1{}, t + 1);
  }
  pf_vmcnt<0>();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  pfk_close<MT, CT, NG, EPI, L::KEEP, L::TOTAL>(a, acc, m0, n0, sp, S, tile, ntile, last_flag, rows);
}

template <int QT0, int QT1, int MT, int CT, int NG, int EPI>
__global__ void __launch_bounds__(256 * NG) __attribute__((amdgpu_waves_per_eu(NG, NG))) gemm_pfk_kernel(GemmQArgs a) {
  constexpr int BM = 32 * MT, BN = 32 * CT;
  const int nM = (a.M + BM - 1) / BM, ntile = a.N / BN * nM, S = gridDim.y, sp = blockIdx.y;
  const int L = xcd_remap(blockIdx.x, ntile), tn = L / nM, tm = L - tn * nM;  // (a column tile's row tiles: W once from memory)
  const int m0 = tm * BM, n0 = tn * BN;
  int seg = 0;
  if (a.nseg > 1 && n0 >= a.seg_n0[1]) seg = 1;
  if (a.nseg > 2 && n0 >= a.seg_n0[2]) seg = 2;
  const int nb = a.K / 256;
  const int b0 = sp * nb / S, b1 = (sp + 1) * nb / S;
  __shared__ int last_flag;
  if constexpr (QT0 != QT1) {
    if (seg == a.nseg - 1) {
      pfk_body<QT1, MT, CT, NG, EPI>(a, m0, n0, seg, b0, b1, sp, S, L, ntile, last_flag);
      return;
    }
  }
  pfk_body<QT0, MT, CT, NG, EPI>(a, m0, n0, seg, b0, b1, sp, S, L, ntile, last_flag);
}

template <int QT0, int QT1, int MT, int CT, int NG>
void pfk_launch(const GemmQArgs& a, int S, hipStream_t st) {
  constexpr int lds = std::max(PfkLayout<QT0, MT, CT, NG>::TOTAL, PfkLayout<QT1, MT, CT, NG>::TOTAL);
  const dim3 grid((a.N / (32 * CT)) * ((a.M + 32 * MT - 1) / (32 * MT)), S), block(256 * NG);
  switch (a.epi) {
    case GEPI_STORE: hipLaunchKernelGGL((gemm_pfk_kernel<QT0, QT1, MT, CT, NG, GEPI_STORE>), grid, block, lds, st, a); break;
    case GEPI_ACCUM: hipLaunchKernelGGL((gemm_pfk_kernel<QT0, QT1, MT, CT, NG, GEPI_ACCUM>), grid, block, lds, st, a); break;
    case GEPI_QKV: hipLaunchKernelGGL((gemm_pfk_kernel<QT0, QT1, MT, CT, NG, GEPI_QKV>), grid, block, lds, st, a); break;
    case GEPI_ACCUM_NORM:
      if constexpr (QT0 == QT1 && CT > 1) hipLaunchKernelGGL((gemm_pfk_kernel<QT0, QT1, MT, CT, NG, GEPI_ACCUM_NORM>), grid, block, lds, st, a);
      break;
    default:
      if constexpr (QT0 == QT1) hipLaunchKernelGGL((gemm_pfk_kernel<QT0, QT1, MT, CT, NG, GEPI_SWIGLU_BF16>), grid, block, lds, st, a);
      break;
  }
}

}  // namespace aios
