// Prefill GEMM with K over the waves (gemm_pfk.h), bf16 weights:
//   C[M][N] (epilogue) = A[M][K] (bf16) x W[N][K]^T
//
// The tiles, the meeting of the partial sums and the slices of K are gemm_pfk.h's.  X and W lie side by side in slots of 128 k, rows of
// 256 bytes each; of both a wave reads the 32 k that are its own.
// Bound: from 33 to ~200 rows the weights and ~5 us of launch, first loads and output; above, L2 and LDS traffic beside the matrix
// instructions.  Weights from memory, us, the best of the column-split tiles (gemm_pf.h) -> of these:
//   2560 x 2048, 50 / 130 / 300 rows 9.5 -> 7.8, 11.6 -> 7.3, 13.8 -> 9.1    2048 x 2048, 130 / 300 / 700 rows 9.7 -> 6.9, 11.8 -> 9.4, 17.8 -> 14.6
//   11264 x 2048 SwiGLU, 50 / 130 / 300 rows 19.3 -> 12.7, 22.0 / 22.5, 27.1 / 31.9    2048 x 8704, 50 / 130 / 700 rows 14.2 -> 11.6, 19.0 -> 15.9, 43.3 -> 39.5
// Wide products from ~200 rows and all from ~1500 keep the others (10496 x 2048, 1500 rows: 69 / 110): which runs is timed at load.
// Prompts, ms: TinyLlama bf16, 60 / 130 / 400 / 1000 tokens 1.68 -> 1.48, 1.99 -> 1.77, 2.89 -> 2.45, 4.58 -> 4.06; Seledra, 130 / 400 /
// 1000 tokens 2.77 -> 2.44, 4.23 -> 3.78, 7.20 -> 6.52 (with vector stores in the 8-wave tiles).
#include "gemm_pfk.h"

namespace aios {

template <int MT, int CT, int NG>
struct PfkbLayout {
  static constexpr int BM = 32 * MT, BN = 32 * CT, XS = BM * 256, SLOT = XS + BN * 256;
  static constexpr int NS = PFK_LDS / SLOT < 4 ? PFK_LDS / SLOT : 4;
  static constexpr int NW = 4 * NG, NX = BM / 4 / NW, NB = BN / 4 / NW, NR = NX + NB;  // waves; DMA requests a wave, per slot
  static constexpr int RED_BYTES = 2 * 4 * 32 * BN * 4 + BM * 4;
  static constexpr int USED = NS * SLOT + BM * 4, TOTAL = USED > RED_BYTES ? USED : RED_BYTES;
  static_assert(NS >= 2 && TOTAL <= PFK_LDS && NX * 4 * NW == BM && NB * 4 * NW == BN, "pfkb slots");
};

template <int MT, int CT, int NG, int EPI>
__global__ void __launch_bounds__(256 * NG) __attribute__((amdgpu_waves_per_eu(NG, NG))) gemm_pfkb_kernel(GemmQArgs a) {
  using L = PfkbLayout<MT, CT, NG>;
  constexpr int BM = L::BM, BN = L::BN, NS = L::NS, NX = L::NX, NR = L::NR, CW = CT / NG, NM = MT * CW;
  extern __shared__ __attribute__((aligned(16))) uint8_t pf_smem0[];
  __shared__ int last_flag;
  const int nM = (a.M + BM - 1) / BM, ntile = a.N / BN * nM, S = gridDim.y, sp = blockIdx.y;
  const int tile = xcd_remap(blockIdx.x, ntile), tn = tile / nM, tm = tile - tn * nM;
  const int m0 = tm * BM, n0 = tn * BN;
  int seg = 0;
  if (a.nseg > 1 && n0 >= a.seg_n0[1]) seg = 1;
  if (a.nseg > 2 && n0 >= a.seg_n0[2]) seg = 2;
  const int t0 = (int)((long)sp * (a.K / 128) / S), t1 = (int)((long)(sp + 1) * (a.K / 128) / S), tlast = t1 - 1;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wv = wave & 3, cg = wave >> 2;  // its quarter of K, column group
  const int r32 = lane & 31, h = lane >> 5;
  const uint8_t* p0 = seg == 0 ? a.seg[0].p0 : (seg == 1 ? a.seg[1].p0 : a.seg[2].p0);
  const int col0 = n0 - (seg == 0 ? a.seg_n0[0] : (seg == 1 ? a.seg_n0[1] : a.seg_n0[2]));
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(pf_lds_addr(pf_smem0));

  // ---- requests: this wave's pieces of a slot (4 rows x 256 B each; 16-B units swizzled by the row)
  uint32_t off[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int row = 4 * (wave * (i < NX ? NX : L::NB) + (i < NX ? i : i - NX)) + (lane >> 4), u = (lane & 15) ^ (row & 15);
    off[i] = (i < NX ? (uint32_t)min(m0 + row, a.M - 1) * (uint32_t)a.lda : (uint32_t)(col0 + row) * (uint32_t)a.K) * 2u + (uint32_t)u * 16u;
  }
  auto req = [&](int i, int t, uint32_t dst) __attribute__((always_inline)) {
    const uint8_t* from = (i < NX ? (const uint8_t*)a.A : p0) + (size_t)(uint32_t)min(t, tlast) * 256;
    pfk_dma1(from, off[i], lds0 + dst + (i < NX ? (wave * NX + i) * 1024 : L::XS + (wave * L::NB + i - NX) * 1024));
  };

  gf32x16 acc[MT][CW];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][c][e] = 0.f;

  // ---- fragments.  Lane (r32, h), part j: k 16 h + 8 j .. of the wave's 32, of X and W alike
  gbf16x8 fa[MT], fb[MT], wa[CW], wb[CW];
  const uint32_t xa = r32 * 256 + (((4 * wv + 2 * h) ^ (r32 & 15)) << 4);
  auto rd = [&](gbf16x8(&f)[MT], gbf16x8(&w)[CW], uint32_t slot, int j, int i) __attribute__((always_inline)) {
    if (i < CW) w[i] = *(const gbf16x8*)(pf_smem0 + slot + L::XS + (xa ^ (16 * j)) + 8192 * (cg * CW + i));
    else f[i - CW] = *(const gbf16x8*)(pf_smem0 + slot + (xa ^ (16 * j)) + 8192 * (i - CW));
  };
  auto mfma = [&](const gbf16x8(&w)[CW], const gbf16x8(&f)[MT], int k) __attribute__((always_inline)) {
    acc[k % MT][k / MT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[k / MT], f[k % MT], acc[k % MT][k / MT], 0, 0, 0);
  };

  // ---- pipeline: NS slots.  Before the barrier B(t + 1), in step t, a wave has waited for its own pieces of slot t + 1 and read its
  // last of slot t; the requests that B(t + 1) lets go, slot t + NS, go out over the rest of step t and the start of step t + 1
  constexpr int UB = NM > 2 ? 6 * NM / 10 : 1, UF = NM > 4 ? NM / 4 : 1;
  auto part = [](int n, int u, int from, int to) constexpr { return u <= from ? 0 : (u >= to ? n : n * (u - from) / (to - from)); };
  constexpr int PA = part(NR, 2 * NM, UB, UB + 2 * NM);  // of them, in step t
  PfkRows<BM, L::NW> rows;
  if (a.nrm_in) rows.request(a, m0, wave, lane, lds0 + (NS - 1) * L::SLOT);
#pragma unroll
  for (int p = 0; p < NS - 1; ++p)
#pragma unroll
    for (int i = 0; i < NR; ++i) req(i, t0 + p, p * L::SLOT);
  pf_vmcnt<(NS - 2) * NR>();
  if (a.nrm_in) {
    rows.done(a, wave, lane, pf_smem0 + (NS - 1) * L::SLOT);
    rows.put(wave, lane, (float*)(pf_smem0 + L::TOTAL - BM * 4));
  }
#pragma unroll
  for (int i = 0; i < PA; ++i) req(i, t0 + NS - 1, (NS - 1) * L::SLOT);
  pf_barrier();
#pragma unroll
  for (int i = 0; i < MT + CW; ++i) rd(fa, wa, 0, 0, i);
  uint32_t cur = 0, before = (NS - 1) * L::SLOT;
  for (int t = t0; t < t1; ++t) {
    const uint32_t nxt = cur == (NS - 1) * L::SLOT ? 0 : cur + L::SLOT;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 2 * NM; ++u) {
      if (u == UB) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        pf_vmcnt<(NS - 2) * NR>();
        pf_barrier();
        __builtin_amdgcn_sched_barrier(0);
      }
      if (u < NM) mfma(wa, fa, u);
      else mfma(wb, fb, u - NM);
#pragma unroll
      for (int i = part(MT + CW, u, 0, UF); i < part(MT + CW, u + 1, 0, UF); ++i) rd(fb, wb, cur, 1, i);
#pragma unroll
      for (int i = part(MT + CW, u, NM, NM + UF); i < part(MT + CW, u + 1, NM, NM + UF); ++i) rd(fa, wa, nxt, 0, i);
#pragma unroll
      for (int i = part(NR, u < UB ? u + 2 * NM : u, UB, UB + 2 * NM); i < part(NR, u < UB ? u + 1 + 2 * NM : u + 1, UB, UB + 2 * NM); ++i) {
        if (u < UB) req(i, t - 1 + NS, before);
        else req(i, t + NS, cur);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    before = cur;
    cur = nxt;
  }
  pf_vmcnt<0>();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  pfk_close<MT, CT, NG, EPI, false, L::TOTAL>(a, acc, m0, n0, sp, S, tile, ntile, last_flag, rows);
}

// bm x bn tiles divide N and every segment (pf_plan_ok).  Slots of 128 k; 32-bit offsets into X and W
bool pfkb_serves(const GemmQArgs& a, int bm, int bn, int S) {
  if (!pfk_epi_ok(a, bn)) return false;
  if (S < 1 || S > a.K / 128 || a.K % 128) return false;
  if ((size_t)a.M * a.lda * 2 >= 0xfffffff0u) return false;
  for (int s = 0; s < a.nseg; ++s)
    if (a.seg[s].qtype != QT_BF16 || (size_t)a.seg[s].rows * a.K * 2 >= 0xfffffff0u || ((uintptr_t)a.seg[s].p0 & 15)) return false;
  if (!pfk_slabs_ok(a, bm, bn, S)) return false;
  return pfk_tile(bm, bn, [](auto, auto, auto) { return true; });
}

bool pfkb_run(const GemmQArgs& a, int bm, int bn, int S, hipStream_t st) {
  return pfk_tile(bm, bn, [&](auto mt, auto ct, auto ng) {
    constexpr int MT = decltype(mt)::value, CT = decltype(ct)::value, NG = decltype(ng)::value;
    constexpr int lds = PfkbLayout<MT, CT, NG>::TOTAL;
    const dim3 grid((a.N / bn) * ((a.M + bm - 1) / bm), S), block(256 * NG);
    switch (a.epi) {
      case GEPI_STORE: hipLaunchKernelGGL((gemm_pfkb_kernel<MT, CT, NG, GEPI_STORE>), grid, block, lds, st, a); break;
      case GEPI_ACCUM: hipLaunchKernelGGL((gemm_pfkb_kernel<MT, CT, NG, GEPI_ACCUM>), grid, block, lds, st, a); break;
      case GEPI_QKV: hipLaunchKernelGGL((gemm_pfkb_kernel<MT, CT, NG, GEPI_QKV>), grid, block, lds, st, a); break;
      case GEPI_ACCUM_NORM:
        if constexpr (CT > 1) hipLaunchKernelGGL((gemm_pfkb_kernel<MT, CT, NG, GEPI_ACCUM_NORM>), grid, block, lds, st, a);
        break;
      case GEPI_STORE16: hipLaunchKernelGGL((gemm_pfkb_kernel<MT, CT, NG, GEPI_STORE16>), grid, block, lds, st, a); break;
      default: hipLaunchKernelGGL((gemm_pfkb_kernel<MT, CT, NG, GEPI_SWIGLU_BF16>), grid, block, lds, st, a); break;
    }
    return true;
  });
}

}  // namespace aios
