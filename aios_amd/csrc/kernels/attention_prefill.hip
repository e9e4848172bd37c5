// Causal flash attention for prefill (prefill column: "[T,H,hd]^2 causal
// flash-attention (MFMA)"), reading K/V from the bf16 KV cache the QKV epilogue just wrote, so a
// chunk of T new tokens attends over every cached position [0, start + T) of its slot.
//
// GQA packing: a workgroup owns one KV head and BQ = 128 / G query positions x all G query heads
// of that group = 128 query rows, so every K/V tile staged in LDS is used by 4x32 rows.  Wave w
// owns rows [32w, 32w + 32) (row = position * G + head).  Per 64-key tile:
//   S^T[key][row] = K Q^T   -- v_mfma_f32_32x32x16_bf16, K rows straight from LDS (A operand),
//                              Q^T from registers (B operand, loaded once, pre-scaled by
//                              scale*log2 e): the lane then holds one query row's 32 keys, so
//                              the row max / sum need one cross-half shuffle, not a 32-lane tree.
//   O^T[dim][row] += V^T P^T -- P^T is taken straight from the S^T accumulator registers: the key
//                              order of the k-dimension is permuted (rho below) to match the
//                              accumulator layout; V is staged ROW-major (16-byte stores) and the
//                              V^T fragment is two gfx950 transposed LDS reads (ds_read_b64_tr_b16:
//                              4 keys x 16 dims per 16-lane group, delivered column-major) at rho.
//                              (Round 2 staged V transposed with 2-byte stores: 32 ds_write_b16
//                              per thread per tile and the kernel's worst bank conflicts.)
// Online softmax per row in the log2 domain; fully masked rows cannot occur (key 0 <= pos).
// Output: bf16 [T][n_heads * hd] (the O-projection GEMM's A operand).
//
// Splits over the keys: a launch of few (query block, KV head) workgroups -- a further turn of a
// conversation, 300 new tokens behind 6000 cached ones: 80 workgroups for 256 CUs, each 98 tiles long --
// cuts every workgroup's tiles into a.ns runs.  Each run leaves its unnormalised O (fp32), row max and
// row sum in the workspace and attn_prefill_combine adds them up (fp32, in the order of the runs): 160 us
// -> 62 us for both launches there (32 / 8 heads of 128, fp8 cache).
//
// VALU diet (rocprofv3 PMC at 2048 tokens: ~12 VALU instructions per MFMA, 129 TF/s): bf16 packing
// in hardware (v_cvt_pk_bf16_f32, not a software RNE with a NaN test), raw v_exp_f32 (ocml's
// exp2f adds range scaling), and the O rescale skipped when no row max of the wave moved.
#include "../common.h"
#include "../ops.h"
#include "gemm_common.h"

namespace aios {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
// native vector type for register arrays (HIP's uint4 is a struct; arrays of it copied with
// memcpy defeat SROA and land in scratch)
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef short v8i16_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ float raw_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

constexpr int FP_KT = 64;  // keys per tile

typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));

// the tiles of run z of the ns runs over the keys that query block [t0, t0 + BQ) sees
struct FpRun {
  int kt0, kt1;
};
__device__ __forceinline__ FpRun fp_run(int start, int T, int t0, int BQ, int ns, int z) {
  const int ntiles = (start + min(T, t0 + BQ) - 1) / FP_KT + 1;  // to the block's highest query position
  const int per = (ntiles + ns - 1) / ns;
  return {min(z * per, ntiles), min((z + 1) * per, ntiles)};
}

// F8: the pool holds fp8 e4m3 codes (EngineConfig::kv_fp8): the tile loads move half the bytes and
// staging converts the codes to bf16 (exact; v_cvt_scalef32_pk_bf16_fp8 at scale 1 -- its scale
// operand is applied as a power of two, so the layer's K scale is folded into q and its V scale into
// the output instead) -- the LDS tiles and the MFMA math are the bf16 kernel's
// KG = 2 (prefill_groups): eight waves, of which the first four take the even tiles of the workgroup's 128 rows and the others the odd ones;
// their sums meet in LDS at the end.
template <int HD, int G, bool F8, int KG>
__global__ void __launch_bounds__(256 * KG) __attribute__((amdgpu_waves_per_eu(2, 2))) attn_prefill_kernel(AttnPrefillArgs a) {
  constexpr int NT = 256 * KG;
  constexpr int BQ = 128 / G;          // query positions per workgroup
  constexpr int QS = HD / 16;          // k-steps of the S MFMA
  constexpr int OT = HD / 32;          // O^T accumulator tiles (32 dims each)
  constexpr int KROW = HD + 8;         // padded LDS row (bf16) of the K tile
  // padded LDS row (bf16) of the row-major V tile: a 16-lane transposed read takes 4 rows x 4
  // 8-byte column chunks and its 32-lane half two such groups 16 dims apart; rows HD + 32 elements
  // apart put the 4 rows 16 banks apart (mod 64) and the two groups 8 banks apart: conflict-free
  constexpr int VROW = HD + 32;
  // two LDS buffers (dynamic) of KG tiles (37 KB for HD 128), K then V in each
  constexpr int TILE_ELEMS = FP_KT * (KROW + VROW);
  extern __shared__ __attribute__((aligned(16))) bf16_t fp_smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, half = lane >> 5;
  const int wr = __builtin_amdgcn_readfirstlane(wave & 3), kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(wave >> 2);
  // An XCD works on as few KV heads as there are for it, so their K and V stay in its L2: m XCDs share a list of hx heads' (query
  // block, run) items, the longest first.  Causal balance: where the list fills its CUs twice at most, what comes after the
  // first 32 m items (a CU's second workgroup) goes from the shortest up, so every CU gets about the same number of tiles.
  // us, heads over all XCDs -> so: 1852 tokens behind 2048, 32 / 8 heads of 128 127 -> 112; 300 behind 6000, fp8, six runs 53 -> 49;
  // 1500 tokens, 32 / 4 heads of 64 35 -> 27.
  const int nx = (a.T + BQ - 1) / BQ, m = 1 << a.lm;
  const int xcd = blockIdx.x & 7, W = a.hx * nx * a.ns, w = ((blockIdx.x >> 3) << a.lm) + (xcd & (m - 1));
  if (w >= W) return;
  int item = KG > 1 || w < 32 * m || W > 64 * m ? w : W - 1 - (w - 32 * m);  // (of eight waves one workgroup fits a CU)
  int kvh = xcd >> a.lm, run_z = 0;
  if (a.hx > 1) {  // (divisions only where there is something to divide: 0.3 us of a short prompt's 6)
    kvh = kvh * a.hx + item % a.hx;
    item /= a.hx;
  }
  if (a.ns > 1) {
    run_z = item % a.ns;
    item /= a.ns;
  }
  const int qb = nx - 1 - item;
  const int T = a.T, start = a.start;
  const int t0 = qb * BQ;
  // this lane's query row (column of S^T / O^T)
  const int row = wr * 32 + l32;
  const int tq = t0 + row / G, g = row % G;
  const bool qvalid = tq < T;
  const int tql = qvalid ? tq : T - 1;
  const int qpos = start + tql;  // absolute position: keys <= qpos are visible
  const int h = kvh * G + g;

  // Q^T fragments (B operand): lane holds Q[row][16s + 8*half + 0..7] for s = 0..QS-1
  bf16x8_t qf[QS];
  {
    const float* qp = a.q + ((size_t)tql * a.n_heads + h) * HD + 8 * half;
    const float sc = a.scale * 1.4426950408889634f * (F8 ? a.kv_scale_k : 1.f);
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      const float4 x0 = *(const float4*)(qp + 16 * s), x1 = *(const float4*)(qp + 16 * s + 4);
      const uint4 u = make_uint4(pk_bf16(x0.x * sc, x0.y * sc), pk_bf16(x0.z * sc, x0.w * sc),
                                 pk_bf16(x1.x * sc, x1.y * sc), pk_bf16(x1.z * sc, x1.w * sc));
      __builtin_memcpy(&qf[s], &u, 16);
    }
  }

  f32x16_t o[OT];
#pragma unroll
  for (int i = 0; i < OT; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[i][e] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // paged KV: 64-key tile kt lives in block bt[kt / 2] at key offset (kt % 2) * 64
  static_assert(KV_BLOCK == 2 * FP_KT, "two prefill key tiles per paged KV block");
  const int maxb = a.max_ctx / KV_BLOCK;
  const size_t blk_stride = (size_t)a.n_kv_heads * KV_BLOCK * HD;
  constexpr int ES = F8 ? 1 : 2;  // bytes per cached element
  const uint8_t* kc = (const uint8_t*)a.k_cache + (size_t)kvh * KV_BLOCK * HD * ES;
  const uint8_t* vc = (const uint8_t*)a.v_cache + (size_t)kvh * KV_BLOCK * HD * ES;
  // this run's tiles [kt0, kt1) of the block's (a.ns == 1: all of them)
  const FpRun run = fp_run(start, T, t0, BQ, a.ns, run_z);
  const int kt0 = run.kt0, kt1 = run.kt1;
  if (kt0 >= kt1) return;  // (uniform; the combine counts the runs the same way)
  const int klim = min(qpos, kt1 * FP_KT - 1);  // keys this lane sees in this run
  // ... and the least of them over the wave's rows: a tile that ends there needs no mask
  const int klim_w = min(start + min(T - 1, t0 + wr * 32 / G), kt1 * FP_KT - 1);
  const int khi_w = start + min(T - 1, t0 + (wr * 32 + 31) / G);  // the most of them: tiles behind it are nothing to this wave

  // tile loader: 64 keys x HD dims of K and of V, 16 B per piece, into register buffer r (2 of
  // them: tile kt + 2 is requested while tile kt is computed, so two tiles of math cover the
  // memory latency); stage() writes one buffer to an LDS tile buffer
  constexpr int PIECES = FP_KT * HD / 8;      // 16-B pieces per tensor per tile
  constexpr int PPT = KG * PIECES / NT;       // per thread, of KG tiles
  using PT = typename std::conditional<F8, u32x2_t, u32x4_t>::type;  // one 8-element piece
  struct Regs {
    PT k[PPT], v[PPT];
  };
  const int nt_last = kt1 - 1;
  static_assert(PIECES % NT == 0, "a thread's pieces of a tile");
  auto load = [&](Regs& r, int kt0_) {  // tiles kt0_ .. + KG - 1
    size_t tbase[KG];  // (once a tile: once a piece was a scalar load and a wait for each)
    static_for<KG>([&](auto I) {
      constexpr int t = decltype(I)::value;
      const int kt = min(kt0_ + t, nt_last);  // (clamped: the pipeline's tail requests are re-reads, never unmapped blocks)
      tbase[t] = (size_t)kv_block(a.block_table, maxb, a.slot, kt * FP_KT) * blk_stride + (size_t)(kt & 1) * FP_KT * HD;
    });
    static_for<PPT>([&](auto I) {
      constexpr int i = decltype(I)::value, t = i / (PIECES / NT);
      const int idx = tid + NT * (i % (PIECES / NT)), key = idx / (HD / 8), c = idx % (HD / 8);
      const size_t off = (tbase[t] + (size_t)key * HD + c * 8) * ES;
      r.k[i] = *(const PT*)(kc + off);
      r.v[i] = *(const PT*)(vc + off);
    });
  };
  auto stage = [&](const Regs& r, bf16_t* buf0) {
    static_for<PPT>([&](auto I) {
      constexpr int i = decltype(I)::value, t = i / (PIECES / NT);
      const int idx = tid + NT * (i % (PIECES / NT)), key = idx / (HD / 8), c = idx % (HD / 8);
      bf16_t* sK = buf0 + t * TILE_ELEMS;
      bf16_t* sV = sK + FP_KT * KROW;
      if constexpr (F8) {
        auto cv = [](u32x2_t w) {
          u32x4_t o;
          o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[0], 1.f, false));
          o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[0], 1.f, true));
          o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[1], 1.f, false));
          o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[1], 1.f, true));
          return o;
        };
        *(u32x4_t*)(sK + key * KROW + c * 8) = cv(r.k[i]);
        *(u32x4_t*)(sV + key * VROW + c * 8) = cv(r.v[i]);
      } else {
        *(u32x4_t*)(sK + key * KROW + c * 8) = r.k[i];
        *(u32x4_t*)(sV + key * VROW + c * 8) = r.v[i];
      }
    });
  };
  // one 64-key tile of math on LDS buffer buf.  ALL: every wave of the workgroup sees keys of the tile, as it does of those up to the first row
  auto math = [&](const bf16_t* buf0, int kt_, auto ALL) {
    const bf16_t* buf = buf0 + kg * TILE_ELEMS;
    const int kt = kt_ + kg;
    if constexpr (!decltype(ALL)::value)
      if ((KG > 1 && kt >= kt1) || kt * FP_KT > khi_w) return;  // (uniform over the wave)
    const bf16_t* sK = buf;
    const bf16_t* sV = buf + FP_KT * KROW;
    // ---- S^T = K Q^T for the tile's two 32-key halves
    f32x16_t st[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int e = 0; e < 16; ++e) st[t][e] = 0.f;
      const bf16_t* kr = sK + (t * 32 + l32) * KROW + 8 * half;
#pragma unroll
      for (int s = 0; s < QS; ++s) {
        const uint4 u = *(const uint4*)(kr + 16 * s);
        bf16x8_t kf;
        __builtin_memcpy(&kf, &u, 16);
        st[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[s], st[t], 0, 0, 0);
      }
    }
    // ---- causal mask + online softmax for this lane's row (32 of the 64 keys; partner lane^32)
    const int kbase = kt * FP_KT;
    if (kbase + FP_KT - 1 > klim_w) {  // (wave-uniform)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (kbase + t * 32 + (r & 3) + 8 * (r >> 2) + 4 * half > klim) st[t][r] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[t][r]);
    mx = lane_xor32(mx, LaneMax{});
    const float mx_run = fmaxf(m_run, mx);
    // -inf only where a run or key group has shown this row no key yet (never with one of each: key 0 is visible): p = 0 then
    const float mn = (KG > 1 || a.ns > 1) && mx_run == -INFINITY ? 0.f : mx_run;
    const float alpha = raw_exp2(m_run - mn);  // exp2(-inf) = 0 on the first tile
    float ps = 0.f;
    uint32_t pb[2][8];  // P^T as packed bf16 pairs, accumulator order
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float p0 = raw_exp2(st[t][r] - mn), p1 = raw_exp2(st[t][r + 1] - mn);
        ps += p0 + p1;
        pb[t][r >> 1] = pk_bf16(p0, p1);
      }
    ps = lane_xor32(ps, LaneAdd{});
    l_run = l_run * alpha + ps;
    // the O rescale only when some row max of this wave moved (alpha == 1 on every lane otherwise)
    if (__any(mn != m_run)) {
#pragma unroll
      for (int i = 0; i < OT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] *= alpha;
    }
    m_run = mx_run;
    // ---- O^T += V^T P^T over 4 k-steps of 16 keys: step s uses accumulator half t = s/2,
    //      registers 8*(s%2) .. +7, i.e. keys rho = 16s + 4*half + {0..3} and 16s + 8 + 4*half + {0..3}
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int t = s >> 1, rb = (s & 1) * 4;
      const uint4 pu = make_uint4(pb[t][rb], pb[t][rb + 1], pb[t][rb + 2], pb[t][rb + 3]);
      bf16x8_t pf;
      __builtin_memcpy(&pf, &pu, 16);
#pragma unroll
      for (int i = 0; i < OT; ++i) {
        // lane 4q+p of each 16-lane group addresses key row (16s + 4 half + q), dims
        // 32 i + 16 (group & 1) + 4p .. +3; lane l32 receives dim 32 i + l32 of those 4 keys
        const bf16_t* va = sV + (16 * s + 4 * half + ((lane & 15) >> 2)) * VROW + i * 32 + 16 * ((lane >> 4) & 1) +
                           4 * (lane & 3);
        const v4i16_t x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16_t*)va);
        const v4i16_t x1 =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4i16_t*)(va + 8 * VROW));
        const v8i16_t xv = __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
        bf16x8_t vf;
        __builtin_memcpy(&vf, &xv, 16);
        o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, o[i], 0, 0, 0);
      }
    }
  };

  // Pipeline (with one register buffer, stage and two barriers per tile: 130-150 us per
  // 2k-token layer): two register buffers A / B and two LDS tile buffers L0 / L1, ONE barrier per
  // tile.  Iteration kt computes tile kt from L[kt & 1] while tile kt + 2 is requested into the
  // register buffer just staged, then stages tile kt + 1 into the other LDS buffer (last read two
  // iterations ago, before the previous barrier) and barriers.  Pairs without a branch, so that a tile's staging is dealt out over the one
  // before; an odd one behind them by itself (a fully masked tile to make a pair of it was 1.5 us of a short prompt's launch).
  // us, pairs with that tile / an exit behind every tile / so: 32 / 4 heads of 64, 23 tokens 6.0 / 4.9 / 4.8, 32 / 8 of 128, 130 tokens 10.1 / 9.2 / 9.1,
  // 711 (two key groups below) 23.7 / 22.8 / 21.5, 3000 102 / 102 / 95, 16 / 8 of 128, 4096 tokens 100 / 109 / 99, 3840 behind 500 111 / 119 / 110,
  // fp8, 16 / 16 of 128, 2304 behind 2000 104 / 116 / 103.  (Half of what the exits lost was the block table, looked up for every piece.)
  bf16_t* L0 = fp_smem;
  bf16_t* L1 = fp_smem + KG * TILE_ELEMS;
  Regs A, B;
  load(A, kt0);
  load(B, kt0 + KG);
  stage(A, L0);
  __syncthreads();
  int kt = kt0;
  for (; kt + 2 * KG <= kt1; kt += 2 * KG) {
    load(A, kt + 2 * KG);
    math(L0, kt, std::true_type{});
    stage(B, L1);
    __syncthreads();
    load(B, kt + 3 * KG);
    math(L1, kt + KG, std::true_type{});
    stage(A, L0);
    __syncthreads();
  }
  if (kt < kt1) math(L0, kt, std::false_type{});
  if (KG > 1 && kt + KG < kt1) {
    stage(B, L1);
    __syncthreads();
    math(L1, kt + KG, std::false_type{});
  }
  if constexpr (KG > 1) {  // ---- the second group's sums to the first
    static_assert(KG == 2, "two key groups");
    float* xo = (float*)fp_smem + wr * (OT * 16 * 64);
    float* xm = (float*)fp_smem + 4 * (OT * 16 * 64) + wr * 128;
    __syncthreads();  // every wave is done with its tiles
    if (kg) {
#pragma unroll
      for (int i = 0; i < OT; ++i)
#pragma unroll
        for (int r = 0; r < 16; r += 4) *(float4*)(xo + ((i * 4 + (r >> 2)) * 64 + lane) * 4) = make_float4(o[i][r], o[i][r + 1], o[i][r + 2], o[i][r + 3]);
      xm[lane] = m_run;
      xm[64 + lane] = l_run;
    }
    __syncthreads();
    if (kg) return;
    const float m1 = xm[lane], M = fmaxf(m_run, m1), M0 = M == -INFINITY ? 0.f : M;
    const float w0 = raw_exp2(m_run - M0), w1 = raw_exp2(m1 - M0);
    l_run = l_run * w0 + xm[64 + lane] * w1;
    m_run = M;
#pragma unroll
    for (int i = 0; i < OT; ++i)
#pragma unroll
      for (int r = 0; r < 16; r += 4) {
        const float4 x = *(const float4*)(xo + ((i * 4 + (r >> 2)) * 64 + lane) * 4);
        o[i][r] = o[i][r] * w0 + x.x * w1;
        o[i][r + 1] = o[i][r + 1] * w0 + x.y * w1;
        o[i][r + 2] = o[i][r + 2] * w0 + x.z * w1;
        o[i][r + 3] = o[i][r + 3] * w0 + x.w * w1;
      }
  }
  // ---- O^T[dim][row], dim = 32 i + (r&3) + 8 (r>>2) + 4 half
  if (a.ns > 1) {  // this run's part: O, row max and row sum in fp32
    if (qvalid) {
      const size_t pr = ((size_t)run_z * T + tq) * a.n_heads + h;
      float* op = a.ws + pr * HD;
#pragma unroll
      for (int i = 0; i < OT; ++i)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
          *(float4*)(op + i * 32 + 8 * (r >> 2) + 4 * half) = make_float4(o[i][r], o[i][r + 1], o[i][r + 2], o[i][r + 3]);
      if (half == 0) *(float2*)(a.ws + (size_t)a.ns * T * a.n_heads * HD + pr * 2) = make_float2(m_run, l_run);
    }
    return;
  }
  // ---- normalise and store bf16
  if (qvalid) {
    const float inv = (F8 ? a.kv_scale_v : 1.f) / l_run;
    bf16_t* op = a.out + (size_t)tq * a.ldo + (size_t)h * HD;
#pragma unroll
    for (int i = 0; i < OT; ++i)
#pragma unroll
      for (int r = 0; r < 16; r += 4) {
        const int d = i * 32 + 8 * (r >> 2) + 4 * half;
        const uint2 u = make_uint2(pk_bf16(o[i][r] * inv, o[i][r + 1] * inv), pk_bf16(o[i][r + 2] * inv, o[i][r + 3] * inv));
        *(uint2*)(op + d) = u;
      }
  }
}

// One wave per (token, head): its runs' O added up by their row maxima, normalised, stored as bf16.
// Bound by the partials' bytes (300 tokens, 32 heads of 128, 6 runs: 30 MB, most of them still cached).
template <int HD>
__global__ void __launch_bounds__(256) attn_prefill_combine(AttnPrefillArgs a, int BQ, float vscale) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int rows = a.T * a.n_heads;
  if (row >= rows) return;
  const int t = row / a.n_heads, h = row - t * a.n_heads;
  const FpRun r0 = fp_run(a.start, a.T, t - t % BQ, BQ, a.ns, 0);
  const int ntiles = (a.start + min(a.T, t - t % BQ + BQ) - 1) / FP_KT + 1;
  const int n = (ntiles + r0.kt1 - 1) / r0.kt1;  // runs that hold tiles (r0.kt1: tiles of a run)
  const float* ml = a.ws + (size_t)a.ns * rows * HD;
  float M = -INFINITY;
  for (int z = 0; z < n; ++z) M = fmaxf(M, ml[((size_t)z * rows + row) * 2]);
  constexpr int V = HD / 64;
  float L = 0.f, acc[V] = {};
#pragma unroll 4
  for (int z = 0; z < n; ++z) {
    const size_t pr = (size_t)z * rows + row;
    const float2 p = *(const float2*)(ml + pr * 2);
    const float w = raw_exp2(p.x - M);
    L += w * p.y;
    const float* op = a.ws + pr * HD + lane * V;
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] += w * op[j];
  }
  const float inv = vscale / L;
  bf16_t* out = a.out + (size_t)t * a.ldo + (size_t)h * HD + lane * V;
  if constexpr (V == 2) *(uint32_t*)out = pk_bf16(acc[0] * inv, acc[1] * inv);
  else *out = f32_to_bf16(acc[0] * inv);
}

bool attn_prefill_supports(int n_heads, int n_kv_heads, int head_dim) {
  if (n_kv_heads <= 0 || n_heads % n_kv_heads) return false;
  const int G = n_heads / n_kv_heads;
  return (head_dim == 64 || head_dim == 128) && (G == 1 || G == 2 || G == 4 || G == 8);
}

// Workgroups that a launch split over the keys has at most: two per CU (the two LDS tile buffers), and
// one more wave of them would only lengthen the tail.
constexpr int FP_WG = 512;
// Tiles of a run at the least: below, the partials' traffic and the second launch cost what the run saves.
constexpr int FP_RUN = 8;
// A launch with room for fewer than four runs stays whole: causal blocks differ in length, so its CUs are kept busy
// by the long ones anyway, and two or three runs only pay the second launch (TinyLlama, 909 tokens behind 179 in two
// runs: the whole prefill 0.9 % slower; Mistral, 300 behind 6000 in six: 15035 -> 11880 us).

// KG: key groups of a workgroup; of eight waves one is resident on a CU, of four two
static int prefill_runs(const AttnPrefillArgs& a, int BQ, int KG) {
  const int wg = (a.T + BQ - 1) / BQ * a.n_kv_heads, ntiles = (a.start + a.T - 1) / FP_KT + 1, slots = std::min(FP_WG, 2 * device_cu_count());
  if (4 * wg > slots) return 1;
  const int ns = std::min(slots / (KG * wg), ntiles / FP_RUN);
  const size_t need = (size_t)ns * a.T * a.n_heads * (a.head_dim + 2) * sizeof(float);
  return ns > 1 && a.ws && need <= a.ws_bytes ? ns : 1;
}

// Key groups of a launch with ten tiles or more.  A CU holds one workgroup of two groups or two of one, so two groups win where no CU has a second
// workgroup, or a second one that is much shorter than the first, and lose where it is as long: then it is two rounds in a row.
// us in one / two groups:
// Workgroups for every CU at most: 32 / 8 heads of 128, 512 tokens 17.1 / 17.5 (eight tiles), 1024 28.1 / 26.3, behind 2000 73.3 / 61.4.
// More: 1504 tokens 41.7 / 38.0, 16 / 8 of 128, 3520 82.4 / 74.0, 4096 97.7 / 91.6, fp8, 8 / 2 of 128, 4800 behind 2000 150 / 116; but the fuller the second round 1920
// 52.0 / 54.2, 2048 of 32 / 4 of 64 33.1 / 34.0; with G = 8, whose workgroups have few tiles, 64 / 8 of 128, 1024 tokens 33.5 / 38.4; and behind a
// prefix, which makes all of them long, 2048 behind 2000 120 / 127, 32 / 4 of 64 73.5 / 80.7.
// In runs, which fill the CUs in either form, two groups halve the partials, but the runs of late rows are the longer ones: 32 / 8 of 128, 512 behind
// 2000 44.3 / 41.4, 16 / 8 of 64, 512 behind 4000 35.0 / 27.2; but 4 / 1 of 128, 4096 tokens 44.9 / 50.5; and where their whole runs fill fewer
// CUs, fp8, 16 / 8 of 128, 768 behind 4000 53.0 / 57.6 (96 workgroups in five runs, or in two of two groups).
static int prefill_groups(const AttnPrefillArgs& a, int BQ) {
  const int wg = (a.T + BQ - 1) / BQ * a.n_kv_heads, ntiles = (a.start + a.T - 1) / FP_KT + 1, cus = device_cu_count();
  if (ntiles < 10) return 1;
  const int runs = prefill_runs(a, BQ, 1);
  if (runs > 1) return 2 * prefill_runs(a, BQ, 2) >= runs && 2L * a.T <= 3L * a.start && a.T <= 2048 ? 2 : 1;
  if (wg <= cus) return 2;
  return a.T >= 17 * FP_KT && 4L * (wg - cus) * (a.T + a.start) <= (a.T < 36 * FP_KT ? 3L : 4L) * cus * (a.T - a.start) ? 2 : 1;
}

void attn_prefill_form(const AttnPrefillArgs& a, int* groups, int* runs) {
  const int BQ = 128 / (a.n_heads / a.n_kv_heads);
  *groups = prefill_groups(a, BQ);
  *runs = prefill_runs(a, BQ, *groups);
}

// FP_WG workgroups of 128 rows each, O and (max, sum) in fp32
size_t attn_prefill_ws_bytes(int head_dim) { return (size_t)FP_WG * 128 * (head_dim + 2) * sizeof(float); }

template <int HD, int G, bool F8, int KG>
static void prefill_go(AttnPrefillArgs a, hipStream_t st) {
  constexpr int BQ = 128 / G;
  a.ns = prefill_runs(a, BQ, KG);
  const int ny = a.n_kv_heads;
  a.lm = ny % 8 == 0 ? 0 : (ny == 4 ? 1 : (ny == 2 ? 2 : 3));  // (neither a divisor nor a multiple of 8: all XCDs share all heads)
  a.hx = ny % 8 == 0 ? ny / 8 : (8 % ny == 0 ? 1 : ny);
  const int m = 1 << a.lm;
  const int W = a.hx * ((a.T + BQ - 1) / BQ) * a.ns;
  const dim3 grid(8 * ((W + m - 1) / m));  // (the kernel's lists, one place in turn on each XCD)
  const size_t lds = (size_t)2 * KG * FP_KT * ((HD + 8) + (HD + 32)) * sizeof(bf16_t);  // two buffers of KG K|V tiles
  hipLaunchKernelGGL((attn_prefill_kernel<HD, G, F8, KG>), grid, dim3(256 * KG), lds, st, a);
  if (a.ns > 1)
    hipLaunchKernelGGL((attn_prefill_combine<HD>), dim3((a.T * a.n_heads + 3) / 4), dim3(256), 0, st, a, BQ,
                       F8 ? a.kv_scale_v : 1.f);
}

template <int HD, int G, bool F8>
static void prefill_form(const AttnPrefillArgs& a, hipStream_t st) {
  if (prefill_groups(a, 128 / G) == 2) prefill_go<HD, G, F8, 2>(a, st);
  else prefill_go<HD, G, F8, 1>(a, st);
}

template <int HD, bool F8>
static void prefill_hd(const AttnPrefillArgs& a, int G, hipStream_t st) {
  switch (G) {
    case 1: prefill_form<HD, 1, F8>(a, st); break;
    case 2: prefill_form<HD, 2, F8>(a, st); break;
    case 4: prefill_form<HD, 4, F8>(a, st); break;
    case 8: prefill_form<HD, 8, F8>(a, st); break;
    default: throw std::runtime_error("attn_prefill: unsupported GQA group size");
  }
}

void launch_attn_prefill(const AttnPrefillArgs& a, hipStream_t st) {
  if (!attn_prefill_supports(a.n_heads, a.n_kv_heads, a.head_dim))
    throw std::runtime_error("attn_prefill: unsupported head configuration");
  if (a.T <= 0) return;
  if (a.start + a.T > a.max_ctx) throw std::runtime_error("attn_prefill: context overflow");
  const int G = a.n_heads / a.n_kv_heads;
  if (a.head_dim == 128) {
    if (a.kv_fp8) prefill_hd<128, true>(a, G, st);
    else prefill_hd<128, false>(a, G, st);
  } else {
    if (a.kv_fp8) prefill_hd<64, true>(a, G, st);
    else prefill_hd<64, false>(a, G, st);
  }
}

}  // namespace aios
