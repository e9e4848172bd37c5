// Batched-decode GEMM, K over the waves (M = 2..32 rows of bf16 activations):
//   C[M][N] = X[M][K] x W[N][K]^T,  W in the repacked Q4_K / Q6_K planes or bf16 (qweight.h).
//
// A workgroup's eight waves share K between them: a wave keeps its slice of X as MFMA operands in registers (256 k of
// 16 rows = 32 VGPRs), and the workgroup walks 16-row tiles of W, every wave its own k of them.  Weights go from
// memory to the wave's registers and are decoded there; the eight partial sums of a tile meet in LDS, and the waves take
// turns at the output stage, so the stream has one barrier a tile and no ring, slot or X traffic in it.  The tiles are
// 16 rows, so 256 CUs share any N evenly, and most shapes need no K split over workgroups, whose slabs and ticket cost
// ~4 us of a launch.
//
// The weights of a stage are asked for in whole lines, eight lanes to a row's 128 bytes, and take the order of the matrix instruction's
// lanes through the wave's own LDS.  Asked for in that order (16 lanes, 16 rows) each lane is an address of its own to the address unit,
// and a launch was as long as those take.  us, so -> in whole lines, 16 rows (3 rows alike, 30 rows 0.9 to 2.9 less):
//   bf16 8704 x 2048 12.1 -> 9.9   2048 x 8704 13.1 -> 11.8   8192 x 2048 10.3 -> 8.8   2048 x 2048 6.2 -> 5.3   11264 x 2048 12.8 -> 10.9
//   Q4_K 4096 x 14336 15.0 -> 13.9   4096 x 4096 6.6 -> 6.3   6144 x 4096 8.7 -> 8.0   28672 x 4096 19.8 -> 19.2   Q6_K 32000 x 4096 30.0 -> 28.5
// Bounds: a launch of few tiles, ~4 us of launch, first loads and output; bf16, the stream (11264 x 2048 4.2 TB/s of the launch); a long quantised
// one, the decode beside the stream (28672 x 4096: the vector unit is issued to for 58 % of a launch, the waves wait for 36 %).
// Measured in us, the LDS ring GEMM (gemm_ring.hip) -> this before it asked for whole lines, 16 / 32 rows, weights from memory:
//   4096 x 4096 Q4_K 10.1 -> 6.3 / 12.1 -> 8.2     28672 x 4096 Q4_K 20.6 -> 18.0 / 26.1 -> 20.8
//   6144 x 4096 Q4_K 11.4 -> 8.5 / 13.2 -> 10.7    4096 x 14336 Q4_K 15.5 -> 14.6 / 18.4 -> 17.1
//   2048 x 2048 Q4_K 8.0 -> 4.5 / 10.0 -> 5.5      2048 x 5632 Q4_K 10.1 -> 7.5 / 12.6 -> 9.4
//   2048 x 2048 bf16 10.4 -> 5.9 / 12.4 -> 7.0     11264 x 2048 bf16 13.4 -> 12.6 / 15.1 -> 14.0
// Not better: X streamed with the weights instead of kept (4096 x 14336 in one slice 19.0), two tiles of weights in
// flight (gate/up 20.1: longer code, and the decode is the bound), 16 waves (22), weights requested before X (O 7.4), by LDS-DMA into a ring of
// the wave's own (20.3), all of a tile's next requests before its decode (21.3: the waves stand before the address unit), the records of
// scales in whole lines too (the same).
#include "gemm_pf.h"
#include "skinny_epi.h"

namespace aios {

constexpr int WK_W = 8;     // waves
constexpr int WK_SMAX = 8;  // K slices at most (the split-K slabs are sized for 8: gemm_skinny_ws_bytes)

// How a launch is dealt out; the divisions are the host's (a 64-bit one in the kernel is ~130 dependent instructions
// before the first load).  Groups [0, g0) of the G share the tiles below nt0 (QT0), the others the rest (QT1: the packed
// QKV's Q6_K V): q0 / q1 tiles each, one more for the first r0 / r1.  K: S slices of ku units, one more for the first kr.
struct WkPlan {
  int S, G, g0, nt0, q0, r0, q1, r1, ku, kr;
  int n_last;      // QT1 tiles: all of them in the last segment, from this column
  QWeight w_last;
};

// one stage: 256 k of a tile's 16 rows.  a: as loaded, row 8i + lane / 8 of 16 B; turned (turn_w), lane (row rr, quarter q) holds the
// chunks 2q and 2q + 1 (k 64 q .. + 63), bf16: the MFMA operands as they are
template <int QT>
struct WkRaw {
  gu32x4 a[2], b;
};
template <>
struct WkRaw<QT_Q6_K> {
  gu32x4 a[2], h;
  uint32_t sc, d;
};
template <>
struct WkRaw<QT_BF16> {
  gu32x4 a[8];
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t wk_rsrc(const void* p, uint32_t n) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)n, 0x00020000);
}

// X unit swizzle (16-B units of a 512-B row): 16 rows' reads of one unit fall on distinct banks
__device__ __forceinline__ int wk_xh(int m) { return (m ^ (m << 1)) & 15; }
// ... for 128-B rows of weights (two rows to the banks)
__device__ __forceinline__ int wk_wh(int r) { return (r & 6) | (r >> 3); }

// LAST: the tiles lie in the last segment (p.w_last)
template <int QT, int NS, int MT, int EPI, bool LAST>
__device__ __forceinline__ void wk_body(const GemmQArgs& a, const WkPlan& p, int rg, int sp, int t0, int t1, uint8_t* smem,
                                        float* inv_s, int& last_flag) {
  constexpr bool BF = QT == QT_BF16, Q6 = QT == QT_Q6_K;
  constexpr int UK = BF ? 64 : 256;  // k of a unit (of K's split); a stage is 256
  using Ahead = SkAhead<EPI, BF>;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rr = lane & 15, q = lane >> 4;
  const int S = p.S, ntile = a.N >> 4;
  const int s0 = sp * p.ku + min(sp, p.kr), n = p.ku + (sp < p.kr ? 1 : 0);
  const int u0 = s0 + n * wave / WK_W, u1 = s0 + n * (wave + 1) / WK_W;  // this wave's units of UK k
  const bool nrm = a.nrm_in != nullptr;
  NrmRows<16 * MT, WK_W> nr;
  if (nrm) nr.load(a, wave, lane);
  uint8_t* own = smem + wave * 8192;

  // ---- X, a stage: rows of 512 B, coalesced; past M or the wave's k: zeros (out of the buffer)
  gu32x4 x[NS][MT][8];
  const auto rx = wk_rsrc(a.A, (uint32_t)(((size_t)(a.M - 1) * a.lda + a.K) * 2));
  auto load_x = [&](gu32x4 (&xs)[MT][8], int s) __attribute__((always_inline)) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int m = 16 * mt + 2 * j + (lane >> 5), k = u0 * UK + 256 * s + 8 * (lane & 31);
        xs[mt][j] = __builtin_amdgcn_raw_buffer_load_b128(
            rx, m < a.M && k < u1 * UK ? (uint32_t)(m * a.lda + k) * 2 : 0xfffffff0u, 0, 0);
      }
  };
  // into operand order through the wave's own 8 KB of LDS (a wave's LDS operations are in order: no barrier)
  auto turn_x = [&](gu32x4 (&xs)[MT][8]) __attribute__((always_inline)) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int m = 2 * j + (lane >> 5);
        *(gu32x4*)(own + m * 512 + 16 * ((lane & 31) ^ wk_xh(m))) = xs[mt][j];
      }
#pragma unroll
      for (int f = 0; f < 8; ++f) {
        // bf16: fragment f is k 32 f ..; else f = 4 u + 2 run + h: chunk 2q + u, weights 8h.. of its run
        const int unit = BF ? 4 * f + q : 8 * q + 2 * (f >> 2) + 4 * ((f >> 1) & 1) + (f & 1);
        xs[mt][f] = *(const gu32x4*)(own + rr * 512 + 16 * (unit ^ wk_xh(rr)));
      }
    }
  };
  // ---- weights: stage s of tile t (past the last tile or the wave's units: zeros, no memory access)
  const uint32_t nbk = a.K >> 8;
  auto load = [&](WkRaw<QT>& w, int s, int t) __attribute__((always_inline)) {
    const bool live = t < t1;
    const int n0 = min(t, t1 - 1) * 16;
    int sg = 0;
    if (!LAST && a.nseg > 1 && n0 >= a.seg_n0[1]) sg = 1;
    if (!LAST && a.nseg > 2 && n0 >= a.seg_n0[2]) sg = 2;
    const size_t row0 = n0 - (LAST ? p.n_last : sg == 0 ? a.seg_n0[0] : (sg == 1 ? a.seg_n0[1] : a.seg_n0[2]));
    auto plane = [&](auto get) __attribute__((always_inline)) {
      if constexpr (LAST) return get(p.w_last);
      else return sg == 0 ? get(a.seg[0]) : (sg == 1 ? get(a.seg[1]) : get(a.seg[2]));
    };
    const uint8_t* p0 = plane([](const QWeight& v) { return v.p0; });
    if constexpr (BF) {
      const uint32_t rb = (uint32_t)a.K * 2;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int uu = u0 + 4 * s + u;
        const auto r = wk_rsrc(p0 + row0 * rb, live && uu < u1 ? 16 * rb : 0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          w.a[2 * u + i] = __builtin_amdgcn_raw_buffer_load_b128(r, (8 * i + (lane >> 3)) * rb + 16 * (lane & 7), uu * 128, 2);
      }
    } else {
      const int uu = u0 + s;
      const bool on = live && uu < u1;
      const auto rc = wk_rsrc(p0 + row0 * nbk * 128, on ? 16 * nbk * 128 : 0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        w.a[i] = __builtin_amdgcn_raw_buffer_load_b128(rc, (8 * i + (lane >> 3)) * nbk * 128 + 16 * (lane & 7), uu * 128, 2);
      if constexpr (Q6) {
        const auto rh = wk_rsrc(plane([](const QWeight& v) { return v.p1; }) + row0 * nbk * 64, on ? 16 * nbk * 64 : 0);
        const auto rs = wk_rsrc(plane([](const QWeight& v) { return v.p2; }) + row0 * nbk * 16, on ? 16 * nbk * 16 : 0);
        const auto rd = wk_rsrc(plane([](const QWeight& v) { return v.p3; }) + row0 * nbk * 2, on ? 16 * nbk * 2 : 0);
        w.h = __builtin_amdgcn_raw_buffer_load_b128(rh, rr * nbk * 64 + 16 * q, uu * 64, 2);
        w.sc = __builtin_amdgcn_raw_buffer_load_b32(rs, rr * nbk * 16 + 4 * q, uu * 16, 0);
        w.d = __builtin_amdgcn_raw_buffer_load_b16(rd, rr * nbk * 2, uu * 2, 0);
      } else {
        const auto rm = wk_rsrc(plane([](const QWeight& v) { return v.p1; }) + row0 * nbk * 16, on ? 16 * nbk * 16 : 0);
        w.b = __builtin_amdgcn_raw_buffer_load_b128(rm, rr * nbk * 16, uu * 16, 0);
      }
    }
  };
  // a stage from whole lines to the lanes' own rows, through the wave's own LDS (behind the partial sums)
  uint8_t* const codes = own + 4096;
  auto turn_w = [&](WkRaw<QT>& w) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < (BF ? 4 : 1); ++u) {
      uint8_t* const to = codes + 2048 * (u & 1);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 8 * i + (lane >> 3);
        *(gu32x4*)(to + r * 128 + 16 * ((lane & 7) ^ wk_wh(r))) = w.a[2 * u + i];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) w.a[2 * u + i] = *(const gu32x4*)(to + rr * 128 + 16 * ((BF ? 4 * i + q : 2 * q + i) ^ wk_wh(rr)));
    }
  };
  gf32x4 acc[MT][2];
  auto compute = [&](const WkRaw<QT>& w, const gu32x4 (&xs)[MT][8]) __attribute__((always_inline)) {
    float sc[2], of[2];
    if constexpr (Q6) {
      sc[0] = h2f((uint16_t)w.d);  // (times the chunk's int8 scales below)
    } else if constexpr (!BF) {
      const float d = h2f((uint16_t)(w.b[0] & 0xffff)), dmin = h2f((uint16_t)(w.b[0] >> 16));
      const uint32_t fl = kq_field(w.b[1], w.b[2], w.b[3], q);
      sc[0] = d * (float)(fl & 63);
      sc[1] = d * (float)((fl >> 6) & 63);
      of[0] = dmin * (float)((fl >> 12) & 63);
      of[1] = dmin * (float)((fl >> 18) & 63);
    }
#pragma unroll
    for (int f = 0; f < 8; ++f) {
      gbf16x8 wf;
      if constexpr (BF) {
        wf = __builtin_bit_cast(gbf16x8, w.a[f]);
      } else {
        const int u = f >> 2, run = (f >> 1) & 1, j = 2 * (f & 1);
        const uint32_t c0 = w.a[u][j], c1 = w.a[u][j + 1];
        if constexpr (Q6) {
          const uint32_t hv = w.h[2 * u + run];
          const uint32_t l0 = (run ? c0 >> 4 : c0) & 0x0f0f0f0fu, l1 = (run ? c1 >> 4 : c1) & 0x0f0f0f0fu;
          const float ds = sc[0] * (float)(int8_t)(w.sc >> (16 * u + 8 * run));
          wf = pf_dq8<0x3f>(l0 | (((hv >> (2 * j)) & 0x03030303u) << 4), l1 | (((hv >> (2 * j + 2)) & 0x03030303u) << 4),
                            ds, 32.f * ds);
        } else {
          wf = run ? pf_dq8<0xf, 4>(c0, c1, sc[1], of[1]) : pf_dq8<0xf, 0>(c0, c1, sc[0], of[0]);
        }
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt][f & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, __builtin_bit_cast(gbf16x8, xs[mt][f]), acc[mt][f & 1], 0, 0, 0);
    }
  };
  // one lane's outputs of tile t, rows 16 mt ..
  auto finish = [&](int t, int mt, gf32x4 v, const Ahead& res) __attribute__((always_inline)) {
    float ss = res.finish(a, nrm ? inv_s : nullptr, 16 * mt + rr, 16 * t + 4 * q, v);
    if constexpr (EPI == GEPI_ACCUM_NORM) {
      ss = lane_xor32(lane_xor16(ss, LaneAdd{}), LaneAdd{});
      if (q == 0 && 16 * mt + rr < a.M) a.nrm_part[(size_t)(16 * mt + rr) * a.nrm_parts + t] = ss;
    }
  };
  // the waves' parts of tile t (double-buffered in each wave's own LDS), one barrier, and wave (t MT + mt) mod 8 adds them
  // up; it has read them before it reaches the next barrier, which the next write to them follows
  auto meet = [&](int t, const Ahead (&res)[MT]) __attribute__((always_inline)) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) *(gf32x4*)(own + ((t & 1) * MT + mt) * 1024 + 16 * lane) = acc[mt][0] + acc[mt][1];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (wave != ((t * MT + mt) & (WK_W - 1))) continue;
      gf32x4 v = gf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < WK_W; ++i) v += *(const gf32x4*)(smem + i * 8192 + ((t & 1) * MT + mt) * 1024 + 16 * lane);
      if (S == 1) finish(t, mt, v, res[mt]);
      else
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(gu32x4, v), wk_rsrc(a.ws, 0x7fffffff),
                                               ((sp * ntile + t) * MT + mt) * 1024 + 16 * lane, 0, 16 /* sc1 */);
    }
  };

  // (the scheduler may not sink the requests to where they are waited for)
  WkRaw<QT> w[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) load_x(x[s], s);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < NS; ++s) load(w[s], s, t0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < NS; ++s) turn_x(x[s]);
  if (nrm) nr.done(a, wave, lane, inv_s);  // (read after the first tile's barrier)
  // what the outputs need besides their sums is requested before the tile's products (by every wave: which of them adds the tile up
  // is not worth a branch here).  Behind the sums it was one or two trips to memory at the end of a launch.
  // bf16 weights, 8 steps of TinyLlama with 12 rows 8.57 -> 8.43 ms, with 6 8.03 -> 7.90 (with 3, and Seledra's 16, no more than the runs differ,
  // 1 to 2 %); beside a quantised format's decode nothing that shows (8 rows of TinyLlama and Mistral within 1 %): there the residual only
  int pos[MT], slot[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    pos[mt] = slot[mt] = 0;
    if constexpr (EPI == GEPI_QKV && BF) {
      const int m = min(16 * mt + rr, a.M - 1);
      pos[mt] = a.pos[m];
      if (a.slot) slot[mt] = a.slot[m];
    }
  }
  auto ahead = [&](Ahead& res, int t, int mt) __attribute__((always_inline)) {
    res.load(a, min(16 * mt + rr, a.M - 1), 16 * t + 4 * q, pos[mt], slot[mt]);
  };
  for (int t = t0; t < t1; ++t) {
    Ahead res[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      acc[mt][0] = acc[mt][1] = gf32x4{0.f, 0.f, 0.f, 0.f};
      ahead(res[mt], t, mt);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (s + 1 < NS || u0 + s * (256 / UK) < u1) {
        turn_w(w[s]);
        compute(w[s], x[s]);
      }
      load(w[s], s, t + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    meet(t, res);
  }
  if (S == 1) return;
  // ---- K split over workgroups: slabs written through, the range's last arriver adds them up in slice order
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every storing wave drains its slab stores
  __syncthreads();
  if (threadIdx.x == 0) {
    const int k = __hip_atomic_fetch_add(a.cnt + rg, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int last = k == S - 1;
    if (last) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __hip_atomic_store(a.cnt + rg, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-arm
    }
    last_flag = last;
  }
  __syncthreads();
  if (!last_flag) return;
  for (int i = wave; i < (t1 - t0) * MT; i += WK_W) {
    const int t = t0 + i / MT, mt = i % MT;
    Ahead res;
    ahead(res, t, MT == 1 ? 0 : mt);
    gf32x4 v = gf32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < S; k0 += 4) {  // four slabs' loads in flight (past the last: read again, not added)
      gf32x4 part[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        part[k] = *(const gf32x4*)(a.ws + ((size_t)(min(k0 + k, S - 1) * ntile + t) * MT + mt) * 256 + 4 * lane);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k0 + k < S) v += part[k];
    }
    finish(t, mt, v, res);
  }
}

template <int QT0, int QT1, int NS, int MT, int EPI>
__global__ void __launch_bounds__(WK_W * 64) __attribute__((amdgpu_waves_per_eu(WK_W / 4))) gemm_wk_kernel(
    GemmQArgs a, WkPlan p) {
  kernarg_warm<sizeof(GemmQArgs) + sizeof(WkPlan)>();
  __shared__ __attribute__((aligned(16))) uint8_t smem[WK_W * 8192];
  __shared__ float inv_s[16 * MT];
  __shared__ int last_flag;
  int rg = blockIdx.x, sp = 0;
  if (p.S > 1) {  // a group's slices on one XCD
    const uint32_t L = xcd_remap(blockIdx.x, p.G * p.S);
    rg = L / (uint32_t)p.S;
    sp = L - rg * p.S;
  }
  if constexpr (QT0 != QT1) {
    if (rg >= p.g0) {
      const int g = rg - p.g0, t0 = p.nt0 + g * p.q1 + min(g, p.r1);
      wk_body<QT1, NS, MT, EPI, true>(a, p, rg, sp, t0, t0 + p.q1 + (g < p.r1 ? 1 : 0), smem, inv_s, last_flag);
      return;
    }
  }
  const int t0 = rg * p.q0 + min(rg, p.r0);
  wk_body<QT0, NS, MT, EPI, false>(a, p, rg, sp, t0, t0 + p.q0 + (rg < p.r0 ? 1 : 0), smem, inv_s, last_flag);
}

// what a launch is given: K slices, stages of the longest wave (NS), 16-row groups (MT), workgroups that share the tiles
struct WkRoute {
  int S, ns, mt, G;
};

bool gemm_wk_on() {
  const char* e = std::getenv("AIOS_GEMM_WK");  // (read per call: tests compare both)
  return !e || std::atoi(e);
}

// AIOS_GEMM_WK: 1 (default) = this serves M = 2..32 of Q4_K / Q6_K / bf16 and the packed Q4_K | Q6_K QKV; 0 = the ring
// (quantised) and skinny GEMMs
static bool wk_route(const GemmQArgs& a, WkRoute& r) {
  if (!gemm_wk_on() || a.M < 2 || a.M > 32 || a.N % 16 || a.lda % 8) return false;
  const int qt0 = a.seg[0].qtype, qt1 = a.seg[a.nseg - 1].qtype;
  const bool bf = qt0 == QT_BF16, mixed = qt0 == QT_Q4_K && qt1 == QT_Q6_K;
#ifdef AIOS_BF16_ONLY
  if (!bf) return false;
#endif
  if (!mixed && (qt0 != qt1 || (!bf && qt0 != QT_Q4_K && qt0 != QT_Q6_K))) return false;
  if (mixed && a.epi != GEPI_QKV && a.epi != GEPI_STORE) return false;
  if ((a.epi == GEPI_STORE16 || a.epi == GEPI_STORE_GLU) && !bf) return false;
  if (a.K % (bf ? 64 : 256) || ((uintptr_t)a.A & 3)) return false;
  if (((size_t)(a.M - 1) * a.lda + a.K) * 2 >= 0xfffffff0u || (size_t)a.K * 32 >= 0x7fffffffu) return false;
  if (a.nrm_in && (a.nrm_parts <= 0 || a.nrm_parts % 4)) return false;
  if (a.epi == GEPI_SWIGLU_BF16 && a.ldc % 2) return false;
  if (a.epi == GEPI_QKV && bf && a.head_dim % 4) return false;  // (SkAhead: a lane's four columns in one head; quantised formats go by pairs)
  if (a.epi == GEPI_STORE_GLU && (a.glu_n0 % 4 || a.ldc16 % 2)) return false;
  if (a.epi != GEPI_SWIGLU_BF16 && a.ldc % 4) return false;
  if (a.epi == GEPI_ACCUM_NORM && (!a.nrm_g || !a.nrm_out16 || !a.nrm_part || a.N / 16 != a.nrm_parts)) return false;
  for (int s = 0; s < a.nseg; ++s)
    if (a.seg_n0[s] % 16 || a.seg[s].rows % 16 || (s + 1 < a.nseg && a.seg[s].qtype != qt0)) return false;
  // K's slices: as few as leave a wave at most NSM stages.  Two (X: 64 or 128 registers; a bf16 stage's weights take 32):
  // with four at 16 rows the longer prologue costs more than slabs save, 4096 x 14336 in two slices 16.3 us, in four 14.6,
  // 2048 x 5632 in one 8.7, in two 7.5; but a second slice that the registers do not ask for loses, 4096 x 4096 6.3 -> 8.5.
  r.mt = a.M <= 16 ? 1 : 2;
  const int NSM = bf ? 2 / r.mt : 2, un = bf ? 64 : 256, nu = a.K / un, ups = 256 / un;
  auto stages = [&](int S) {  // of the longest wave
    const int n = (nu + S - 1) / S;
    return ((n + WK_W - 1) / WK_W + ups - 1) / ups;
  };
  r.S = std::max(1, std::min(a.ksplit, nu));
  while (stages(r.S) > NSM) ++r.S;
  if (r.S > WK_SMAX) return false;
  r.ns = stages(r.S);
  // Q6_K in three slices, K of 10240 at most, up to 16 rows: the ring's deeper stream where its 128-row tiles in eight slices cover three
  // quarters of the CUs.  us here / ring, 4 and 16 rows: 4096 x 9216 14.6 / 14.0, 14.8 / 15.0   4096 x 10240 15.1 / 14.8, 15.6 / 15.9
  //   6144 x 8448 17.1 / 17.0, 17.5 / 18.0   4096 x 8448 13.5 / 13.7, 13.5 / 14.5; but 4096 x 11008 15.0 / 16.0, 15.7 / 16.8
  //   4096 x 12288 15.8 / 16.7, 16.5 / 17.4   4096 x 14336 17.8 / 18.6, 18.3 / 19.2   8192 x 28672 50.5 / 54.9, 53.4 / 57.6
  const int cus = device_cu_count(), round = a.N / 128 * 8;
  if (qt0 == QT_Q6_K && r.S == 3 && nu <= 40 && r.mt == 1 && a.N % 128 == 0 && 4 * round >= 3 * cus) return false;
  // bf16 where a tile has little k for eight waves to share: the skinny GEMM.  us here / skinny, 16 rows: 128256 x 512 44 / 33, 32000 x 64 9.7 / 5.5;
  // but 32000 x 512 13.2 / 15.4, 128256 x 4096 170 / 224, 32 rows 188 / 233.  And where slabs cost (long K and a wide output; two 16-row groups
  // of one round of its tiles): it was ahead there before whole lines and is no longer, 4096 x 14336 24 / 27, 4096 x 8192, 32 rows 19 / 20, but
  // this line is where test_gemm_wk_leaves_some_bf16_to_skinny holds it
  if (bf && (a.N > 125L * a.K || (a.K > 12288 && a.N >= 4096) || (r.mt == 2 && r.S >= 4 && 4 * round >= 3 * cus && round <= cus))) return false;
  // (three segments' four planes and the cache's arguments: more scalars than there are)
  if (a.epi == GEPI_QKV && qt0 == QT_Q6_K && r.ns * r.mt == 4) return false;
  // One slice more where that deals the tiles out more evenly: G ranges of whole tiles leave CUs idle while the longer ranges end.  With a split
  // that there is anyway, from a fifth less for the longest range up, if a quarter of the ranges are longer ones; us before / so, 16 and 30 rows:
  // 2048 x 8704 (three slices of 85 ranges, 43 of them two tiles long) bf16 12.7 / 11.8 (30 rows: five slices already), Q6_K 11.1 / 10.2, 13.6 / 12.5,
  // Q4_K 9.2 / 8.8, 11.4 / 10.8; 2048 x 5632 bf16, 30 rows 10.6 / 9.9; but 4096 x 12288 (one of 85 ranges is longer) Q4_K 12.5 / 13.2, 14.9 / 15.9,
  // Q6_K 16.5 / 17.2; 5120 x 17408 Q4_K, 8 % less 18.4 / 18.8.
  // bf16, two slices instead of one where its tiles are for three eighths of the CUs at most and a wave has two stages: 1024 x 4096 7.2 / 6.5,
  // 1280 x 4096 7.3 / 6.8, 1536 x 4096 7.4 / 7.1, 1024 x 3072 6.7 / 6.3; but 2048 x 4096 7.5 / 7.8, 2048 x 2048, one stage, 5.3 / 6.6, Q4_K 2048 x 4096
  // 5.8 / 6.8.  Four instead of two, which leave a wave one stage of more tiles, up to 7168 k and where the longest range gets shorter: 2048 x 5632
  // 9.6 / 8.7, 2048 x 6912 10.2 / 9.4, 1536 x 5632 9.0 / 8.3, 4096 x 5632 12.9 / 12.4, 3072 x 8192 15.4 / 13.1; but 2048 x 8192 10.8 / 13.1.
  auto groups = [&](int S) { return std::min(a.N / 16, std::max(1, cus / S)); };
  auto longest = [&](int S) { return (long)((a.N / 16 + groups(S) - 1) / groups(S)) * ((nu + S - 1) / S); };
  auto room = [&](int S) { return a.ws && a.cnt && a.cnt_len >= groups(S) && a.ws_bytes >= (size_t)S * 16 * r.mt * a.N * 4; };
  auto shorter = [&](int S) { return 5 * longest(S) <= 4 * longest(r.S); };
  if (a.ksplit == 0 && r.S < WK_SMAX && r.S < nu && room(r.S + 1) &&
      (r.S > 1 ? shorter(r.S + 1) && 4 * (a.N / 16 % groups(r.S)) >= groups(r.S) : bf && r.ns == 2 && 8 * (a.N / 16) <= 3 * cus))
    ++r.S;
  else if (a.ksplit == 0 && bf && r.mt == 1 && r.S == 2 && room(4) && (a.K <= 7168 || shorter(4)))
    r.S = 4;
  r.ns = stages(r.S);
  r.G = groups(r.S);
  if (mixed && r.G < 2) return false;
  return r.S == 1 || room(r.S);
}

int gemm_wk_slices(const GemmQArgs& a) {
  WkRoute r;
  return wk_route(a, r) ? r.S : 0;
}
bool gemm_wk_serves(const GemmQArgs& a) { return gemm_wk_slices(a) > 0; }

template <int QT0, int QT1, int NS, int MT>
static void wk_launch(const GemmQArgs& a, const WkRoute& r, hipStream_t st) {
  const int nt = a.N / 16, S = r.S, G = r.G;
  const int nt0 = QT0 != QT1 ? a.seg_n0[a.nseg - 1] / 16 : nt;
  int g0 = G;
  if (QT0 != QT1) {  // groups in the share of the bytes (144 and 210 per 256 weights)
    g0 = std::max(1, std::min({G - 1, nt0, (int)((long)G * nt0 * 144 / ((long)nt0 * 144 + (long)(nt - nt0) * 210))}));
    if (G - g0 > nt - nt0) g0 = G - (nt - nt0);
  }
  const int nu = a.K / (QT0 == QT_BF16 ? 64 : 256), n1 = nt - nt0, g1 = std::max(G - g0, 1);
  const WkPlan p = {S, G, g0, nt0, nt0 / g0, nt0 % g0, n1 / g1, n1 % g1, nu / S, nu % S, a.seg_n0[a.nseg - 1], a.seg[a.nseg - 1]};
  const dim3 grid(G * S), block(WK_W * 64);
#define WK_GO(E) hipLaunchKernelGGL((gemm_wk_kernel<QT0, QT1, NS, MT, E>), grid, block, 0, st, a, p)
  if constexpr (QT0 != QT1) {
    if (a.epi == GEPI_QKV) WK_GO(GEPI_QKV);
    else WK_GO(GEPI_STORE);
  } else {
    switch (a.epi) {
      case GEPI_STORE: WK_GO(GEPI_STORE); break;
      case GEPI_QKV:
        if constexpr (QT0 != QT_Q6_K || NS * MT < 4) WK_GO(GEPI_QKV);  // (else: wk_route)
        break;
      case GEPI_ACCUM: WK_GO(GEPI_ACCUM); break;
      case GEPI_ACCUM_NORM: WK_GO(GEPI_ACCUM_NORM); break;
      case GEPI_STORE16:
        if constexpr (QT0 == QT_BF16) WK_GO(GEPI_STORE16);
        break;
      case GEPI_STORE_GLU:
        if constexpr (QT0 == QT_BF16) WK_GO(GEPI_STORE_GLU);
        break;
      default: WK_GO(GEPI_SWIGLU_BF16); break;
    }
  }
#undef WK_GO
}

bool launch_gemm_wk(const GemmQArgs& a, hipStream_t st) {
  WkRoute r;
  if (!wk_route(a, r)) return false;
  auto go = [&](auto q0, auto q1) {
    constexpr int A = decltype(q0)::value, B = decltype(q1)::value;
    if (r.mt == 1) {
      if (r.ns <= 1) wk_launch<A, B, 1, 1>(a, r, st);
      else wk_launch<A, B, 2, 1>(a, r, st);
    } else {
      if (A == QT_BF16 || r.ns <= 1) wk_launch<A, B, 1, 2>(a, r, st);
      else if constexpr (A != QT_BF16) wk_launch<A, B, 2, 2>(a, r, st);
    }
  };
#define WK_T(Q) std::integral_constant<int, Q>{}
  const int qt0 = a.seg[0].qtype, qt1 = a.seg[a.nseg - 1].qtype;
  if (qt0 == QT_BF16) go(WK_T(QT_BF16), WK_T(QT_BF16));
#ifndef AIOS_BF16_ONLY
  else if (qt0 == QT_Q6_K) go(WK_T(QT_Q6_K), WK_T(QT_Q6_K));
  else if (qt1 == QT_Q6_K) go(WK_T(QT_Q4_K), WK_T(QT_Q6_K));
  else go(WK_T(QT_Q4_K), WK_T(QT_Q4_K));
#endif
#undef WK_T
  return true;
}

}  // namespace aios
