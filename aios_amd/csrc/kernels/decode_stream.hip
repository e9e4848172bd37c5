// A decode step of one row, or of up to four against bf16 weights, as ONE resident launch: a workgroup per CU runs the layers' products and the attention, and the
// vectors between them go from workgroup to workgroup through memory.
//
// What bounds a step of one row is not its bytes: a chain of five launches a layer pays for each of them the launch, the
// operand's round trip, the first weights' and the drain, 3.5 to 4 us in which the weight stream stands (gemv_lds.h).  Here the
// stream does not stand: two waves of every workgroup copy the whole step's weights HBM -> LDS through one ring of 128 KB,
// four slots ahead of the fourteen that multiply, across products and layers, so what the next product needs lies in LDS while
// its operand is on its way.
//
// Exchanges.  A product's result is written as 64-bit words of (value, number of the exchange) with agent-scope stores, and
// read the same way until every word carries the number: one trip through memory, no fence, no flag behind the data, no
// barrier over the chip.  4096 values from and to 256 workgroups take 1.8 us (with a flag per workgroup written behind the
// data 6.3).  Numbers run on from launch to launch (DsCtl::epoch), so nothing is cleared.  A buffer is used once a layer;
// its words are overwritten only after an exchange that every reader of the old ones has contributed to (each workgroup owns
// rows of O, gate/up and down).
//
// Waiting.  Workgroups wait for each other, so all of them have to be on the chip.  The first thing a workgroup does is to
// sign in; the last one to do so opens the gate, and a workgroup that waited gate_ticks for it closes it for good: then all
// of them leave, also those that come later, and the launch behind (one workgroup that takes every part in turn and so waits
// for nobody) does the step.  Behind the open gate every wait is for a workgroup that runs; it is bounded all the same
// (wait_ticks), with the same way out.
//
// A step with its sampler, us, chain -> resident (MI355X).  Q4_K_M: TinyLlama 128 keys 596 -> 453, 1000 keys 674 -> 534; Mistral-7B 128 keys
// 1412 -> 1138, 2000 keys 1551 -> 1280, 3900 keys 1610 -> 1365; with the fp8 cache 2000 keys 1512 -> 1238, 16000 keys 1657 -> 1508; Qwen3-8B 128
// keys 1733 -> 1269.  TinyLlama bf16, 128 / 1000 keys: one row 722 -> 584 / 799 -> 648, two 794 -> 603 / 862 -> 665, three 822 -> 625 / 873 -> 689,
// four 822 -> 672 / 887 -> 733 (five and more stay with the GEMMs: a fifth row is a second matrix instruction for the same weights, and its operand
// leaves the ring three slots).
#include "decode_stream.h"

#include <algorithm>
#include <numeric>

#include "attn_decode.h"
#include "gemv_impl.h"

namespace aios {

namespace {

constexpr int DS_NG = 14, DS_NL = 2, DS_CT = DS_NG * 64, DS_THREADS = (DS_NG + DS_NL) * 64;
constexpr int DS_SLOT = 32768, DS_R = 4;
constexpr int DS_AW = 8;  // waves that attend
constexpr unsigned DS_LATE = 1 << 16;  // of DsCtl::done: a workgroup that gave up waiting

// bf16 weights, up to four rows: a slot is four groups of four rows by 512 columns, a KB a row; 8 waves take half a group each
constexpr int DS_BROWS = 4, DS_BSLOT = 16384, DS_BGROUPS = 4, DS_BPAD = 64;
constexpr int DS_BRING = 8;  // slots, at most (the requests of seven are 56 of a wave's 63)
template <bool BF>
constexpr int ds_red() { return BF ? 64 : 16; }  // floats of one buffer of squares

// a slot: chunks (32 weights) and their planes, each a run of its own (1 KB an LDS-DMA; the last plane of Q6_K 256 B)
template <int QT>
struct DsFmt;
template <>
struct DsFmt<QT_Q4_K> {
  static constexpr int CH = 1792, PAIRS = 1;  // a lane takes two chunks of a slot
  static constexpr int off[4] = {0, 28672, 0, 0};
  static constexpr int per_loader = 16;
};
template <>
struct DsFmt<QT_Q6_K> {
  static constexpr int CH = 896, PAIRS = 0;
  static constexpr int off[4] = {0, 14336, 21504, 23552};
  static constexpr int per_loader = 12;
};

// tables of the step through the scalar cache (uniform addresses, written before the launch): a vector load would be waited for
// behind every weight request of a loader
template <typename T>
using ds_const = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ T ds_table(const T* p, int i) {
  ds_const<uint32_t> q = (ds_const<uint32_t>)(uint64_t)(p + __builtin_amdgcn_readfirstlane(i));
  uint32_t w[sizeof(T) / 4];
#pragma unroll
  for (int k = 0; k < (int)(sizeof(T) / 4); ++k) w[k] = q[k];
  T v;
  __builtin_memcpy(&v, w, sizeof(T));
  return v;
}

enum { DS_QKV = 0, DS_O = 1, DS_GU = 2, DS_DOWN = 3 };

// a loader's half of slot s, every other KB of each plane: every slot of a format is as many requests, what lies behind the
// workgroup's rows reads as zeros without a memory access.  (No branch a request: with one each, a slot took 1 us to ask for.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ds_rsrc(const uint8_t* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)sgpr_ptr(p), (short)0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}
template <int S>
__device__ __forceinline__ void ds_request(__amdgpu_buffer_rsrc_t r, uint8_t* dst, int voff, int at) {
  // (non-temporal: each byte is read once a step)
  auto* to = (__attribute__((address_space(3))) void*)(dst + at);
  if constexpr (S == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 16, voff + at, 0, 0, 2);
  else __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 4, voff + at, 0, 0, 2);
}
template <int QT>
__device__ __forceinline__ void ds_copy(const DsCopy& j, int s, uint8_t* dst, int lw) {
  using F = DsFmt<QT>;
  const int lane = threadIdx.x & 63;
  const int c = s * F::CH, left = (j.job.chunks & ~DS_Q6) - c;
  dst += lw * 1024;
  const int v = lane * 16 + lw * 1024;
  const auto r0 = ds_rsrc(j.p[0] + (size_t)c * 16, left * 16);
  if constexpr (QT == QT_Q4_K) {
    const auto r1 = ds_rsrc(j.p[1] + (size_t)c * 2, left * 2);
    static_for<14>([&](auto i) { ds_request<16>(r0, dst, v, 2048 * i); });
    static_for<2>([&](auto i) { ds_request<16>(r1, dst + F::off[1], v, 2048 * i); });
  } else {
    const auto r1 = ds_rsrc(j.p[1] + (size_t)c * 8, left * 8);
    const auto r2 = ds_rsrc(j.p[2] + (size_t)c * 2, left * 2);
    const auto r3 = ds_rsrc(j.p[3] + (c >> 2), left >> 2);
    static_for<7>([&](auto i) { ds_request<16>(r0, dst, v, 2048 * i); });
    static_for<3>([&](auto i) { ds_request<16>(r1, dst + F::off[1], v, 2048 * i); });
    ds_request<16>(r2, dst + F::off[2], v, 0);
    if (lw == 0) ds_request<16>(r1, dst + F::off[1], v, 6144);
    else ds_request<4>(r3, dst - 1024 + F::off[3], lane * 4, 0);
  }
}

// bf16: a request is a KB of one row, lane l's sixteen bytes 4 x row places further on (mod 64), so that the lanes of the products below
// read their four rows from different banks.  base, kq: of the next group, from the workgroup's first row on, from its row's first column on
__device__ __forceinline__ void ds_copy16(const DsCopy& j, int& base, int& kq, uint8_t* dst, int lw) {
  const int lane = threadIdx.x & 63, rb = __builtin_amdgcn_readfirstlane((int)(uint64_t)j.p[1]);
  const auto r = ds_rsrc(j.p[0], j.job.nrows * rb);
  const int v0 = lw * rb + ((lane - 4 * lw) & 63) * 16, v1 = (lw + 2) * rb + ((lane - 4 * lw - 8) & 63) * 16;
  dst += lw * 1024;
  static_for<DS_BGROUPS>([&](auto g) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(dst + 4096 * g), 16, v0 + base, 0, 0, 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(dst + 4096 * g + 2048), 16, v1 + base, 0, 0, 2);
    base += 1024;
    const bool wrap = ++kq * 1024 == rb;
    base += wrap ? 3 * rb : 0;
    kq = wrap ? 0 : kq;
  });
}

// at most n of this wave's requests outstanding (n: a sum of slots' counts)
__device__ __forceinline__ void ds_wait(int n) {
  switch (n) {
    case 8: lg_vmcnt<8>(); break;
    case 12: lg_vmcnt<12>(); break;
    case 16: lg_vmcnt<16>(); break;
    case 24: lg_vmcnt<24>(); break;
    case 28: lg_vmcnt<28>(); break;
    case 32: lg_vmcnt<32>(); break;
    case 36: lg_vmcnt<36>(); break;
    case 40: lg_vmcnt<40>(); break;
    case 44: lg_vmcnt<44>(); break;
    case 48: lg_vmcnt<48>(); break;
    case 56: lg_vmcnt<56>(); break;
    default: lg_vmcnt<0>(); break;
  }
}

// the thread's number, opaque: what is worked out of it in one part of the step is not kept in registers through the others
__device__ __forceinline__ int ds_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// ---- exchanges ---------------------------------------------------------------------------------------------------------
// place of element e among a vector's words: the octets of a wave's lanes are a word apart, so that the loads that gather them are
// whole lines (K a multiple of 512); two bf16 to a word: of word w of an octet of four
__device__ __forceinline__ int ds_at(int e) { return (e & ~511) | ((e & 7) << 6) | ((e >> 3) & 63); }
__device__ __forceinline__ int ds_at16(int w) { return (w & ~255) | ((w & 3) << 6) | ((w >> 2) & 63); }

__device__ __forceinline__ void ds_put(uint64_t* p, uint32_t v, uint32_t no) {
  __hip_atomic_store(p, (uint64_t)no << 32 | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t ds_get(const uint64_t* p) {
  return __hip_atomic_load(const_cast<uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct DsClock {
  unsigned long long t0, limit;
  unsigned* late;  // (LDS: signed out with)
};
__device__ __forceinline__ bool ds_late(const DsClock& c) {
  if (__builtin_expect(__builtin_amdgcn_s_memrealtime() - c.t0 <= c.limit, 1)) return false;
  *c.late = 1;
  return true;
}

// N words of each lane, stride apart, until all carry the number (or the time is up).  What waits must not keep the memory from
// those it waits for (with all words asked for again and again an exchange beside a full stream took 5 us, and left it 4.5 TB/s):
// a lane asks memory for its first word only, and for the others, which come with it, once that is there and through the XCD's L2,
// where 32 workgroups share them.  An exchange has words of its own in each layer, so L2 holds none of an older number; one that
// it took in too early is asked for from memory.
template <int N, int U>
__device__ __forceinline__ void ds_poll(const uint64_t* const (&p)[U], int stride, uint32_t no, uint32_t (&v)[U][N], const DsClock& c) {
  uint64_t w[U][N];
  for (int it = c.limit ? 1 : 64;; ++it) {  // (the time is looked at every 64 rounds; with none to wait, in the first)
    bool ok = true;
#pragma unroll
    for (int u = 0; u < U; ++u) w[u][0] = ds_get(p[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) ok = ok && (uint32_t)(w[u][0] >> 32) == no;
    if (ok || (__builtin_expect((it & 63) == 0, 0) && ds_late(c))) break;
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int i = 1; i < N; ++i)
      w[u][i] = __hip_atomic_load(const_cast<uint64_t*>(p[u] + i * stride), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  bool ok = true;
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int i = 0; i < N; ++i) {
      v[u][i] = (uint32_t)w[u][i];
      ok = ok && (uint32_t)(w[u][i] >> 32) == no;
    }
  for (int it = c.limit ? 1 : 64; !ok; ++it) {
    ok = true;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < N; ++i) {
        w[u][i] = ds_get(p[u] + i * stride);
        v[u][i] = (uint32_t)w[u][i];
        ok = ok && (uint32_t)(w[u][i] >> 32) == no;
      }
    if (__builtin_expect((it & 63) == 0, 0) && ds_late(c)) break;
  }
}
__device__ __forceinline__ float ds_word(const uint64_t* p, uint32_t no, const DsClock& c) {
  const uint64_t* const q[1] = {p};
  uint32_t w[1][1];
  ds_poll<1, 1>(q, 0, no, w, c);
  return __uint_as_float(w[0][0]);
}

struct DsLds {
  uint8_t* ring;
  float *sums, *red;    // of the rows (ds_sum); squares, two buffers
  DsJob* jobs;          // of this workgroup (the launch with all workgroups)
  float* scale;         // of the caches, per layer
  float* gains;         // of this workgroup's rows, per norm behind a residual
  uint8_t* area;
};

// ---- a product's operand: gathered, multiplied by the norm's gains, quantised to int8 (gemv_q8.h) ------------------------
// one octet to int8 codes in chunk order and {dx, dx * sum of codes} per 16 (q8_octet of gemv_q8.h; the codes rounded by
// the addition of a number whose last place is 1, and their low bytes put together: a fifth of its instructions)
__device__ __forceinline__ void ds_octet(int o, float (&v)[8], int8_t* xq, float2* ms) {
  float am = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) am = fmaxf(am, fabsf(v[i]));
  am = fmaxf(am, dpp_xor1(am));
  am = fmaxf(am, dpp_xor2(am));
  const float dx = am * (1.f / 127.f), inv = am > 0.f ? 127.f / am : 0.f;
  uint32_t w[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    uint32_t t[4];  // 1.5 * 2^23 + the code
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = __float_as_uint(fmaf(v[4 * j + e], inv, 12582912.f));
    w[j] = __builtin_amdgcn_perm(t[1], t[0], 0x0c0c0400u) | __builtin_amdgcn_perm(t[3], t[2], 0x04000c0cu);
  }
  int sum = __builtin_amdgcn_sdot4((int)w[0], 0x01010101, __builtin_amdgcn_sdot4((int)w[1], 0x01010101, 0, false), false);
  sum += dpp_xor1_i(sum);  // the other octet of this 16-run
  const int quarter = o & 3;
  int c, s0;
  QFmt<QT_Q4_K>::run_pos(2 * (o >> 2) + (quarter >> 1), c, s0);
  const int piece = ((s0 >> 4) + (c >> 3)) & 1;
  *(uint2*)(xq + c * 32 + 16 * piece + 8 * (quarter & 1)) = make_uint2(w[0], w[1]);
  if (!(quarter & 1)) ms[c * 2 + (s0 >> 4)] = make_float2(dx, dx * (float)sum);
}

// IN_X: plain values x and gains, the sum of squares to red; IN_F32: the exchange's values (multiplied by the gains where a norm is in
// front); IN_BF16: pairs
enum { IN_X, IN_F32, IN_BF16 };
template <int IN, bool BF>
__device__ __forceinline__ void ds_stage(const float* x, const uint64_t* ex, uint32_t no, int rows, int K, const float* gain, uint8_t* xq,
                                         float2* ms, float* red, const DsClock& clk) {
  const int tid = ds_tid(), noct = K >> 3, all = BF ? rows * noct : noct;
  constexpr int NW = IN == IN_BF16 ? 4 : 8;
  constexpr int U = IN == IN_BF16 ? (BF ? 3 : 2) : 1;  // octets of a lane that are waited for together
  float ssq = 0.f;
  auto row_of = [&](int o) { return BF ? (o >= noct) + (o >= 2 * noct) + (o >= 3 * noct) : 0; };
  auto keep = [&](int o, float (&v)[8]) __attribute__((always_inline)) {
    if constexpr (BF) {
      const int b = row_of(o);
      *(uint4*)(xq + (size_t)b * (2 * K + DS_BPAD) + (o - b * noct) * 16) =
          make_uint4(pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3]), pk_bf16(v[4], v[5]), pk_bf16(v[6], v[7]));
    } else {
      ds_octet(o, v, (int8_t*)xq, ms);
    }
  };
  // (whole waves: K is a multiple of 512, a wave takes 512 elements of one row)
#pragma clang loop unroll(disable)
  for (int o = tid; o < all; o += U * DS_CT) {
    if constexpr (IN == IN_X) {
      const int b = row_of(o), oc = o - b * noct;
      const float4 f0 = *(const float4*)(x + 8 * o), f1 = *(const float4*)(x + 8 * o + 4);
      const float4 g0 = *(const float4*)(gain + 8 * oc), g1 = *(const float4*)(gain + 8 * oc + 4);
      const float f[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w}, g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
      float v[8];
      if constexpr (BF) ssq = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        ssq = fmaf(f[i], f[i], ssq);
        v[i] = f[i] * g[i];
      }
      if constexpr (BF) {
        const float t = wave_sum(ssq);
        if ((tid & 63) == 0) red[o >> 6] = t;
      }
      keep(o, v);
    } else {
      const uint64_t* p[U];
      uint32_t w[U][NW];
#pragma unroll
      for (int u = 0; u < U; ++u) {  // (rows of words follow each other as those of octets do)
        const int ou = o + u * DS_CT < all ? o + u * DS_CT : o;
        p[u] = ex + (size_t)(ou >> 6) * (NW * 64) + (ou & 63);
      }
      ds_poll<NW, U>(p, 64, no, w, clk);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (u && o + u * DS_CT >= all) continue;
        float v[8];
        if constexpr (IN == IN_BF16) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[2 * i] = __uint_as_float(w[u][i] << 16);
            v[2 * i + 1] = __uint_as_float(w[u][i] & 0xffff0000u);
          }
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i) v[i] = __uint_as_float(w[u][i]);
        }
        keep(o + u * DS_CT, v);
      }
    }
  }
  if constexpr (IN == IN_X && !BF) {
    const float t = wave_sum(ssq);
    if ((tid & 63) == 0) red[tid >> 6] = t;
  }
}

// the sums of squares of the residual's rows: a word of each workgroup, gathered by the waves in front of the last one (which writes this
// workgroup's results, and came to these 0.3 to 0.5 us after the others to the operand)
template <bool BF>
__device__ __forceinline__ void ds_squares(const DsArgs& a, const uint64_t* ex, uint32_t no, int rows, float* red, const DsClock& clk) {
  const int tid = ds_tid();
  if constexpr (BF) {  // (64 workgroups, of one row, to a wave)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = rows * (a.parts >> 6);
#pragma clang loop unroll(disable)
    for (int i = DS_NG - 2 - wave + (wave == DS_NG - 1 ? DS_NG : 0); i < n; i += DS_NG) {
      const float t = wave_sum(ds_word(ex + i * 64 + lane, no, clk));
      if (lane == 0) red[i] = t;
    }
  } else {
    float v = 0.f;
#pragma clang loop unroll(disable)
    for (int i = DS_CT - 65 - tid + (tid >= DS_CT - 64 ? DS_CT : 0); i < a.parts; i += DS_CT) v += ds_word(ex + i, no, clk);
    const float t = wave_sum(v);
    if ((tid & 63) == 0) red[tid >> 6] = t;
  }
}

// sum over the first n = 8, 16, 32 or 64 lanes of every n
__device__ __forceinline__ float ds_lanes(float v, int n) {
  v = lanes_sum<8>(v);
  if (n > 8) v += lane_dpp<0x140>(v);
  if (n > 16) v = lane_xor16(v, LaneAdd{});
  if (n > 32) v = lane_xor32(v, LaneAdd{});
  return v;
}

// A row's sum has a term from each group of lanes that holds a run of its columns, and a step done again gives the same logits whatever the order
// in which the waves come (added to a word of 32 bits in that order, logits of three bf16 rows were 3e-3 apart: an operand on the border between
// two bf16 values is enough).  Int8 products: each term has a word of LDS, [term][row], and who writes the result adds them up in their order; the
// words of one product are read before a wave can be past the barrier behind the next operand, so one buffer serves all.  Bf16 products, of more
// terms for up to four operand rows: sums of 64 bits, in which terms of 24 bits add up without rounding while their exponents lie within 2^24 of
// each other; two buffers, one of zeros.  us, added in any order / so / the other way: 8 steps of TinyLlama Q4_K_M 3735 / 3755 / 3855, of three rows
// of TinyLlama bf16 5395 / 5410 / 5620
// lanes that share a term, of a row of n chunks (or pairs); words of a row's sum
__host__ __device__ constexpr int ds_run(int n) { return (n & -n) < 64 ? n & -n : 64; }
__host__ __device__ constexpr int ds_terms(int K, bool q6) {
  const int n = q6 ? K / 32 : K / 64;
  return n / ds_run(n);
}
// a row's sum of n terms, `stride` apart
__device__ __forceinline__ float ds_sum(const float* p, int stride, int n) {
  float v = p[0];
  int t = 1;
#pragma clang loop unroll(disable)
  for (; t + 3 < n; t += 4) {
    const float a = p[t * stride], b = p[(t + 1) * stride], c = p[(t + 2) * stride], d = p[(t + 3) * stride];
    v = v + a + b + c + d;
  }
#pragma clang loop unroll(disable)
  for (; t < n; ++t) v += p[t * stride];
  return v;
}

// where a thread stands in a product: row and column of its (pair of) chunk(s), or group, in the first slot; what a slot advances them by.  (Worked
// out before the operand is waited for.)
struct DsAt {
  int row, c, drow, dc;
};
__device__ __forceinline__ DsAt ds_at_first(int first, int slot, int n) {
  DsAt p;
  p.row = first / n;
  p.c = first - p.row * n;
  p.drow = slot / n;
  p.dc = slot - p.drow * n;
  asm volatile("" : "+v"(p.row), "+v"(p.c), "+s"(p.drow), "+s"(p.dc));
  return p;
}

// one slot after the other against the staged operand; the terms of the rows' sums to acc.  A barrier behind each slot (or one)
template <int QT>
__device__ __forceinline__ void ds_dot(const DsJob& j, const DsAt& p, int nch, int run, int& slot, const DsLds& s, const int8_t* xq, const float2* ms,
                                       float* acc) {
  using F = DsFmt<QT>;
  const int tid = ds_tid(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // this lane's (pair of) chunk(s): place within the slot, and its row and column, which advance by a slot's chunks
  const int at = F::PAIRS ? 2 * tid : tid;
  int row = p.row, c = p.c;
  const int drow = p.drow, dc = p.dc;
  const int wfirst = F::PAIRS ? 128 * wave : 64 * wave;
  const int tsh = __builtin_ctz(run) + F::PAIRS;  // chunks of a term
  const bool same = dc == 0;  // the same columns in every slot: the operand stays in registers
  Q4PairX X;
  int xv[8];
  float4 m;
  auto load = [&]() __attribute__((always_inline)) {
    if constexpr (F::PAIRS) {
      q4p_load_x(xq, ms, c, X);
    } else {
      const int8_t* xc = xq + (size_t)c * 32;
      const int rot = (c >> 3) & 1;
      const uint4 p0 = *(const uint4*)(xc + 16 * rot), p1 = *(const uint4*)(xc + 16 * (rot ^ 1));
      xv[0] = p0.x; xv[1] = p0.y; xv[2] = p0.z; xv[3] = p0.w;
      xv[4] = p1.x; xv[5] = p1.y; xv[6] = p1.z; xv[7] = p1.w;
      m = *(const float4*)(ms + (size_t)c * 2);
    }
  };
  auto one = [&](const uint8_t* sl) __attribute__((always_inline)) {
    float v;
    if constexpr (F::PAIRS) {
      const uint4 a0 = *(const uint4*)(sl + F::off[0] + at * 16), a1 = *(const uint4*)(sl + F::off[0] + at * 16 + 16);
      const uint4 mt = *(const uint4*)(sl + F::off[1] + (at >> 3) * 16);
      v = q4p_dot(a0, a1, mt, (c >> 1) & 3, X);
    } else {
      RawChunk r;
      r.a = *(const uint4*)(sl + F::off[0] + at * 16);
      const uint2 h = *(const uint2*)(sl + F::off[1] + at * 8);
      r.b.x = h.x;
      r.b.y = h.y;
      r.c.x = *(const uint16_t*)(sl + F::off[2] + at * 2);
      r.d = *(const uint16_t*)(sl + F::off[3] + (at >> 3) * 2);
      float sc[2], of[2];
      q8_scales_bf<QT>(r, c, sc, of);
      int is[2];
      QDot<QT>::isums(r, c, xv, is);
      v = sc[0] * m.x * (float)is[0] - of[0] * m.y + sc[1] * m.z * (float)is[1] - of[1] * m.w;
    }
    v = ds_lanes(row < j.nrows ? v : 0.f, run);
    if ((lane & (run - 1)) == 0 && row < j.nrows) acc[(c >> tsh) * j.nrows + row] = v;
  };
  if (same && j.slots) load();
#pragma clang loop unroll(disable)
  for (int t = 0; t < j.slots; ++t) {
    if (t * F::CH + wfirst < j.chunks) {
      if (!same) load();
      one(s.ring + (size_t)((slot + t) % DS_R) * DS_SLOT);
    }
    row += drow;
    c += dc;
    if (c >= nch) {
      c -= nch;
      ++row;
    }
    if (t + 1 < j.slots) lg_barrier();
  }
  slot += j.slots;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lg_barrier();
}

// ... of bf16 weights against up to four rows: sixteen 4 x 4 products of four columns a matrix instruction (lane 4 b + i: weight row i or
// operand row i, columns 8 b ..), so each byte of weights is read from LDS once whatever the rows, beside as much of the operand
typedef short ds_s16x4 __attribute__((ext_vector_type(4)));
typedef float ds_f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void ds_dot16(const DsJob& j, const DsAt& p, int K, int rows, int ring, int& cur, const DsLds& s, const uint8_t* xb,
                                         double* acc) {
  const int tid = ds_tid(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 3, b = lane >> 2, g = wave >> 1, half = wave & 1;
  const int KQ = K >> 9;
  int rg = p.row, kq = p.c;
  const uint8_t* x = xb + (size_t)min(i, rows - 1) * (2 * K + DS_BPAD) + (half * 32 + b) * 16;
  const int w0 = g * 4096 + i * 1024 + ((half * 32 + b + 4 * i) & 63) * 16, w1 = g * 4096 + i * 1024 + ((half * 32 + 16 + b + 4 * i) & 63) * 16;
#pragma clang loop unroll(disable)
  for (int t = 0; t < j.slots; ++t) {
    if (wave < 2 * DS_BGROUPS && t * DS_BGROUPS + g < j.chunks) {
      const uint8_t* sl = s.ring + (size_t)cur * DS_BSLOT;
      const uint4 wa = *(const uint4*)(sl + w0), wb = *(const uint4*)(sl + w1);
      const uint4 xa = *(const uint4*)(x + kq * 1024), xc = *(const uint4*)(x + kq * 1024 + 256);
      auto mul = [](uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, ds_f32x4 c) {
        return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(ds_s16x4, make_uint2(a0, a1)), __builtin_bit_cast(ds_s16x4, make_uint2(b0, b1)), c, 0, 0, 0);
      };
      ds_f32x4 c0 = {0.f, 0.f, 0.f, 0.f}, c1 = c0;
      c0 = mul(wa.x, wa.y, xa.x, xa.y, c0);
      c1 = mul(wa.z, wa.w, xa.z, xa.w, c1);
      c0 = mul(wb.x, wb.y, xc.x, xc.y, c0);
      c1 = mul(wb.z, wb.w, xc.z, xc.w, c1);
      c0 += c1;
      // the sixteen blocks together: weight row r's sum goes to the lanes of row r of the wave
      const auto r0 = __builtin_amdgcn_permlane16_swap(__float_as_uint(c0[0]), __float_as_uint(c0[1]), false, false);
      const auto r1 = __builtin_amdgcn_permlane16_swap(__float_as_uint(c0[2]), __float_as_uint(c0[3]), false, false);
      const float p0 = __uint_as_float(r0[0]) + __uint_as_float(r0[1]), p1 = __uint_as_float(r1[0]) + __uint_as_float(r1[1]);
      const auto r2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(p0), __float_as_uint(p1), false, false);
      float v = __uint_as_float(r2[0]) + __uint_as_float(r2[1]);
      v += lane_dpp<0x124>(v);  // row_ror:4
      v += lane_dpp<0x128>(v);  // row_ror:8
      const int row = rg * 4 + (lane >> 4);
      if ((lane & 15) < rows && row < j.nrows) __hip_atomic_fetch_add(acc + row * DS_BROWS + i, (double)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    rg += p.drow;
    kq += p.dc;
    if (kq >= KQ) {
      kq -= KQ;
      ++rg;
    }
    if (++cur == ring) cur = 0;
    if (t + 1 < j.slots) lg_barrier();
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lg_barrier();
}

// keys of a workgroup's pass: a tile of four requests (of 1 KB, of fp8 512 B) a wave
template <int HD>
constexpr int ds_pass() { return DS_AW * 4 * (512 / HD); }

// ---- attention -----------------------------------------------------------------------------------------------------------
// G query heads of one KV head over the passes sp, sp + P, .. of its keys (attn_lanes of attn_decode.h, with the heads sharing what is
// read); the row's own key is taken from the exchange, as the cache will hold it.
// Four barriers.  LDS: queries in bf16, the own key and value as cached, the raw vectors and then the waves' results.
// Four heads: a lane has one head's scores (its number mod 4's) and not all four, an exp2 instead of four and 18 registers less.
// sum over a key's LPK lanes of four heads' terms, of head lane & 3
template <int LPK>
__device__ __forceinline__ float ds_quad_sum(const float (&d)[4]) {
  const bool b0 = threadIdx.x & 1, b1 = threadIdx.x & 2;
  const float r0 = (b0 ? d[1] : d[0]) + lane_dpp<0xB1>(b0 ? d[0] : d[1]);
  const float r1 = (b0 ? d[3] : d[2]) + lane_dpp<0xB1>(b0 ? d[2] : d[3]);
  float r = (b1 ? r1 : r0) + lane_dpp<0x4E>(b1 ? r0 : r1);
  if constexpr (LPK == 8) return r + lane_dpp<0x141>(lane_dpp<0x1B>(r));  // the other quad of eight, in its order
  r += lane_dpp<0x124>(r);
  return r + lane_dpp<0x128>(r);
}

template <int HD, int G, bool F8>
struct DsAttnLds {
  uint16_t q[G][HD];
  uint16_t own[2][HD];  // (fp8: bytes)
  float m[DS_AW][G], l[DS_AW][G];
  union {
    float vec[G + 2][HD];
    float o[DS_AW][G][HD];
  };
};

// a part that attends: row, unit of heads, run of its keys.  (One workgroup a unit: the heads of a KV head on one XCD; workgroups go
// round the eight in turn)
struct DsPlace {
  int b, unit, sp;
};
__device__ __forceinline__ DsPlace ds_place(int wg, int units, int rows, int P) {
  const int all = units * rows;
  const int u = P > 1 ? wg / P : ((all & 7) == 0 ? (wg & 7) * (all >> 3) + (wg >> 3) : wg);
  const int b = rows > 1 ? min(u / units, rows - 1) : 0;
  return {b, u - b * units, P > 1 ? wg - u * P : 0};
}

template <int HD, int G, bool F8, bool BF>
__device__ __forceinline__ void ds_attend(const DsArgs& a, int l, int wg, int P, int pos, uint32_t no, float2 cs, const DsLds& s,
                                          const DsClock& clk) {
  using S = DsAttnLds<HD, G, F8>;
  S& L = *(S*)s.area;
  constexpr int LPK = HD / 8, KPS = 64 / LPK;  // lanes of a key (8 elements each), keys of a request
  constexpr int STEPS = 4, KPW = STEPS * KPS;  // requests of a tile, its keys
  constexpr int PASS = ds_pass<HD>(), ES = F8 ? 1 : 2;
  using KVT = typename std::conditional<F8, uint2, uint4>::type;
  const int units = a.n_heads / G;
  const int tid = ds_tid(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rows = BF ? a.rows : 1;
  if (wg >= rows * units * P) {
    lg_barrier();
    lg_barrier();
    lg_barrier();
    lg_barrier();
    return;
  }
  const DsPlace at = ds_place(wg, units, rows, P);
  const int sp = at.sp, lb = l * rows + at.b;
  const int* blocks = a.blocks + (BF ? at.b * a.bt_stride : 0);
  const int h0 = at.unit * G, gq = a.n_heads / a.n_kv_heads, kvh = h0 / gq;
  const int ksub = lane / LPK, dsl = lane % LPK;
  uint8_t *kc = a.kc + (size_t)l * a.kv_layer, *vc = a.vc + (size_t)l * a.kv_layer;
  KVT kr[STEPS], vr[STEPS];
  auto first_key = [&](int pass) { return pass * PASS + wave * KPW; };
  // a tile is a buffer of its live keys' bytes: what lies behind them reads as zeros without a memory access
  const int voff = (ksub * HD + dsl * 8) * ES;
  auto request = [&](KVT (&r)[STEPS], const uint8_t* pool, int k0) __attribute__((always_inline)) {
    const int blk = ds_table(blocks, min(k0 / KV_BLOCK, a.max_ctx / KV_BLOCK - 1));
    const int live = __builtin_amdgcn_readfirstlane(min(max(pos - k0, 0), KPW));
    const auto rs = uniform_rsrc(pool + (((size_t)blk * a.n_kv_heads + kvh) * KV_BLOCK + (k0 % KV_BLOCK)) * HD * ES, live * HD * ES);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      if constexpr (F8) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, voff + i * KPS * HD * ES, 0, 0);
        r[i] = make_uint2(v[0], v[1]);
      } else {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, voff + i * KPS * HD * ES, 0, 0);
        r[i] = make_uint4(v[0], v[1], v[2], v[3]);
      }
    }
  };
  const int npass = pos / PASS + 1;
  if (wave < DS_AW) {
    request(kr, kc, first_key(sp));
    request(vr, vc, first_key(sp));
  }
  // ---- the heads' raw vectors
  if (tid < (G + 2) * HD) {
    const int v = tid / HD, i = tid - v * HD;
    const int row = v < G ? (h0 + v) * HD + i : (a.n_heads + (v == G ? kvh : a.n_kv_heads + kvh)) * HD + i;
    const float b = a.bias ? a.bias[(size_t)l * a.nqkv + row] : 0.f;
    L.vec[v][i] = ds_word(a.qkv + (size_t)lb * a.nqkv + row, no, clk) + b;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lg_barrier();
  if (wave < G + 2) {
    constexpr int HALF = HD / 2;
    const int p = lane & (HALF - 1);  // (heads of 64: lanes 32 up repeat the lower ones)
    const bool isq = wave < G, isv = wave == G + 1;
    const bool neox = a.rope_neox && !isv;
    const int ia = neox ? p : 2 * p, ib = neox ? p + HALF : 2 * p + 1;
    float v0 = L.vec[wave][ia], v1 = L.vec[wave][ib];
    if (!isv) {
      if (a.qk_gains) {
        const float* g = a.qk_gains + (size_t)(2 * l + !isq) * HD;
        const float inv = rsqrtf(lanes_sum<HALF>(v0 * v0 + v1 * v1) / (float)HD + a.eps);
        v0 *= inv * g[ia];
        v1 *= inv * g[ib];
      }
      const float o0 = v0 * cs.x - v1 * cs.y, o1 = v0 * cs.y + v1 * cs.x;
      v0 = o0;
      v1 = o1;
    }
    if (lane < HALF) {
      if (isq) {
        const float qs = a.scale * kLog2e * (F8 ? s.scale[2 * l] : 1.f);  // scores in the log2 domain
        const uint32_t u = pk_bf16(v0 * qs, v1 * qs);
        L.q[wave][ia] = (uint16_t)u;
        L.q[wave][ib] = (uint16_t)(u >> 16);
      } else {
        const float inv = F8 ? 1.f / (isv ? s.scale[2 * l + 1] : s.scale[2 * l]) : 1.f;
        kv_store_pair((bf16_t*)L.own[isv], ia, ib, v0, v1, F8, inv);
        if (sp == 0 && h0 % gq == 0) {  // one workgroup a KV head keeps it
          const size_t i0 = (((size_t)ds_table(blocks, pos / KV_BLOCK) * a.n_kv_heads + kvh) * KV_BLOCK + pos % KV_BLOCK) * HD;
          kv_store_pair((bf16_t*)(isv ? vc : kc), i0 + ia, i0 + ib, v0, v1, F8, inv);
        }
      }
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lg_barrier();
  if (wave < DS_AW) {
    uint4 q[G];  // (read for each tile: kept through the loop they spill)
    auto read_q = [&]() __attribute__((always_inline)) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int g = 0; g < G; ++g) q[g] = *(const uint4*)&L.q[g][dsl * 8];
    };
    constexpr bool QUAD = G == 4;
    constexpr int NS = QUAD ? 1 : G;  // heads whose scores a lane has
    float m[NS], sum[NS], o[G][8];
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      m[n] = kNeg;
      sum[n] = 0.f;
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int i = 0; i < 8; ++i) o[g][i] = 0.f;
    auto of_head = [&](const float (&v)[NS], auto g) __attribute__((always_inline)) {
      if constexpr (QUAD) return lane_dpp<0x55 * g.value>(v[0]);
      else return v[g.value];
    };
    auto score = [&](const KVT& r, float (&sc)[NS], bool live) __attribute__((always_inline)) {
      uint32_t kb[4];
      if constexpr (F8) {
        kb[0] = fp8x2_bf16x2<false>(r.x); kb[1] = fp8x2_bf16x2<true>(r.x);
        kb[2] = fp8x2_bf16x2<false>(r.y); kb[3] = fp8x2_bf16x2<true>(r.y);
      } else {
        kb[0] = r.x; kb[1] = r.y; kb[2] = r.z; kb[3] = r.w;
      }
      float d[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        d[g] = dot2_bf16(kb[0], q[g].x, 0.f);
        d[g] = dot2_bf16(kb[1], q[g].y, d[g]);
        d[g] = dot2_bf16(kb[2], q[g].z, d[g]);
        d[g] = dot2_bf16(kb[3], q[g].w, d[g]);
      }
      if constexpr (QUAD) {
        const float t = ds_quad_sum<LPK>(d);
        sc[0] = live ? t : kNeg;
      } else {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const float t = lanes_sum<LPK>(d[g]);
          sc[g] = live ? t : kNeg;
        }
      }
    };
    auto weigh = [&](const float (&mx)[NS]) __attribute__((always_inline)) {  // the heads' running max, at least mx
      bool more = false;
      float mn[NS];
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        mn[n] = fmaxf(m[n], mx[n]);
        more = more || mn[n] > m[n];
      }
      if (__builtin_amdgcn_ballot_w64(more)) {
        float alpha[NS];
#pragma unroll
        for (int n = 0; n < NS; ++n) {
          alpha[n] = fast_exp2(m[n] - mn[n]);
          sum[n] *= alpha[n];
          m[n] = mn[n];
        }
        static_for<G>([&](auto g) {
          const float f = of_head(alpha, g);
#pragma unroll
          for (int i = 0; i < 8; ++i) o[g][i] *= f;
        });
      }
    };
    auto add = [&](const KVT& r, const float (&p)[NS]) __attribute__((always_inline)) {
      float vf[8];
      if constexpr (F8) {
        const gf32x2 f0 = fp8x2_f32x2<false>(r.x), f1 = fp8x2_f32x2<true>(r.x), f2 = fp8x2_f32x2<false>(r.y), f3 = fp8x2_f32x2<true>(r.y);
        vf[0] = f0.x; vf[1] = f0.y; vf[2] = f1.x; vf[3] = f1.y;
        vf[4] = f2.x; vf[5] = f2.y; vf[6] = f3.x; vf[7] = f3.y;
      } else {
        const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vf[2 * e] = __uint_as_float(w[e] << 16);
          vf[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
        }
      }
      static_for<G>([&](auto g) {
        const float f = of_head(p, g);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[g][e] = fmaf(f, vf[e], o[g][e]);
      });
    };
    for (int pass = sp; pass < npass; pass += P) {
      const int k0 = first_key(pass), kn = first_key(pass + P);
      float sc[STEPS][NS], mx[NS];
      read_q();
#pragma unroll
      for (int i = 0; i < STEPS; ++i) {
        score(kr[i], sc[i], k0 + ksub + i * KPS < pos);
        __builtin_amdgcn_sched_barrier(0);  // (steps interleaved spill)
      }
      if (pass + P < npass) request(kr, kc, kn);
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        mx[n] = sc[0][n];
#pragma unroll
        for (int i = 1; i < STEPS; ++i) mx[n] = fmaxf(mx[n], sc[i][n]);
      }
      weigh(mx);
#pragma unroll
      for (int n = 0; n < NS; ++n)
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
          sc[i][n] = fast_exp2(sc[i][n] - m[n]);
          sum[n] += sc[i][n];
        }
#pragma unroll
      for (int i = 0; i < STEPS; ++i) {
        add(vr[i], sc[i]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (pass + P < npass) request(vr, vc, kn);
    }
    if (wave == 0 && sp == 0) {  // the row's own key, by the first key group
      float sc[NS];
      read_q();
      score(*(const KVT*)((const uint8_t*)L.own[0] + dsl * 8 * ES), sc, ksub == 0);
      weigh(sc);
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        sc[n] = fast_exp2(sc[n] - m[n]);
        sum[n] += sc[n];
        if (ksub) sc[n] = 0.f;
      }
      add(*(const KVT*)((const uint8_t*)L.own[1] + dsl * 8 * ES), sc);
    }
    // the key groups of a wave, then (below) the waves
    float w[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      const float M = keys_max<LPK>(m[n]);
      w[n] = fast_exp2(m[n] - M);
      const float S1 = keys_sum<LPK>(sum[n] * w[n]);
      if (lane < (QUAD ? 4 : 1)) {
        L.m[wave][QUAD ? lane : n] = M;
        L.l[wave][QUAD ? lane : n] = S1;
      }
    }
    static_for<G>([&](auto g) {
      const float f = of_head(w, g);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[g][e] = keys_sum<LPK>(o[g][e] * f);
      if (ksub == 0) {
        float4* dst = (float4*)&L.o[wave][g][dsl * 8];
        dst[0] = make_float4(o[g][0], o[g][1], o[g][2], o[g][3]);
        dst[1] = make_float4(o[g][4], o[g][5], o[g][6], o[g][7]);
      }
    });
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lg_barrier();
  if (tid < G * HD) {
    const int g = tid / HD, d = tid - g * HD;
    float W = L.m[0][g];
#pragma unroll
    for (int w = 1; w < DS_AW; ++w) W = fmaxf(W, L.m[w][g]);
    float S1 = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < DS_AW; ++w) {
      const float f = fast_exp2(L.m[w][g] - W);
      S1 += f * L.l[w][g];
      acc += f * L.o[w][g][d];
    }
    if (F8) acc *= s.scale[2 * l + 1];
    if (P == 1) {
      ds_put(a.attn + (size_t)lb * a.n_heads * HD + ds_at((h0 + g) * HD + d), __float_as_uint(acc / S1), no);
    } else {
      uint64_t* p = a.part + ((size_t)(at.b * a.n_heads + h0 + g) * DS_PMAX + sp) * (HD + 2);
      ds_put(p + d, __float_as_uint(acc), no);
      if (d < 2) ds_put(p + HD + d, __float_as_uint(d ? S1 : W), no);
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lg_barrier();  // (the area is the next operand's)
}

// the runs of a head's keys together: 16 elements of a head at a time.  Two barriers.
template <int HD, bool BF>
__device__ __forceinline__ void ds_combine(const DsArgs& a, int l, int unit, int P, uint32_t no, const DsLds& s, const DsClock& clk) {
  const int tid = ds_tid(), h = unit / (HD / 16), d0 = unit % (HD / 16) * 16;
  float* v = (float*)s.area;  // [P][18]
  const int rows = BF ? a.rows : 1;
  const bool on = unit < rows * a.n_heads * (HD / 16);
  if (on && tid < P * 18) {
    const int sp = tid / 18, j = tid - sp * 18;
    v[tid] = ds_word(a.part + ((size_t)h * DS_PMAX + sp) * (HD + 2) + (j < 16 ? d0 + j : HD + j - 16), no, clk);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lg_barrier();
  if (on && tid < 16) {
    float W = v[16];
    for (int p = 1; p < P; ++p) W = fmaxf(W, v[p * 18 + 16]);
    float S1 = 0.f, acc = 0.f;
    for (int p = 0; p < P; ++p) {
      const float f = fast_exp2(v[p * 18 + 16] - W);
      S1 += f * v[p * 18 + 17];
      acc += f * v[p * 18 + tid];
    }
    const int b = BF ? h / a.n_heads : 0;
    ds_put(a.attn + (size_t)(l * rows + b) * a.n_heads * HD + ds_at((h - b * a.n_heads) * HD + d0 + tid), __float_as_uint(acc / S1), no);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lg_barrier();
}

// ---- the step ---------------------------------------------------------------------------------------------------------------
// Keys below which a head has one workgroup, that needs no exchange of partial results (3.8 us a layer with the combination), and how many
// workgroups share the others.  A step, us, one workgroup / several: heads of 64 (TinyLlama bf16) 750 keys 625 / 689, 1250 660 / 687, 1500 688 / 692
// (four rows: 1250 767 / 801, 1500 798 / 811; Q4_K 1250 559 / 569, 1500 581 / 572); of 128 (Mistral-7B) 400 keys 1228 / 1241, 500 1231 / 1243, 600
// 1261 / 1248 (Qwen3-8B 500 1375 / 1385, 600 1412 / 1389)
template <int HD>
constexpr int ds_brief() { return HD == 64 ? 1280 : 512; }
template <int HD>
__device__ __forceinline__ int ds_runs(const DsArgs& a, int G, int pos) {
  if (pos < ds_brief<HD>()) return 1;
  return min(min(pos / ds_pass<HD>() + 1, a.parts / (a.rows * (a.n_heads / G))), DS_PMAX);
}

template <int HD, int G, bool F8, bool BF>
__global__ void __launch_bounds__(DS_THREADS) decode_stream_kernel(DsArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  if (a.alone && !a.ctl->failed) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int first = blockIdx.x, step = gridDim.x;  // (parts of this workgroup: one, or all of them in turn)
  DsLds s;
  s.ring = smem;
  s.area = smem + (BF ? a.ring * DS_BSLOT : DS_R * DS_SLOT);
  s.sums = (float*)(s.area + a.area_bytes);
  s.red = s.sums + (BF ? 2 : 1) * a.row_sums;
  constexpr int RED = ds_red<BF>();
  unsigned* gate = (unsigned*)(s.red + 2 * RED);
  s.scale = s.red + 2 * RED + 4;
  s.jobs = (DsJob*)(s.scale + (2 * a.n_layers + 3) / 4 * 4);
  s.gains = (float*)(s.jobs + 4 * a.n_layers + 1);
  constexpr int SH = BF ? 2 : 0;  // a product's row is four threads' that write it, of the operand's rows, or one's
  const int rows = BF ? a.rows : 1;
  auto pos_of = [&](int b) { return min(ds_table(a.pos, b), a.max_ctx - 1); };
  const int qd = a.n_heads * HD;
  int pos = pos_of(0);  // the farthest
  if constexpr (BF)
    for (int b = 1; b < rows; ++b) pos = max(pos, pos_of(b));
  const bool brief = pos < ds_brief<HD>();
  const int P = ds_runs<HD>(a, G, pos);
  const int nattend = rows * (brief ? a.n_heads : a.n_heads / G * P);  // parts that attend
  const int ncomb = (rows * a.n_heads * (HD / 16) + a.parts - 1) / a.parts;

  if (wave >= DS_NG) {
    // ---- loaders: the step's slots in order, as many ahead as the ring holds; they pass every barrier of the others
    const int lw = wave - DS_NG;
    // (Q4_K / Q6_K: their requests in front of fourteen waves of vector work, 0.5 to 1 % of a step; bf16, which has little, lost 0.7 %)
    if constexpr (!BF) __builtin_amdgcn_s_setprio(2);
    const int last = 4 * a.n_layers;
    int iq = 0, iw = first, is = 0, at = 0;  // next slot: product, part, slot of it; ring place
    int h0 = 0, h1 = 0, h2 = 0;              // requests of the last three slots
    int base = 0, kq = 0, ahead = 0;         // (bf16) next group; slots asked for, less those the others have had
    DsCopy J = ds_table(a.jobs, first), N;              // the job being requested, the one after it
    auto after = [&]() {
      if ((iw += step) >= a.parts) {
        iw = first;
        ++iq;
      }
      N = ds_table(a.jobs, min(iq, last) * a.parts + iw);
    };
    after();
    bool more = true;
    auto issue = [&]() {
      h2 = h1;
      h1 = h0;
      h0 = 0;
      while (more && is >= J.job.slots) {
        is = base = kq = 0;
        more = iq <= last;
        J = N;
        after();
      }
      if (!more) return;
      if constexpr (BF) {
        ds_copy16(J, base, kq, s.ring + (size_t)at * DS_BSLOT, lw);
        if (++at == a.ring) at = 0;
        ++is;
        ++ahead;
        return;
      }
      uint8_t* dst = s.ring + (size_t)(at % DS_R) * DS_SLOT;
      if (J.job.chunks & DS_Q6) {
        ds_copy<QT_Q6_K>(J, is, dst, lw);
        h0 = DsFmt<QT_Q6_K>::per_loader;
      } else {
        ds_copy<QT_Q4_K>(J, is, dst, lw);
        h0 = DsFmt<QT_Q4_K>::per_loader;
      }
      ++is;
      ++at;
    };
    for (int i = 0; i < (BF ? a.ring : DS_R); ++i) issue();
    lg_barrier();  // the gate's answer
    unsigned go;
    asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                 : "=v"(go)
                 : "v"((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) unsigned*)gate)
                 : "memory");
    if (__builtin_amdgcn_readfirstlane(go) != 1) {
      lg_vmcnt<0>();
      return;
    }
    int slots = ds_table(&a.jobs->job.slots, first * 16);  // of the product that the others are at
    // The slot that a product's end leaves free is asked for when the next operand is staged: a CU's loads return in order, and those
    // that gather the operand would wait for it.  Workgroups that don't attend ask for it right away.
    bool owed = false;
    auto pass = [&](int q) {
      for (int wg = first; wg < a.parts; wg += step) {
        const int n = slots;
        const bool wrap = wg + step >= a.parts;
        slots = ds_table(&a.jobs->job.slots, (min(q + wrap, last) * a.parts + (wrap ? first : wg + step)) * 16);
        if (!n) lg_barrier();
        if constexpr (BF)
          if (a.alone && q == last) lg_barrier();
        for (int t = 0; t < n; ++t) {
          if constexpr (BF) ds_wait(2 * DS_BGROUPS * --ahead);
          else ds_wait(t || owed ? h0 + h1 : h0 + h1 + h2);
          lg_barrier();
          if (t || owed) issue();
          owed = false;
        }
        lg_barrier();
        if (n) owed = true;
      }
    };
#pragma clang loop unroll(disable)
    for (int q = 0; q <= last; ++q) {
      if ((q & 3) == DS_O) {
        int n = 4;
        if (P > 1) n += 2 * ncomb;
        if (owed && first >= nattend) {
          issue();
          owed = false;
        }
        for (int wg = first; wg < a.parts; wg += step)
          for (int i = 0; i < n; ++i) lg_barrier();
      }
      pass(q);
    }
    return;
  }

  // ---- sign in, wait for the others
  DsCtl* ctl = a.ctl;
  DsClock clk{__builtin_amdgcn_s_memrealtime(), a.wait_ticks, gate + 2};
  if (tid == 0) {
    unsigned go = 1;
    const unsigned no = __hip_atomic_load(&ctl->epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!a.alone) {
      if (__hip_atomic_fetch_add(&ctl->arrive, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == gridDim.x) {
        unsigned want = 0;
        __hip_atomic_compare_exchange_strong(&ctl->state, &want, 1u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      while ((go = __hip_atomic_load(&ctl->state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0) {
        if (__builtin_amdgcn_s_memrealtime() - clk.t0 > a.gate_ticks) {
          unsigned want = 0;
          __hip_atomic_compare_exchange_strong(&ctl->state, &want, 2u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
    gate[0] = go;
    gate[1] = no;
    gate[2] = 0;
  }
  for (int i = tid; i < 2 * RED; i += DS_CT) s.red[i] = 0.f;
  if constexpr (BF)
    for (int i = tid; i < 2 * a.row_sums; i += DS_CT) s.sums[i] = 0.f;
  for (int i = tid; i < 2 * a.n_layers; i += DS_CT) s.scale[i] = a.kv_scale[i];
  for (int i = tid; i <= 4 * a.n_layers; i += DS_CT) s.jobs[i] = a.jobs[(size_t)i * a.parts + first].job;
  {
    const int r0 = a.jobs[(size_t)DS_O * a.parts + first].job.r0;
    for (int i = tid; i < 2 * a.n_layers * a.own_rows; i += DS_CT) {
      const int n = i / a.own_rows, r = i - n * a.own_rows;
      s.gains[i] = a.gains[(size_t)(n + 1) * a.d + min(r0 + r, a.d - 1)];
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  lg_barrier();
  const bool go = __builtin_amdgcn_readfirstlane(gate[0]) == 1;
  const uint32_t no0 = __builtin_amdgcn_readfirstlane(gate[1]) + 1;

  if (go) {
    uint8_t* xq = s.area;
    int slot = 0, par = 0;
    // of this workgroup's row (the launch with all workgroups): its position, and RoPE of the lane's pair, in every layer
    auto row_of = [&](int wg) { return BF && wg < nattend ? ds_place(wg, brief ? a.n_heads : a.n_heads / G, rows, P).b : 0; };
    auto rope_at = [&](int p) { return a.rope_cs[(size_t)p * (HD / 2) + (ds_tid() & (HD / 2 - 1))]; };
    const int mine = BF ? pos_of(row_of(first)) : pos;
    const float2 rope = rope_at(mine);
    const int last = 4 * a.n_layers;
    // the residual at this thread's row (of O and of down alike, in reverse order of the threads)
    float own = 0.f;
    const int rt0 = DS_CT - 1 - tid, b0 = BF ? rt0 & 3 : 0;
    if (!a.alone && rt0 < s.jobs[DS_O].nrows << SH && b0 < rows) own = a.x[(size_t)b0 * a.d + s.jobs[DS_O].r0 + (rt0 >> SH)];
    // one product after the other, with the attention in front of O's; the code of all of them is one (what a layer runs
    // through stays in the instruction cache)
#pragma clang loop unroll(disable)
    for (int q = 0; q <= last; ++q) {
      const int l = q >> 2, kind = q & 3;
      const uint32_t no = no0 + l;
      if (kind == DS_O) {
        for (int wg = first; wg < a.parts; wg += step) {
          const int p = BF && a.alone ? pos_of(row_of(wg)) : mine;
          const float2 cs = BF && a.alone ? rope_at(p) : rope;
          if (brief) ds_attend<HD, 1, F8, BF>(a, l, wg, 1, p, no, cs, s, clk);
          else ds_attend<HD, G, F8, BF>(a, l, wg, P, p, no, cs, s, clk);
        }
        if (P > 1)
          for (int wg = first; wg < a.parts; wg += step)
            for (int i = 0; i < ncomb; ++i) ds_combine<HD, BF>(a, l, wg + i * a.parts, P, no, s, clk);
      }
#pragma clang loop unroll(disable)
      for (int wg = first; wg < a.parts; wg += step) {
        // (results are written, and the residual they are added to read, by the last waves: a wave's loads are counted behind
        // its stores, and the first ones have the next operand to wait for)
        const int tid = ds_tid(), rt = DS_CT - 1 - tid, b = BF ? rt & 3 : 0;  // (and of operand row b)
        const DsJob job = a.alone ? ds_table(a.jobs, q * a.parts + wg).job : s.jobs[q];
        DsJob j;
        j.r0 = __builtin_amdgcn_readfirstlane(job.r0);
        j.nrows = __builtin_amdgcn_readfirstlane(job.nrows);
        j.chunks = __builtin_amdgcn_readfirstlane(job.chunks);
        j.slots = __builtin_amdgcn_readfirstlane(job.slots);
        const bool q6 = j.chunks & DS_Q6;
        j.chunks &= ~DS_Q6;
        const int K = kind == DS_O ? qd : (kind == DS_DOWN ? a.ff : a.d), nch = K >> 5;
        float2* ms = (float2*)(xq + K);
        // (of the head's rows, which are more, from behind its operand on)
        float* acc = q == last ? (float*)(xq + (BF ? rows * (2 * K + DS_BPAD) : K + K / 2)) : s.sums + (BF ? par * a.row_sums : 0);
        float* red = s.red + par * RED;
        par ^= 1;
        const bool resid = kind == DS_O || kind == DS_DOWN;
        const int nr = kind == DS_O ? 2 * l : kind == DS_GU ? 2 * l : kind == DS_DOWN ? 2 * l + 1 : 2 * l - 1;  // the residual it makes or reads
        const int n = j.nrows << SH;
        const bool writes = (DS_NG - 1 - __builtin_amdgcn_readfirstlane(tid >> 6)) * 64 < n;  // waves that have results to write
        if (a.alone && resid && rt < n && b < rows) {
          const size_t at = (size_t)b * a.d + j.r0 + (rt >> SH);
          own = nr ? __hip_atomic_load(a.resid + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : a.x[at];
          asm volatile("" : "+v"(own));  // (waited for here)
        }
        const DsAt place = BF ? ds_at_first(tid >> 7, DS_BGROUPS, K >> 9) : q6 ? ds_at_first(tid, DsFmt<QT_Q6_K>::CH, nch) : ds_at_first(2 * tid, DsFmt<QT_Q4_K>::CH, nch);
        if (kind == DS_DOWN) {
          ds_stage<IN_BF16, BF>(nullptr, a.h + (size_t)l * rows * (a.ff / 2), no, rows, K, nullptr, xq, ms, red, clk);
        } else if (q == 0) {
          ds_stage<IN_X, BF>(a.x, nullptr, 0, rows, K, a.gains, xq, ms, red, clk);
        } else {
          const uint32_t nx = kind == DS_QKV ? no - 1 : no;
          ds_stage<IN_F32, BF>(nullptr, kind == DS_O ? a.attn + (size_t)l * rows * qd : a.xn + (size_t)nr * rows * a.d, nx, rows, K, nullptr, xq,
                               ms, red, clk);
          if (kind != DS_O) ds_squares<BF>(a, a.sq + (size_t)nr * rows * a.parts, nx, rows, red, clk);
        }
        if constexpr (BF)
          if (q == last) {
            if (a.alone) lg_barrier();  // (the part before may still be read)
            for (int i = tid; i < 2 * DS_BROWS * j.nrows; i += DS_CT) acc[i] = 0.f;
          }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        lg_barrier();  // the operand is staged, slot 0 there
        float inv = 1.f;
        if (!resid && writes) {  // (behind the product it took 0.7 us)
          float t = 0.f;
          if constexpr (BF) {
            const int m = q ? a.parts >> 6 : K >> 9;  // sums of a row
            for (int w = 0; w < m; ++w) t += red[min(b, rows - 1) * m + w];
          } else {
            t = lanes_sum<16>((tid & 15) < DS_NG ? red[tid & 15] : 0.f);
          }
          inv = rsqrtf(t / (float)K + a.eps);
        }
        if constexpr (BF) {
          for (int i = tid; i < a.row_sums; i += DS_CT) s.sums[par * a.row_sums + i] = 0.f;  // the next product's
          ds_dot16(j, place, K, rows, a.ring, slot, s, xq, (double*)acc);
        } else {
          if (q6) ds_dot<QT_Q6_K>(j, place, nch, ds_run(nch), slot, s, (int8_t*)xq, ms, acc);
          else ds_dot<QT_Q4_K>(j, place, nch, ds_run(nch >> 1), slot, s, (int8_t*)xq, ms, acc);
        }
        const int n1 = q6 ? nch : nch >> 1, terms = n1 >> __builtin_ctz(ds_run(n1));
        auto sum = [&](int i) __attribute__((always_inline)) {
          if constexpr (BF) return (float)((const double*)acc)[i];
          else return ds_sum(acc + i, j.nrows, terms);
        };
        // (what all other workgroups wait for: in front of the waves that go on to the next operand.  Those may not skip this part, though they
        // have nothing to write: waiting earlier they take more from the writing wave than the priority gives back)
        if (writes) __builtin_amdgcn_s_setprio(3);
        if (resid) {
          // (rows by the last wave's lanes, further ones by those before; the squares go with the first word)
          const int r = rt >> SH;
          const bool on = rt < n && b < rows;
          const float x = on ? own + sum(rt) : 0.f;
          float gain = s.gains[nr * a.own_rows + min(r, a.own_rows - 1)];
          if (a.alone) {
            gain = a.gains[(size_t)(nr + 1) * a.d + j.r0 + (on ? r : 0)];
            asm volatile("" : "+v"(gain));
          }
          own = x;
          if (on) {
            ds_put(a.xn + ((size_t)nr * rows + b) * a.d + ds_at(j.r0 + r), __float_as_uint(x * gain), no);
            if (a.alone) __hip_atomic_store(a.resid + (size_t)b * a.d + j.r0 + r, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
          float sq = x * x;
          if constexpr (BF) {  // over the lanes of an operand row
            sq += lane_dpp<0x124>(sq);
            sq += lane_dpp<0x128>(sq);
            sq = lane_xor32(lane_xor16(sq, LaneAdd{}), LaneAdd{});
          } else {
            sq = wave_sum(sq);
          }
          if (rt < rows) ds_put(a.sq + ((size_t)nr * rows + rt) * a.parts + wg, __float_as_uint(sq), no);
        } else if (b < rows) {
          if (q == last) {
            for (int i = rt; i < n; i += DS_CT) a.logits[(size_t)b * a.ldl + j.r0 + (i >> SH)] = sum(i) * inv;
          } else if (kind == DS_QKV) {
            for (int i = rt; i < n; i += DS_CT) ds_put(a.qkv + ((size_t)l * rows + b) * a.nqkv + j.r0 + (i >> SH), __float_as_uint(sum(i) * inv), no);
          } else {
            for (int i = rt; i < n >> 2; i += DS_CT) {
              const int u = i >> SH;
              float v[4];
#pragma unroll
              for (int k = 0; k < 4; ++k) v[k] = sum(((4 * u + k) << SH) + b);
              const float f0 = glu_act(v[0] * inv, ACT_SILU) * (v[1] * inv), f1 = glu_act(v[2] * inv, ACT_SILU) * (v[3] * inv);
              ds_put(a.h + ((size_t)l * rows + b) * (a.ff / 2) + ds_at16((j.r0 >> 2) + u), (uint32_t)f32_to_bf16(f0) | (uint32_t)f32_to_bf16(f1) << 16, no);
            }
          }
        }
        __builtin_amdgcn_s_setprio(0);
      }
    }
  }
  // ---- sign out, late workgroups with a count of their own in the same word, so that the last one has seen them all; it clears the gate and says
  // whether the step is done
  if (tid == 0) {
    const unsigned mine = go && gate[2] ? DS_LATE + 1 : 1;
    const unsigned gone = __hip_atomic_fetch_add(&ctl->done, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + mine;
    if (gone % DS_LATE == gridDim.x) {
      ctl->arrive = 0;
      ctl->state = 0;
      ctl->done = 0;
      ctl->epoch = no0 - 1 + a.n_layers;
      ctl->failed = !a.alone && (!go || gone > DS_LATE);
      if (a.alone) __hip_atomic_store(a.host_failed, ++ctl->alone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// LDS behind the ring and the operand
int ds_rest(const DsArgs& a) {
  const int red = a.bf16 ? ds_red<true>() : ds_red<false>();
  return ((a.bf16 ? 2 : 1) * a.row_sums + 2 * red + 4 + (2 * a.n_layers + 3) / 4 * 4) * 4 + (4 * a.n_layers + 1) * (int)sizeof(DsJob) + 2 * a.n_layers * a.own_rows * 4;
}
int ds_lds(const DsArgs& a) { return (a.bf16 ? a.ring * DS_BSLOT : DS_R * DS_SLOT) + a.area_bytes + ds_rest(a); }

template <int HD, int G, bool F8, bool BF>
void ds_launch(DsArgs a, hipStream_t st) {
  const int lds = ds_lds(a);
  auto* k = decode_stream_kernel<HD, G, F8, BF>;
  static const hipError_t set = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  HIP_CHECK(set);
  a.alone = 0;
  hipLaunchKernelGGL(k, dim3(a.parts), dim3(DS_THREADS), lds, st, a);
  a.alone = 1;
  a.wait_ticks = ~0ull;
  hipLaunchKernelGGL(k, dim3(1), dim3(DS_THREADS), lds, st, a);
  HIP_CHECK(hipGetLastError());
}

template <int HD, bool F8, bool BF>
void ds_heads(const DsArgs& a, hipStream_t st) {
  const int g = a.n_heads / a.n_kv_heads;
  if (g % 4 == 0) ds_launch<HD, 4, F8, BF>(a, st);
  else if (g == 2) ds_launch<HD, 2, F8, BF>(a, st);
  else ds_launch<HD, 1, F8, BF>(a, st);
}
template <int HD, bool F8>
void ds_format(const DsArgs& a, hipStream_t st) {
  if (a.bf16) ds_heads<HD, F8, true>(a, st);
  else ds_heads<HD, F8, false>(a, st);
}

}  // namespace

DsCopy ds_job(const QWeight& w, int r0, int nrows, int row0) {
  if (w.qtype == QT_BF16) {
    DsCopy j{};
    const uint64_t rb = (uint64_t)w.cols * 2;  // (p[1] .. unused otherwise)
    const int groups = (nrows + 3) / 4 * (w.cols / 512);
    j.p[0] = j.p[2] = j.p[3] = w.p0 + (size_t)r0 * rb;
    j.p[1] = (const uint8_t*)rb;
    j.job = {row0 + r0, nrows, groups, (groups + DS_BGROUPS - 1) / DS_BGROUPS};
    return j;
  }
  const size_t nch = w.cols / 32, c = (size_t)r0 * nch;
  const bool q6 = w.qtype == QT_Q6_K;
  const int chunks = (int)(nrows * nch), ch = q6 ? DsFmt<QT_Q6_K>::CH : DsFmt<QT_Q4_K>::CH;
  DsCopy j{};
  j.p[0] = w.p0 + c * 16;
  j.p[1] = w.p1 + (q6 ? c * 8 : c * 2);
  j.p[2] = q6 ? w.p2 + c * 2 : w.p0;
  j.p[3] = q6 ? w.p3 + c / 4 : w.p0;
  j.job = {row0 + r0, nrows, chunks | (q6 ? DS_Q6 : 0), (chunks + ch - 1) / ch};
  return j;
}

int ds_sums(const QWeight& w, int rows) { return w.qtype == QT_BF16 ? rows * 2 * DS_BROWS : rows * ds_terms(w.cols, w.qtype == QT_Q6_K); }

bool ds_plan(DsArgs& a, int hd, int max_sums, int head_sums, int rows) {
  const int qd = a.n_heads * hd, g = a.n_heads / a.n_kv_heads;
  if ((hd != 64 && hd != 128) || a.n_heads % a.n_kv_heads || !(g == 1 || g == 2 || g == 4 || g == 8)) return false;
  // whole waves of octets, rows that 16 chunks divide; every workgroup with rows of O, gate/up and down (see the exchanges above)
  if (a.d % 512 || qd % 512 || a.ff % 512 || a.d < 2 * a.parts || a.ff / 2 < 2 * a.parts) return false;
  if (rows < 1 || rows > (a.bf16 ? DS_BROWS : 1) || rows * a.n_heads > a.parts) return false;
  const int width = a.bf16 ? DS_BROWS : 1;  // threads of a row that is written
  a.rows = rows;
  a.own_rows = (a.d + a.parts - 1) / a.parts;
  if (a.own_rows * width > 64) return false;  // (a wave holds a workgroup's rows of the residual)
  const int K = std::max({a.d, qd, a.ff});
  const int gl = g % 4 == 0 ? 4 : g;
  const int attn = gl * hd * 2 + 2 * hd * 2 + DS_AW * gl * 2 * 4 + DS_AW * gl * hd * 4;
  auto operand = [&](int k) { return a.bf16 ? rows * (2 * k + DS_BPAD) : k + k / 2; };
  a.row_sums = (max_sums + 63) / 64 * 64;
  // (int8: the head's sums run on into the layers')
  const int head = operand(a.d) + head_sums * 4 - (a.bf16 ? 0 : a.row_sums * 4);
  a.area_bytes = (std::max({operand(K), head, attn, DS_PMAX * 18 * 4}) + 255) / 256 * 256;
  if (a.bf16) {
    // sums of squares: 64 workgroups a word of LDS, or 512 columns
    if (a.parts % 64 || rows * std::max(a.parts / 64, a.d / 512) > ds_red<true>()) return false;
    a.ring = std::min(DS_BRING, (160 * 1024 - a.area_bytes - ds_rest(a)) / DS_BSLOT);
    if (a.ring < 4) return false;  // (what is in flight to a CU: 64 KB)
  }
  return ds_lds(a) <= 160 * 1024;
}

void launch_decode_stream(const DsArgs& a, int hd, hipStream_t st) {
  if (hd == 64) a.kv_fp8 ? ds_format<64, true>(a, st) : ds_format<64, false>(a, st);
  else a.kv_fp8 ? ds_format<128, true>(a, st) : ds_format<128, false>(a, st);
}

}  // namespace aios
