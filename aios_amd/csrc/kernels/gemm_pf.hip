// Host side of the prefill GEMM (gemm_pf.h): which launches it serves and the tile / split-K plan.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <stdexcept>
#include <mutex>
#include <set>
#include <tuple>
#include <vector>

#include "gemm_pf.h"

namespace aios {

extern template bool pf_launch_fmt<QT_BF16, QT_BF16>(const GemmQArgs&, int, int, int, hipStream_t);
#ifndef AIOS_BF16_ONLY
extern template bool pf_launch_fmt<QT_Q4_K, QT_Q4_K>(const GemmQArgs&, int, int, int, hipStream_t);
extern template bool pf_launch_fmt<QT_Q6_K, QT_Q6_K>(const GemmQArgs&, int, int, int, hipStream_t);
extern template bool pf_launch_fmt<QT_Q4_K, QT_Q6_K>(const GemmQArgs&, int, int, int, hipStream_t);
extern template bool pf_launch_fmt<QT_Q5_K, QT_Q5_K>(const GemmQArgs&, int, int, int, hipStream_t);
extern template bool pf_launch_fmt<QT_Q5_K, QT_Q6_K>(const GemmQArgs&, int, int, int, hipStream_t);
extern template bool pf_launch_fmt<QT_Q4_0, QT_Q4_0>(const GemmQArgs&, int, int, int, hipStream_t);
extern template bool pf_launch_fmt<QT_Q8_0, QT_Q8_0>(const GemmQArgs&, int, int, int, hipStream_t);
#endif

bool pfkb_serves(const GemmQArgs& a, int bm, int bn, int S);            // gemm_pfk_bf16.hip
bool pfkb_run(const GemmQArgs& a, int bm, int bn, int S, hipStream_t st);
#ifndef AIOS_BF16_ONLY
bool pfk_serves(const GemmQArgs& a, int bm, int bn, int S);             // gemm_pfk.hip
bool pfk_run(const GemmQArgs& a, int bm, int bn, int S, hipStream_t st);
#else
static bool pfk_serves(const GemmQArgs&, int, int, int) { return false; }
static bool pfk_run(const GemmQArgs&, int, int, int, hipStream_t) { return false; }
#endif

static int pf_env(const char* name, int dflt) {
  const char* e = std::getenv(name);
  return e ? std::atoi(e) : dflt;
}

struct PfPlan {
  int bm = 0, bn = 0, s = 1;  // s < 0: stream-K over the CUs (gemm_pf.h pf_stream_k)
};

// Modelled time of one launch.  Per workgroup: max(MFMA time at the tile's sustained fraction of the
// per-CU peak, its slot bytes at the per-CU L2 gather rate) + a fixed prologue / epilogue; a grid
// larger than the chip runs in rounds (one workgroup per CU: the slots fill the LDS); split-K adds
// its fp32 atomic traffic (and the zeroing of a STORE target).
static double pf_model(const GemmQArgs& a, int bm, int bn, int S, bool bf) {
  const double cus = device_cu_count();
  if (bn < 0) {  // K over the waves (gemm_pfk.h): us of a slot of 128 k, of a workgroup, of its rounds
    const int MT = bm / 32, CT = -bn / 32;
    const double tiles = (double)((a.M + bm - 1) / bm) * (a.N / -bn), q6 = a.seg[0].qtype == QT_Q6_K ? 1.3 : 1.0;
    const double slot = std::max(0.08 + 0.032 * MT * CT + (bf ? 0.02 : 0.07) * CT * q6, (bm * 256.0 + CT * 32 * (bf ? 256 : 72) * q6) / 85e3);
    const double wg = a.K / 128.0 / S * slot + 3.5 + 0.26 * MT * CT;
    return (std::ceil(tiles * S / cus) * wg + (S > 1 ? 3.5 : 0.0) + 1.5) * 1e-6;
  }
  const double tiles = (double)((a.M + bm - 1) / bm) * (a.N / bn);
  const double ksteps = (double)(a.K / 64) / S;
  // sustained MFMA fraction per tile shape (dequant VALU + LDS fragment reads beside the MFMAs)
  double eff = bm == 256 ? 0.55 : (bm == 128 ? 0.48 : 0.32);
  if (bn == 128) eff *= 0.85;
  const double t_mfma = 2.0 * bm * bn * 64 * ksteps / (eff * 9.6e12);
  const double slot = bm * 128.0 + bn * (bf ? 128.0 : 48.0);
  const double t_mem = slot * ksteps / 55e9;
  const double t_wg = std::max(t_mfma, t_mem) + 2.5e-6;
  if (S < 0) {  // stream-K: every CU the same share of the tile x K-step iterations, ~2 partial tiles each
    const double iters = tiles * (a.K / 64.0), per = std::ceil(iters / cus);
    const double t_it = std::max(t_mfma, t_mem) / ksteps;
    return per * t_it + 2 * 2.5e-6 + (double)cus * 2 * bm * bn * 4 / 1.2e12 +
           (a.epi == GEPI_STORE ? (double)a.M * a.N * 4 / 4e12 : 0.0);
  }
  double t = std::ceil(tiles * S / cus) * t_wg;
  const double R = std::fmod(tiles, cus);
  if (bm == 256 && S == 1 && (bn == 128 || !bf) && tiles > cus && R > 0 && 2 * R <= cus)  // tail split
    t = (std::floor(tiles / cus) + (bn == 256 && 4 * R <= cus ? 0.4 : 0.6)) * t_wg;
  if (S > 1) t += (double)a.M * a.N * 4 * S / 1.2e12 + (a.epi == GEPI_STORE ? (double)a.M * a.N * 4 / 4e12 : 0.0);
  return t;
}

// the tiles there are, largest first: gemm_pf.h pf_launch_fmt, and with a minus before the columns gemm_pfk.hip (K over the waves)
static const struct { int bm, bn; } PF_TILES[] = {{256, 256}, {256, 128}, {160, 128}, {128, 256}, {128, 128}, {96, 128}, {64, 256}, {64, 128},
                                                  {160, -128}, {128, -128}, {96, -128}, {64, -128}, {160, -64}, {128, -64}, {96, -64}, {64, -64},
                                                  {160, -32}, {128, -32}, {96, -32}, {64, -32}};
static bool pf_tile_ok(const GemmQArgs& a, int bn) {
  if (a.N % bn) return false;
  for (int s = 0; s < a.nseg; ++s)
    if (a.seg_n0[s] % bn || a.seg[s].rows % bn) return false;
  return true;
}

// Measured plans: one per (shape, formats, epilogue, M bucket), filled by gemm_pf_autotune (the
// engine tunes its projection shapes at finalize); the model below is the fallback.
using PfKey = std::tuple<int, int, int, int, int, int, int, int, int, int>;
// (Two or three to a doubling, where tiles of 32 rows more or less change the plan: 130 rows ran the plan of 256, whose
// gate/up took 83 us where one 160-row tile takes 58.)
int gemm_pf_bucket(int M) {
  for (int b : {64, 96, 128, 160, 192, 256, 320, 384, 512, 640, 768, 1024, 1280, 1536, 2048, 2560, 3072})
    if (M <= b) return b;
  return (M + 2047) / 2048 * 2048;
}
static PfKey pf_key(const GemmQArgs& a) {
  // (+ the CU budget: a CU-masked co-resident engine plans for its own CUs)
  return PfKey(a.N, a.K, gemm_pf_bucket(a.M), a.epi, a.seg[0].qtype, a.seg[a.nseg - 1].qtype, a.nseg,
               a.nseg > 1 ? a.seg_n0[1] : 0, a.nseg > 2 ? a.seg_n0[2] : 0, device_cu_count());
}
static std::mutex pf_mu;
static std::map<PfKey, PfPlan>& pf_tuned() {
  static std::map<PfKey, PfPlan> m;
  return m;
}
// the best plan without split-K per key: GEPI_QKV launches whose STORE shape has a split plan of other tiles than those with K over the waves
// (their RoPE / KV-cache epilogue takes no split partials; tuning it for real would write the KV cache), launches with less workspace than
// the best plan's slabs take, and AIOS_GEMM_PF_DETERMINISTIC
static std::map<PfKey, PfPlan>& pf_tuned_s1() {
  static std::map<PfKey, PfPlan> m;
  return m;
}
// AIOS_GEMM_PF_DETERMINISTIC=1: no split-K / stream-K plans (their fp32 atomics add partial tiles in
// arrival order, so the low bits of a prefill could differ run to run even with the same plan)
static bool pf_deterministic() { return pf_env("AIOS_GEMM_PF_DETERMINISTIC", 0) != 0; }
static bool pf_no_split(const GemmQArgs& a) {
  return a.epi == GEPI_SWIGLU_BF16 || a.epi == GEPI_QKV || a.epi == GEPI_STORE16 || pf_deterministic();
}
// stream-K: STORE / ACCUM launches whose tiles leave CUs idle, with an even K-step count per tile
// (every stream-K segment then spans >= 2 steps / 256-blocks); AIOS_GEMM_PF_SK=0 keeps it out of plans
// 256-column tiles: bf16 only.  Quantised, 711 rows, 256 x 256 in stream-K / the best of the others: 6144 x 4096 Q4_K | Q6_K
// 88 / 67 us, 4096 x 4096 Q4_K 63 / 42, 4096 x 14336 Q4_K 121 / 107, Q6_K 133 / 124
static bool pf_sk_ok(const GemmQArgs& a, int bm, int bn, bool bf) {
  if (pf_no_split(a) || (bn == 256 && !bf) || !pf_env("AIOS_GEMM_PF_SK", 1)) return false;
  const int units = a.K / (64 * (bn == 128 ? pf4_groups(a, bm, -1) : 1));
  const double tiles = (double)((a.M + bm - 1) / bm) * (a.N / bn);
  return units % 2 == 0 && units >= 4 && tiles < 2.0 * device_cu_count();
}

// whether the kernels take this tile and split for these args: candidates, modelled and stored plans alike (a stored one
// may be another build's: pf_launch_fmt would run a slice of no K-steps, or a tile that does not divide N, or nothing)
static bool pf_plan_ok(const GemmQArgs& a, const PfPlan& p, bool bf) {
  bool tile = false;
  for (const auto& t : PF_TILES) tile = tile || (t.bm == p.bm && t.bn == p.bn);
  if (!tile || !pf_tile_ok(a, std::abs(p.bn))) return false;
  if (p.bn < 0) return bf ? pfkb_serves(a, p.bm, -p.bn, p.s) : pfk_serves(a, p.bm, -p.bn, p.s);
  if (a.nrm_in || a.epi == GEPI_ACCUM_NORM || (a.epi == GEPI_QKV && (a.kv_fp8 || p.s != 1))) return false;
  if (p.s < 0) return pf_sk_ok(a, p.bm, p.bn, bf);
  if (p.s == 0 || (p.s > 1 && (pf_no_split(a) || a.K / 64 / p.s < 2))) return false;
  return bf || p.bn != 256 || a.K / 256 / p.s >= 1;  // (pf8c slices whole 256-blocks)
}

// ... with all the workspace it may ask for
static bool pf_plan_fits(GemmQArgs a, const PfPlan& p, bool bf) {
  float none;
  int tickets;
  a.ws = &none; a.ws_bytes = SIZE_MAX; a.cnt = &tickets; a.cnt_len = INT_MAX;
  return pf_plan_ok(a, p, bf);
}

// every plan the launcher could run for these args (ksplit > 0 pins the split)
static std::vector<PfPlan> pf_candidates(const GemmQArgs& a, bool bf) {
  std::vector<PfPlan> out;
  for (const auto& t : PF_TILES) {
    for (int S : {1, 2, 3, 4, 6, 8, 12, 16, -1}) {
      if (a.ksplit > 0 && S != a.ksplit) continue;
      PfPlan p;
      p.bm = t.bm; p.bn = t.bn; p.s = S;
      if (!pf_plan_ok(a, p, bf)) continue;
      // (not timed: slices that make over three rounds of workgroups)
      const double wgs = (double)((a.M + t.bm - 1) / t.bm) * (a.N / std::abs(t.bn)) * S;
      if (S > 1 && a.ksplit <= 0 && wgs > 3.0 * device_cu_count()) continue;
      out.push_back(p);
    }
  }
  return out;
}

static PfPlan pf_model_plan(const GemmQArgs& a, bool bf, bool s1_only);
static PfPlan pf_plan(const GemmQArgs& a, bool bf) {
  if (!std::getenv("AIOS_GEMM_PF_TILE") && !std::getenv("AIOS_GEMM_PF_SPLIT") && a.ksplit <= 0) {
    std::lock_guard<std::mutex> g(pf_mu);
    GemmQArgs b = a;  // (the plans of the plain epilogues)
    if (a.epi == GEPI_QKV) b.epi = GEPI_STORE;
    if (a.epi == GEPI_ACCUM_NORM) b.epi = GEPI_ACCUM;
    const PfKey key = pf_key(b);
    auto at = [&](const std::map<PfKey, PfPlan>& plans) {
      const auto it = plans.find(key);
      return it != plans.end() && pf_plan_ok(a, it->second, bf) ? it->second : PfPlan();
    };
    PfPlan p;
    if (!pf_deterministic()) p = at(pf_tuned());
    if (!p.bm) p = at(pf_tuned_s1());  // (the best without split partials or slabs)
    if (p.bm) return p;
  }
  return pf_model_plan(a, bf, false);
}

// the modelled plan (pf_model), or the one AIOS_GEMM_PF_TILE / _SPLIT / a.ksplit pin
static PfPlan pf_model_plan(const GemmQArgs& a, bool bf, bool s1_only) {
  PfPlan best;
  double bt = 1e30;
  // AIOS_GEMM_PF_TILE=BMxBN / AIOS_GEMM_PF_SPLIT=S pin the plan (sweeps: tools/bench_gemm.py --pf-sweep)
  // (read per call: tests and sweeps change them inside one process)
  const char* tile = std::getenv("AIOS_GEMM_PF_TILE");
  const int split = pf_env("AIOS_GEMM_PF_SPLIT", 0);
  int fbm = 0, fbn = 0;
  if (tile) std::sscanf(tile, "%dx%d", &fbm, &fbn);
  for (const auto& tile_ : PF_TILES) {
    const int bm = tile_.bm, bn = tile_.bn;
    if (fbm ? bm != fbm || bn != fbn : bn < 0) continue;  // (K over the waves: where timed, or pinned)
    for (int S : {1, 2, 3, 4, 6, 8, 12, 16, -1}) {
      if (a.ksplit > 0 && S != a.ksplit) continue;
      if (a.ksplit <= 0 && split != 0 && S != split) continue;  // (AIOS_GEMM_PF_SPLIT=-1: stream-K)
      PfPlan p;
      p.bm = bm; p.bn = bn; p.s = S;
      if ((S != 1 && s1_only) || !pf_plan_ok(a, p, bf)) continue;
      const double t = pf_model(a, bm, bn, S, bf);
      if (t < bt) {
        bt = t;
        best = p;
      }
    }
  }
  return best;
}

// Serves M >= AIOS_GEMM_PF_MIN_M (default 33: gemm_wk.hip keeps 2..32) for Q4_K / Q5_K / Q6_K / mixed
// Q4_K|Q6_K, Q5_K|Q6_K / Q4_0 / Q8_0 / bf16 weight stacks with the STORE / ACCUM / SWIGLU epilogues; false -> the caller's
// fallback (formats and fused epilogues this kernel does not do).
static bool pf_eligible(const GemmQArgs& a);
static bool pf_run(const GemmQArgs& a, const PfPlan& p, hipStream_t st) {
  const int qt0 = a.seg[0].qtype, qt1 = a.seg[a.nseg - 1].qtype;
  if (p.bn < 0) return qt0 == QT_BF16 ? pfkb_run(a, p.bm, -p.bn, p.s, st) : pfk_run(a, p.bm, -p.bn, p.s, st);
  if (p.s != 1 && a.epi == GEPI_STORE)
    launch_zero_rows(a.C, a.ldc, a.M, a.N, st);  // (a kernel: the launch may be captured)
#ifndef AIOS_BF16_ONLY
  if (qt0 == QT_Q4_K && qt1 == QT_Q4_K) return pf_launch_fmt<QT_Q4_K, QT_Q4_K>(a, p.bm, p.bn, p.s, st);
  if (qt0 == QT_Q6_K && qt1 == QT_Q6_K) return pf_launch_fmt<QT_Q6_K, QT_Q6_K>(a, p.bm, p.bn, p.s, st);
  if (qt0 == QT_Q4_K && qt1 == QT_Q6_K) return pf_launch_fmt<QT_Q4_K, QT_Q6_K>(a, p.bm, p.bn, p.s, st);
  if (qt0 == QT_Q5_K && qt1 == QT_Q5_K) return pf_launch_fmt<QT_Q5_K, QT_Q5_K>(a, p.bm, p.bn, p.s, st);
  if (qt0 == QT_Q5_K && qt1 == QT_Q6_K) return pf_launch_fmt<QT_Q5_K, QT_Q6_K>(a, p.bm, p.bn, p.s, st);
  if (qt0 == QT_Q4_0 && qt1 == QT_Q4_0) return pf_launch_fmt<QT_Q4_0, QT_Q4_0>(a, p.bm, p.bn, p.s, st);
  if (qt0 == QT_Q8_0 && qt1 == QT_Q8_0) return pf_launch_fmt<QT_Q8_0, QT_Q8_0>(a, p.bm, p.bn, p.s, st);
#endif
  if (qt0 != QT_BF16) return false;
  return pf_launch_fmt<QT_BF16, QT_BF16>(a, p.bm, p.bn, p.s, st);
}

bool launch_gemm_pf(const GemmQArgs& a, hipStream_t st) {
  const int on = pf_env("AIOS_GEMM_PF", 1);
  const int min_m = pf_env("AIOS_GEMM_PF_MIN_M", 33);
  if (!on || a.M < min_m) return false;
  if (!pf_eligible(a)) return false;
  const PfPlan p = pf_plan(a, a.seg[0].qtype == QT_BF16);
  if (!p.bm) return false;
  return pf_run(a, p, st);
}

static bool pf_eligible(const GemmQArgs& a) {
  if (a.nseg < 1 || a.M < 1) return false;
  if (a.epi != GEPI_STORE && a.epi != GEPI_ACCUM && a.epi != GEPI_SWIGLU_BF16 && a.epi != GEPI_QKV &&
      a.epi != GEPI_STORE16 && a.epi != GEPI_ACCUM_NORM)
    return false;
  if (a.epi == GEPI_STORE16 && (!a.C16 || a.seg[0].qtype != QT_BF16)) return false;
  if (a.epi == GEPI_QKV && (a.col0 != 0 || !a.q_out || !a.k_cache || !a.v_cache || !a.pos || !a.rope_cs ||
                            a.head_dim % 2 || a.N != a.q_dim + 2 * a.kv_dim))
    return false;
  if (a.lda % 8 || ((uintptr_t)a.A & 15)) return false;
  const int qt0 = a.seg[0].qtype, qt1 = a.seg[a.nseg - 1].qtype;
  for (int s = 0; s + 1 < a.nseg; ++s)
    if (a.seg[s].qtype != qt0) return false;
  const bool bf = qt0 == QT_BF16;
  if (bf ? (qt1 != QT_BF16 || a.K % 64) : (a.K % 256)) return false;
  // instantiated stacks (gemm_pf_*.hip): the GGUF recipes' Q4_K_M / Q5_K_M (mixed QKV: Q|K Q4_K or Q5_K, V Q6_K),
  // Q6_K, Q4_0 and Q8_0 matrices
  const bool kq = (qt0 == QT_Q4_K && (qt1 == QT_Q4_K || qt1 == QT_Q6_K)) || (qt0 == QT_Q6_K && qt1 == QT_Q6_K) ||
                  (qt0 == QT_Q5_K && (qt1 == QT_Q5_K || qt1 == QT_Q6_K)) || (qt0 == QT_Q4_0 && qt1 == QT_Q4_0) ||
                  (qt0 == QT_Q8_0 && qt1 == QT_Q8_0);
  if (!bf && !kq) return false;
  if (a.epi == GEPI_SWIGLU_BF16 && (!a.C16 || a.nseg != 1)) return false;
  if (a.epi == GEPI_ACCUM_NORM && a.nseg != 1) return false;
  if (a.epi != GEPI_SWIGLU_BF16 && a.epi != GEPI_QKV && a.epi != GEPI_STORE16 && !a.C) return false;
  return true;
}

// Time the candidate plans of the launches (real buffers; outputs overwritten) and keep the fastest per key.  Launches of
// one key -- a projection, layer by layer -- are timed with their weights in turn, as a pass runs them: the same matrix
// again and again lies in the caches (with it, the plans of 2048-wide bf16 layers changed from process to process, and a
// pass of 1500 rows with them: 8.65 to 9.24 ms; so: 8.61 to 8.63).  Returns the number of plans timed.  A key already
// planned in this process -- tuned by an earlier engine or imported, gemm_pf_import -- is left if the kernels take its
// plan, given the workspace: a second engine never changes the plans a first one runs (one whose workspace, its widest product's, is too
// small for a plan's slabs runs the best plan without).
//
// Every candidate that the model puts within twice its best (no plan within 3 % of the fastest lay beyond, for five models'
// 420 keys) in two launches, then those within 12 % of the fastest in four, forwards and backwards; the modelled plan stays
// where it is within 2 %, and ties keep the earlier candidate.  TP ranks then take rank 0's plans (tp.py broadcasts
// gemm_pf_export), and AIOS_GEMM_PF_PLANS persists them across processes.
int gemm_pf_autotune(const std::vector<GemmQArgs>& launches, hipStream_t st) {
  std::vector<std::pair<PfKey, std::vector<const GemmQArgs*>>> work;  // in the order of the launches
  for (const GemmQArgs& a : launches) {
    if (!pf_eligible(a)) continue;
    const PfKey k = pf_key(a);
    const auto at = std::find_if(work.begin(), work.end(), [&](const auto& w) { return w.first == k; });
    if (at != work.end()) {
      at->second.push_back(&a);
      continue;
    }
    std::lock_guard<std::mutex> g(pf_mu);
    const auto it = pf_tuned().find(k);
    if (it == pf_tuned().end() || !pf_plan_fits(a, it->second, a.seg[0].qtype == QT_BF16)) work.push_back({k, {&a}});
  }
  std::vector<hipEvent_t> ev;
  std::set<std::tuple<int, int, int, int, int, int>> loaded;  // (kernels that have run)
  size_t at = 0;                                              // (the next weights)
  int timed = 0;
  // us of a launch under each plan: one after the other without a gap, n launches each
  auto time = [&](const std::vector<const GemmQArgs*>& v, const std::vector<PfPlan>& plans, int n) {
    const GemmQArgs& a = *v[0];
    auto run = [&](const PfPlan& p) { pf_run(*v[at++ % v.size()], p, st); };
    for (const PfPlan& p : plans) {
      const int form = p.bn < 0 ? 0 : p.s == 1 ? (a.N / p.bn) * ((a.M + p.bm - 1) / p.bm) > device_cu_count() : p.s < 0 ? 2 : 3;
      if (loaded.insert({a.seg[0].qtype, a.seg[a.nseg - 1].qtype, a.epi, p.bm, p.bn, form}).second) run(p);
    }
    while (ev.size() <= plans.size()) {
      ev.push_back(nullptr);
      HIP_CHECK(hipEventCreate(&ev.back()));
    }
    run(plans[0]);
    HIP_CHECK(hipEventRecord(ev[0], st));
    for (size_t i = 0; i < plans.size(); ++i) {
      for (int r = 0; r < n; ++r) run(plans[i]);
      HIP_CHECK(hipEventRecord(ev[i + 1], st));
    }
    HIP_CHECK(hipEventSynchronize(ev[plans.size()]));
    std::vector<float> us(plans.size());
    for (size_t i = 0; i < plans.size(); ++i) {
      HIP_CHECK(hipEventElapsedTime(&us[i], ev[i], ev[i + 1]));
      us[i] *= 1e3f / n;
    }
    return us;
  };
  auto same = [](const PfPlan& x, const PfPlan& y) { return x.bm == y.bm && x.bn == y.bn && x.s == y.s; };
  for (const auto& w : work) {
    const auto& v = w.second;
    const GemmQArgs& a = *v[0];
    const bool bf = a.seg[0].qtype == QT_BF16;
    const PfPlan mp = pf_model_plan(a, bf, false), mp1 = pf_model_plan(a, bf, true);
    auto model = [&](const PfPlan& p) { return pf_model(a, p.bm, p.bn, p.s, bf); };
    const std::vector<PfPlan> all = pf_candidates(a, bf);
    double least = 1e30;
    bool waves = false;
    for (const PfPlan& p : all) {
      least = std::min(least, model(p));
      waves = waves || p.bn < 0;
    }
    std::vector<PfPlan> c;
    for (const PfPlan& p : all) {
      // (quantised: beside K over the waves another tile of 128 columns is the fastest for 2 of three models' 270 keys, by 2 %; Mistral's prompts of
      // 700 to 1536 rows as fast without them, its load 0.93 -> 0.75 s: profiles/prefill_tiles.txt)
      // (above 2048 rows the model's tiles stand closer together, and a launch takes up to a millisecond)
      if ((model(p) <= (a.M > 2048 ? 1.6 : 2) * least && !(waves && !bf && p.bn == 128)) || same(p, mp) || same(p, mp1)) c.push_back(p);
    }
    if (c.empty()) continue;
    if (&w == &work[0]) time(v, {c[0]}, 100);  // (the clocks)
    const std::vector<float> us = time(v, c, 2);
    timed += (int)c.size();
    // the fastest, or the fastest without split partials
    auto pick = [&](bool s1) {
      auto in = [&](size_t i) { return !s1 || c[i].s == 1; };
      float least = 1e30f;
      for (size_t i = 0; i < c.size(); ++i)
        if (in(i)) least = std::min(least, us[i]);
      std::vector<PfPlan> f;
      for (size_t i = 0; i < c.size(); ++i)
        if (in(i) && (us[i] <= 1.12f * least || same(c[i], s1 ? mp1 : mp))) f.push_back(c[i]);
      if (f.size() < 2) return f.empty() ? PfPlan() : f[0];
      const size_t n = f.size();
      std::vector<PfPlan> both(f);
      both.insert(both.end(), f.rbegin(), f.rend());
      const std::vector<float> t = time(v, both, 4);
      // (K over the waves by 4 % or not: 4096 x 4096 at 2048 rows, 3 % faster here, took 86 us of a pass where 128 x 256 tiles took 84.  The
      // plain forms are timed: what the fused ones save, a norm's or RoPE's launch of 5 to 20 us, and cost, 1 to 5 us, is not in it)
      auto sum = [&](size_t i) { return (t[i] + t[2 * n - 1 - i]) * (f[i].bn < 0 ? 1.04f : 1.f); };
      size_t best = 0;
      for (size_t i = 1; i < n; ++i)
        if (sum(i) < sum(best)) best = i;
      for (size_t i = 0; i < n; ++i)
        if (same(f[i], s1 ? mp1 : mp) && sum(i) <= 1.02f * sum(best)) return f[i];
      return f[best];
    };
    const PfPlan best = pick(false), best1 = best.s == 1 ? best : pick(true);
    std::lock_guard<std::mutex> g(pf_mu);
    pf_tuned()[w.first] = best;
    if (best1.bm) pf_tuned_s1()[w.first] = best1;
  }
  for (hipEvent_t e : ev) HIP_CHECK(hipEventDestroy(e));
  return timed;
}

// every tuned plan as flat ints: 10 key fields, bm, bn, s, map (0: best, 1: best without split-K)
std::vector<int> gemm_pf_export() {
  std::lock_guard<std::mutex> g(pf_mu);
  std::vector<int> v;
  for (int m = 0; m < 2; ++m)
    for (const auto& kv : (m ? pf_tuned_s1() : pf_tuned())) {
      const PfKey& k = kv.first;
      for (int x : {std::get<0>(k), std::get<1>(k), std::get<2>(k), std::get<3>(k), std::get<4>(k), std::get<5>(k),
                    std::get<6>(k), std::get<7>(k), std::get<8>(k), std::get<9>(k)})
        v.push_back(x);
      v.push_back(kv.second.bm); v.push_back(kv.second.bn); v.push_back(kv.second.s); v.push_back(m);
    }
  return v;
}

// install plans (replacing any tuned for the same keys): TP workers take the leader's, a process
// takes a persisted set; later autotune calls skip these keys
void gemm_pf_import(const std::vector<int>& v) {
  if (v.size() % 14) throw std::runtime_error("gemm_pf_import: bad plan list");
  std::lock_guard<std::mutex> g(pf_mu);
  for (size_t i = 0; i < v.size(); i += 14) {
    const PfKey k(v[i], v[i + 1], v[i + 2], v[i + 3], v[i + 4], v[i + 5], v[i + 6], v[i + 7], v[i + 8], v[i + 9]);
    PfPlan p;
    p.bm = v[i + 10]; p.bn = v[i + 11]; p.s = v[i + 12];
    (v[i + 13] ? pf_tuned_s1() : pf_tuned())[k] = p;
  }
}

// whether launch_gemm_pf takes these args (the engine asks before choosing the GEPI_QKV epilogue
// for a prefill chunk, which only this kernel and the small-M ones implement)
bool gemm_pf_serves(const GemmQArgs& a) {
  if (!pf_env("AIOS_GEMM_PF", 1) || a.M < pf_env("AIOS_GEMM_PF_MIN_M", 33) || !pf_eligible(a)) return false;
  const PfPlan p = pf_plan(a, a.seg[0].qtype == QT_BF16);
  return p.bm != 0;
}

// ... on tiles with K over the waves: those take GEPI_QKV with any plan, GEPI_ACCUM_NORM and nrm_in (a part per 64 columns)
bool gemm_pf_fuses(const GemmQArgs& a) {
  if (!pf_env("AIOS_GEMM_PF", 1) || a.M < pf_env("AIOS_GEMM_PF_MIN_M", 33) || !pf_eligible(a)) return false;
  const bool bf = a.seg[0].qtype == QT_BF16;
  const PfPlan p = pf_plan(a, bf);
  if (p.bn >= 0) return false;
  // (... and would run the plain product on: a split plan of other tiles falls back to the best unsplit one, which may be of these
  // tiles, but was timed as the slower)
  GemmQArgs b = a;
  b.nrm_in = nullptr;
  if (a.epi == GEPI_ACCUM_NORM) b.epi = GEPI_ACCUM;
  if (a.epi == GEPI_QKV) { b.epi = GEPI_STORE; b.C = a.q_out; b.ldc = a.N; }
  const PfPlan q = pf_plan(b, bf);
  return p.bm == q.bm && p.bn == q.bn && p.s == q.s;
}

// the plan the launcher would pick (bindings / tools)
void gemm_pf_plan(const GemmQArgs& a, int& bm, int& bn, int& s) {
  const PfPlan p = pf_plan(a, a.seg[0].qtype == QT_BF16);
  bm = p.bm; bn = p.bn; s = p.s;
}

}  // namespace aios
