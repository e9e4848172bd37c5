// Host side of the prefill GEMM with K over the waves (gemm_pfk.h): the launches and tiles it takes.
#include "gemm_pfk.h"

namespace aios {

// g(QT0, QT1) of the weights' formats, false for others
template <typename G>
static bool pfk_fmt(const GemmQArgs& a, G g) {
#define PFK_Q(N) std::integral_constant<int, N> {}
  const int q0 = a.seg[0].qtype, q1 = a.seg[a.nseg - 1].qtype;
  for (int s = 0; s + 1 < a.nseg; ++s)
    if (a.seg[s].qtype != q0) return false;
  if (q0 == QT_Q4_K && q1 == QT_Q4_K) return g(PFK_Q(QT_Q4_K), PFK_Q(QT_Q4_K));
  if (q0 == QT_Q6_K && q1 == QT_Q6_K) return g(PFK_Q(QT_Q6_K), PFK_Q(QT_Q6_K));
  if (q0 == QT_Q4_K && q1 == QT_Q6_K) return g(PFK_Q(QT_Q4_K), PFK_Q(QT_Q6_K));
  return false;
#undef PFK_Q
}

template <int QT0, int QT1, int MT, int CT, int NG>
constexpr bool pfk_fits() {  // two blocks of weights beside the slots of X (160 x 128 of Q6_K: no)
  return PfkLayout<QT0, MT, CT, NG>::NWB >= 2 && PfkLayout<QT1, MT, CT, NG>::NWB >= 2;
}

// bm x bn tiles divide N and every segment (pf_plan_ok).  32-bit offsets into X and the planes
bool pfk_serves(const GemmQArgs& a, int bm, int bn, int S) {
  if (a.epi == GEPI_STORE16 || !pfk_epi_ok(a, bn)) return false;
  if (S < 1 || S > a.K / 256 || a.K % 256) return false;
  if ((a.epi == GEPI_SWIGLU_BF16 || a.epi == GEPI_ACCUM_NORM) && a.nseg != 1) return false;
  if ((size_t)a.M * a.lda * 2 >= 0xfffffff0u) return false;
  for (int s = 0; s < a.nseg; ++s)
    if ((size_t)a.seg[s].rows * a.K / 2 >= 0xfffffff0u) return false;
  if (!pfk_slabs_ok(a, bm, bn, S)) return false;
  return pfk_fmt(a, [&](auto q0, auto q1) {
    return pfk_tile(bm, bn, [&](auto mt, auto ct, auto ng) {
      return pfk_fits<decltype(q0)::value, decltype(q1)::value, decltype(mt)::value, decltype(ct)::value, decltype(ng)::value>();
    });
  });
}

bool pfk_run(const GemmQArgs& a, int bm, int bn, int S, hipStream_t st) {
  return pfk_fmt(a, [&](auto q0, auto q1) {
    return pfk_tile(bm, bn, [&](auto mt, auto ct, auto ng) {
      constexpr int Q0 = decltype(q0)::value, Q1 = decltype(q1)::value, MT = decltype(mt)::value, CT = decltype(ct)::value,
                    NG = decltype(ng)::value;
      if constexpr (pfk_fits<Q0, Q1, MT, CT, NG>()) {
        pfk_launch<Q0, Q1, MT, CT, NG>(a, S, st);
        return true;
      }
      return false;
    });
  });
}

}  // namespace aios
