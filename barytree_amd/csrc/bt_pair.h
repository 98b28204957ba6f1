// bt_pair.h -- FP64 pair kernels that depend on r alone, from r^2.
#pragma once
#include <cfloat>

#include "bt_exp.h"
#include "bt_kernels.h"
#include "bt_rsq.h"

namespace btk {

constexpr int KC = 1, KY = 2, KR = 3;
constexpr int KRY = KERNEL_REG_YUKAWA, KAT = KERNEL_ATAN, KSR = KERNEL_SIN_OVER_R, KMQ = KERNEL_MQ,
              KRU = KERNEL_RBS_U, KRV = KERNEL_RBS_V, KUS = KERNEL_USER;
constexpr bool radial(int ker)
{
    return ker == KC || ker == KY || ker == KR || ker == KRY || ker == KSR || ker == KUS;
}
// the kernel's FP64 evaluation reads the table of exp_neg or of sin_kr
constexpr bool exp_kernel(int ker, bool ss) { return ker == KY || ker == KRY || ker == KUS || (ss && ker != KSR); }
// the subtraction's Gaussian e^{-r^2/a^2} as the product of e^{-dx^2/a^2} and
// e^{-(dy^2+dz^2)/a^2}, which tensor grids share over their pencils
constexpr bool separable_gauss(int ker, bool ss) { return ss && (ker == KC || ker == KR); }
// doubles of that table (1 without one)
constexpr int pair_table_len(int ker, bool ss) { return ker == KSR ? 2 * SIN_TAB : (exp_kernel(ker, ss) ? EXP_TAB : 1); }
template <int KER, bool SS>
__device__ __forceinline__ void pair_table(double *tab, int tid, int nthreads)
{
    if constexpr (KER == KSR) sin_table(tab, tid, nthreads);
    else if constexpr (exp_kernel(KER, SS)) exp_table(tab, tid);
}

// e^{-kappa r} and e^{-r^2 inv_a2}: the table form (TAB, bt_exp.h) or the
// library's
template <bool TAB>
__device__ __forceinline__ double exp_kr(double r, const KParams &kp, const double *tab)
{
    if constexpr (TAB) return exp_neg(r, kp.ek, tab);
    else return exp(-kp.p0 * r);
}
template <bool TAB>
__device__ __forceinline__ double exp_r2(double r2, const KParams &kp, const double *tab)
{
    if constexpr (TAB) return exp_neg(r2, kp.eg, tab);
    else return exp(-r2 * kp.inv_a2);
}

// Regularized Yukawa, sin-over-r and the user example: one pair's term
// (r by r^2 rsq64(r^2) with TAB, about 1 ulp; r = 0 for coincident points,
// which the regularized kernel does not skip).  GUARD as for sin_kr.
template <int KER, bool SS, bool CHECK, bool TAB, bool GUARD = true>
__device__ __forceinline__ double term_r2(double r2, double a, double b, double tq, const KParams &kp,
                                          const double *tab)
{
    if constexpr (KER == KRY) {
        const double r = TAB ? r2 * rsq64(fmax(r2, 1e-300)) : sqrt(r2);
        const double e = exp_kr<TAB>(r, kp, tab) * rsq64(r2 + kp.eps2);
        return (SS ? fma(-tq, b, a) : a) * e;
    } else {
        static_assert(KER == KSR || KER == KUS, "term_r2");
        const double ir = rsq64(r2);
        double r = TAB ? r2 * ir : sqrt(r2), v;
        if constexpr (KER == KSR) {
            // the sine sees k times r's rounding: one Newton step makes r
            // as good as the root (half an ulp)
            if constexpr (TAB) r = fma(fma(-r, r, r2), 0.5 * ir, r);
            v = (TAB ? sin_kr<GUARD>(r, kp.p0, kp.sn, tab) : sin(kp.p0 * r)) * ir;
        } else {
            v = exp_kr<TAB>(r, kp, tab) * ir;
        }
        if constexpr (CHECK) v = r > DBL_MIN ? v : 0.0;
        return a * v;
    }
}

// acc += the pair's term; a, b, tq, CHECK as for pair_pot (bt_kernels.hip).
template <int KER, bool SS, bool CHECK, bool TAB>
__device__ __forceinline__ void pair_r2(double r2, double a, double b, double tq, const KParams &kp, double &acc,
                                        const double *tab)
{
    if constexpr (KER == KC) {
        double ir = rsq64(r2);
        if constexpr (CHECK) ir = r2 > (SS ? 0.0 : DBL_MIN) ? ir : 0.0;
        if constexpr (!SS) acc = fma(a, ir, acc);
        else acc = fma(fma(-tq * b, exp_r2<TAB>(r2, kp, tab), a), ir, acc);
    } else if constexpr (KER == KY) {
        const double ir = rsq64(r2);
        double e = exp_kr<TAB>(r2 * ir, kp, tab) * ir;
        if constexpr (CHECK) e = r2 > 0.0 ? e : 0.0;
        if constexpr (!SS) acc = fma(a, e, acc);
        else acc = fma(fma(-tq, b, a), e, acc);
    } else if constexpr (KER == KR) {
        const double ir = rsq64(r2 + kp.eps2);
        if constexpr (!SS) acc = fma(a, ir, acc);
        else acc = fma(fma(-tq * b, exp_r2<TAB>(r2, kp, tab), a), ir, acc);
    } else {
        acc += term_r2<KER, SS, CHECK, TAB>(r2, a, b, tq, kp, tab);
    }
}

}  // namespace btk
