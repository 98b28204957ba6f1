// bt_exp.h -- FP64 exponentials and sines of the gfx950 pair kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "bt_kernels.h"

namespace btk {

// e^{-k u} for the kernels' e^{-kappa r} and e^{-r^2/a^2}, from a table of
// 2^(j/256), j < EXP_TAB = 256 (tab, filled by exp_table) and the rate's
// constants ex (exp_rate on the host): c = 256 k / ln 2, rounded once, and
// the largest u that matters (beyond it e^{-k u} is below half the least
// subnormal; a NaN u takes it too).  t = MAGIC - c u rounds the exponent to
// an integer n, which is then the low word of t, and f = -c u - n is one fma
// (exact but for the rounding of c, a relative error of 2^-53 in k u as the
// rounding of the product k u would be).  |f| <= 1/2, so y = f ln2/256 is
// below 1.36e-3 and the Taylor polynomial of e^y - 1 to degree 4 is
// truncated below 3.9e-17; e^{-k u} = 2^(n/256) (1 + (e^y - 1)) is within
// about 1.5 ulp besides the error of k u.
//
// 11 FP64 instructions with the clamp.  The pair kernels issue FP64
// instructions back to back, so the form before this one (64 entries, degree
// 5, e^x of a product x formed first, rint and conversion, ln2 in two parts:
// 15) cost in proportion: Yukawa, N = 1M cluster-cluster, the symmetric
// launch 91 -> 80 ms for 7.4e10 unordered pairs; Coulomb with subtraction,
// N = 2M, 125 -> 114 ms for 1.02e11 beside its far field.
__device__ __forceinline__ double exp_neg(double u, const ExpRate &ex, const double *tab)
{
    constexpr double MAGIC = 0x1.8p52;
    constexpr double A1 = 2.7076061740622863e-03;  // (ln2/256)^k / k!
    constexpr double A2 = 3.6655655969101062e-06;
    constexpr double A3 = 3.3083026805413713e-09;
    constexpr double A4 = 2.2393951908751570e-12;
    u = __builtin_fmin(u, ex.umax);
    const double t = fma(-u, ex.c, MAGIC);
    const double f = fma(-u, ex.c, MAGIC - t);
    const int n = (int)(unsigned)__builtin_bit_cast(unsigned long long, t);
    double p = fma(f, A4, A3);
    p = fma(f, p, A2);
    p = fma(f, p, A1);
    const double s = tab[n & (EXP_TAB - 1)];
    return __builtin_amdgcn_ldexp(fma(s, f * p, s), n >> 8);
}

// The table by the block's threads (read after the block's next barrier).
__device__ __forceinline__ void exp_table(double *tab, int tid)
{
    static_assert(EXP_TAB == 256, "exp_neg's shift and polynomial");
    if (tid < EXP_TAB) tab[tid] = exp2((double)tid * (1.0 / EXP_TAB));
}

// sin(k r), r >= 0, from a table of (sin, cos)(2 pi j / 512), j < SIN_TAB
// (tab, filled by sin_table) and the constants sr (sin_rate on the host):
// 512 k / (2 pi) as c + clo.  As in exp_neg, n = round(c r) is the low word
// of t and f = c r - n an fma, with clo r added; the angle a = 2 pi f / 512
// has |a| <= 6.2e-3, so sin a to degree 5 is truncated below 1.1e-17
// relative and cos a to degree 4 below 8e-17.  Within about 1.5 ulp of 1
// besides the rounding of k r's own size.  Beyond sr.rmax (c r >= 2^50) the
// library's sin (GUARD; without it the caller keeps r below rmax); a NaN r
// gives NaN.
//
// 12 FP64 instructions and one 16-byte table read.  The library's sin (with
// its reduction for every magnitude) and the square root took most of a
// pair: N = 200k particle-cluster, degree 5, 1.4e10 pairs 55.4 -> 26.1 ms.
template <bool GUARD = true>
__device__ __forceinline__ double sin_kr(double r, double k, const SinRate &sr, const double *tab)
{
    if constexpr (GUARD)
        if (__builtin_expect(r >= sr.rmax, 0)) return sin(k * r);
    constexpr double MAGIC = 0x1.8p52;
    constexpr double S1 = 0.01227184630308513, S3 = -3.080196845561248e-07, S5 = 2.3193606829202922e-12;  // (2 pi/512)^k / k!
    constexpr double C2 = -7.529910584327208e-05, C4 = 9.44992556799382e-10;
    const double t = fma(r, sr.c, MAGIC);
    double f = fma(r, sr.c, MAGIC - t);
    f = fma(r, sr.clo, f);
    const int n = (int)(unsigned)__builtin_bit_cast(unsigned long long, t) & (SIN_TAB - 1);
    const double2 sc = reinterpret_cast<const double2 *>(tab)[n];
    const double f2 = f * f;
    const double sf = f * fma(f2, fma(f2, S5, S3), S1);
    const double cm = f2 * fma(f2, C4, C2);  // cos a - 1
    return fma(sc.x, cm, fma(sc.y, sf, sc.x));
}

__device__ __forceinline__ void sin_table(double *tab, int tid, int nthreads)
{
    static_assert(SIN_TAB == 512, "sin_kr's polynomials");
    for (int j = tid; j < SIN_TAB; j += nthreads) {
        double s, c;
        sincospi((double)j * (2.0 / SIN_TAB), &s, &c);
        reinterpret_cast<double2 *>(tab)[j] = make_double2(s, c);
    }
}

}  // namespace btk
