// math_f64.hpp -- FP64 division, square root, exponential and logarithm of the plain FP64 path
// kernel, for arguments in the normal range.
//
// The compiler's own sequences scale their operands against overflow and denormals (a division is
// 2 v_div_scale, the reciprocal, 5 fused steps, v_div_fmas and v_div_fixup; the library's exp and
// log are 30-40 instructions). The path's operands are variances, prices and probabilities far
// from those limits, so the sequences below keep only the arithmetic. v_rcp_f64 and v_rsq_f64 are
// good to 2^-24 (measured over 2^20 arguments: 2^-24.4 and 2^-24.2): one Newton step gives 2^-48,
// and the correction by the exact residual leaves the quotient or root within its last rounding.
#pragma once
#include <hip/hip_runtime.h>

namespace hexo {

// a / b for normal, finite b with a / b in the normal range; NaN or infinite where 1/b overflows.
__device__ __forceinline__ double div_f64(double a, double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(__builtin_fma(-b, r, 1.0), r, r);
    const double q = a * r;
    return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}

// sqrt(x) for x > 0 in the normal range (NaN at 0).
__device__ __forceinline__ double sqrt_f64(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// Coefficients from math_f64_fit.py: e^r = 1 + r + r^2 Q(r) on |r| <= ln(2)/2 (relative error
// 1.6e-17) and log m = 2 s + s z P(z), s = (m - 1)/(m + 1), z = s^2, on m in [sqrt(1/2), sqrt(2)]
// (4.7e-18).
struct MathF64 {
    static constexpr double q[10] = {0.5000000000000001,     0.16666666666666669,    0.041666666666624164,
                                     0.008333333333330072,   0.0013888888917196836,  0.00019841269863035425,
                                     2.4801521321875824e-05, 2.7557268475291603e-06, 2.762007620330394e-07,
                                     2.5100380460244386e-08};
    static constexpr double p[7] = {0.666666666666667,   0.39999999999899505, 0.285714286259754,  0.22222211134778866,
                                    0.18182889127123197, 0.1533172153403835,  0.1461645048788178};
    // ln 2 in two parts, the first with 21 trailing zero bits (its products with exponents are exact)
    static constexpr double ln2_hi = 0x1.62e42fee00000p-1, ln2_lo = 0x1.a39ef35793c76p-33;
};

// e^y for |y| < 700.
__device__ __forceinline__ double exp_f64(double y) {
    const double n = __builtin_rint(y * 1.4426950408889634074);
    const double r = __builtin_fma(-n, MathF64::ln2_lo, __builtin_fma(-n, MathF64::ln2_hi, y));
    double c = MathF64::q[9];
#pragma unroll
    for (int i = 8; i >= 0; --i) c = __builtin_fma(c, r, MathF64::q[i]);
    const double e = __builtin_fma(r * r, c, r) + 1.0;
    return __builtin_amdgcn_ldexp(e, (int)n);
}

// ln x for x > 0 in the normal range: x = 2^e m, f = m - 1, ln m = f - s (f - s^2 P(s^2)). This form, and
// ln 2 in two parts, are those of the logarithm of fdlibm (Sun Microsystems, 1993); the coefficients are
// from math_f64_fit.py.
__device__ __forceinline__ double log_f64(double x) {
    double m = __builtin_amdgcn_frexp_mant(x);  // [1/2, 1)
    const bool low = m < 0.70710678118654752440;
    m = low ? m + m : m;
    const double e = (double)(__builtin_amdgcn_frexp_exp(x) - (low ? 1 : 0));
    const double f = m - 1.0;
    const double s = div_f64(f, 2.0 + f);
    const double z = s * s;
    double c = MathF64::p[6];
#pragma unroll
    for (int i = 5; i >= 0; --i) c = __builtin_fma(c, z, MathF64::p[i]);
    const double t = __builtin_fma(s, __builtin_fma(-z, c, f), -e * MathF64::ln2_lo);
    return __builtin_fma(e, MathF64::ln2_hi, f - t);
}

}  // namespace hexo
