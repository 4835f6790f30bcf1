// gam_math.h -- FP64 reciprocal, square roots and exponential of the step's
// inner kernels.
//
// The interface fluxes and EMFs are bound as much by FP64 vector issue (and
// the clock it costs) as by memory: on gfx950 a correctly rounded division
// is ~11 vector instructions, a square root ~14 and exp ~30, each 4 cycles.
// These forms take 5, 9-12 and 18.  They start from the hardware's seeds
// (v_rcp_f64, v_rsq_f64) and take two Newton steps, which leaves a relative
// 2^-53 (2.5 times that for the reciprocal square root).  Arguments are normal
// and, but for gam_rcp's (an edge's determinant has either sign), positive:
// densities, pressures, squared speeds, sums of face areas.  A zero or infinite
// argument gives NaN where the plain form gives an infinity or 0, except where
// noted; what a caller may set to 0 (Model%dt) is tested first or divided by.
// The host builds (CPU tests) use the plain operations.
#pragma once
#include <cmath>

#ifdef __HIPCC__
#define GAM_HD __host__ __device__
#else
#define GAM_HD
#endif

// 1 / x
GAM_HD inline double gam_rcp(double x)
{
#ifdef __HIP_DEVICE_COMPILE__
    double y = __builtin_amdgcn_rcp(x);
    y = std::fma(std::fma(-x, y, 1.0), y, y);
    return std::fma(std::fma(-x, y, 1.0), y, y);
#else
    return 1.0 / x;
#endif
}

// s = sqrt(x) and r = 1 / sqrt(x) from one seed (Goldschmidt's iteration:
// g -> sqrt(x), h -> 1 / (2 sqrt(x)))
GAM_HD inline void gam_sqrt_rsqrt(double x, double &s, double &r)
{
#ifdef __HIP_DEVICE_COMPILE__
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    double e = std::fma(-h, g, 0.5);
    g = std::fma(g, e, g);
    h = std::fma(h, e, h);
    e = std::fma(-h, g, 0.5);
    g = std::fma(g, e, g);
    h = std::fma(h, e, h);
    s = std::fma(std::fma(-g, g, x), h, g);
    r = h + h;
#else
    s = std::sqrt(x);
    r = 1.0 / s;
#endif
}

// sqrt(x) for x >= 0, 0 included (below 1e-280 the result is small, not exact)
GAM_HD inline double gam_sqrt(double x)
{
#ifdef __HIP_DEVICE_COMPILE__
    const double y = __builtin_amdgcn_rsq(std::fmax(x, 1.0e-280));
    double g = x * y, h = 0.5 * y;
    double e = std::fma(-h, g, 0.5);
    g = std::fma(g, e, g);
    h = std::fma(h, e, h);
    e = std::fma(-h, g, 0.5);
    g = std::fma(g, e, g);
    return std::fma(std::fma(-g, g, x), h, g);
#else
    return std::sqrt(x);
#endif
}

// exp(x) for x <= 0: x = n ln 2 + r with |r| <= ln(2) / 2, the Taylor
// polynomial of degree 13 in r (remainder below 5e-18) and a scaling by
// 2^n; 0 below -800 (and for -inf, and for NaN).
GAM_HD inline double gam_exp_neg(double x)
{
    x = std::fmax(x, -800.0);
    const double n = std::rint(x * 1.4426950408889634074);          // 1 / ln 2
    const double r = std::fma(-n, 2.3190468138462995584e-17,        // ln 2 to 107 bits
                              std::fma(-n, 0.69314718055994528623, x));
    double p = 1.0 / 6227020800.0;
    p = std::fma(p, r, 1.0 / 479001600.0);
    p = std::fma(p, r, 1.0 / 39916800.0);
    p = std::fma(p, r, 1.0 / 3628800.0);
    p = std::fma(p, r, 1.0 / 362880.0);
    p = std::fma(p, r, 1.0 / 40320.0);
    p = std::fma(p, r, 1.0 / 5040.0);
    p = std::fma(p, r, 1.0 / 720.0);
    p = std::fma(p, r, 1.0 / 120.0);
    p = std::fma(p, r, 1.0 / 24.0);
    p = std::fma(p, r, 1.0 / 6.0);
    p = std::fma(p, r, 0.5);
    p = std::fma(p, r, 1.0);
    p = std::fma(p, r, 1.0);
    return std::ldexp(p, (int)n);
}
