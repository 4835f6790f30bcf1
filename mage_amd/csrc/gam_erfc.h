// gam_erfc.h -- erfc(z) and exp(-z^2) in FP64 for the kinetic fluxes.
// Generated by gen_erfc.py (same directory); do not edit by hand.
//
// a = |z|, t = 2/(2+a), u = 2t-1:  erfc(a) = t * exp(-a^2) * Q(u) with Q a
// degree-25 polynomial (monomial coefficients below), erfc(-a) = 2 - erfc(a).
// exp(-a^2) is formed from the exact split a^2 = hi + lo (one fma), so the
// pair is accurate to about 8e-16 relative for |z| <= 20.  Host and device
// compile the same code (the host build is what the CPU test checks) but
// for the reciprocal, see gam_math.h.
#pragma once
#include "gam_math.h"

static constexpr double GAM_ERFC_Q[26] = {
    0.5107913526210115,
    0.34358034220690514,
    0.13973604627801475,
    0.01822111575345904,
    -0.010755330944036532,
    -0.0032395925345820673,
    0.0015453060141013286,
    0.0004186480432791111,
    -0.0003315365766901461,
    -1.7185831874889752e-05,
    7.223418829504806e-05,
    -1.7073781133818914e-05,
    -1.084298532996441e-05,
    8.05787586714734e-06,
    -5.776423611511427e-07,
    -1.8150355080541665e-06,
    1.0305699215291105e-06,
    -1.3754508233185945e-08,
    -3.262460935296672e-07,
    1.7867229479168533e-07,
    3.6000845292079935e-08,
    -6.965842943409138e-08,
    6.52043461440154e-09,
    1.3216325517632649e-08,
    -1.911173728607894e-09,
    -1.05903331435718e-09};

// Returns erfc(z); e receives exp(-z^2).
GAM_HD inline double gam_erfc_exp(double z, double &e)
{
    const double a = std::fabs(z);
    const double t = 2.0 * gam_rcp(2.0 + std::fmin(a, 1.0e300));
    const double u = std::fma(2.0, t, -1.0);
    double q = GAM_ERFC_Q[25];
#pragma unroll
    for (int n = 24; n >= 0; n--) q = std::fma(q, u, GAM_ERFC_Q[n]);
    const double hi = a * a;
    // 0 for a = inf; a NaN goes through here into both results (the fmin above
    // and gam_exp_neg drop it)
    const double lo = hi >= 1.0e300 ? 0.0 : std::fma(a, a, -hi);
    e = gam_exp_neg(-hi);
    e = std::fma(-e, lo, e);
    const double r = t * e * q;
    return z < 0.0 ? 2.0 - r : r;
}

