#!/usr/bin/env python3
"""Generate gam_erfc.h: coefficients of the FP64 erfc used by the flux
kernels.

For a >= 0 let t = 2/(2+a) and u = 2t - 1 (u in (-1, 1]).  The function
    Q(u) = exp(a^2) erfc(a) / t
is smooth on [-1, 1] (Q(1) = 1, Q(-1) = 1/(2 sqrt(pi))), so a short
polynomial in u represents it: erfc(a) = t exp(-a^2) Q(u).  The change of
variable is Schonfelder's (Math. Comp. 32 (1978) 1232-1240).  Q is
interpolated at 60 Chebyshev nodes in 40-digit arithmetic (mpmath), the
series is cut at degree 25 (the next coefficient is below 4e-17) and turned
into monomial coefficients for Horner evaluation; their absolute sum is
1.03, so the monomial form loses nothing to cancellation.

Usage: python3 gen_erfc.py > gam_erfc.h
"""
import mpmath as mp

DEG = 25
NODES = 60


def q_of_u(u):
    t = (u + 1) / 2
    if t == 0:
        return 1 / (2 * mp.sqrt(mp.pi))
    a = 2 * (1 - t) / t
    return mp.erfc(a) * mp.exp(a * a) / t


def chebyshev(f, n):
    xs = [mp.cos(mp.pi * (k + mp.mpf(1) / 2) / n) for k in range(n)]
    fs = [f(x) for x in xs]
    c = [2 * mp.fsum(fs[k] * mp.cos(mp.pi * j * (k + mp.mpf(1) / 2) / n) for k in range(n)) / n
         for j in range(n)]
    c[0] /= 2
    return c


def to_monomial(c):
    n = len(c)
    T = [[mp.mpf(1)], [mp.mpf(0), mp.mpf(1)]]
    for k in range(2, n):
        a = [mp.mpf(0)] + [2 * x for x in T[k - 1]]
        b = T[k - 2] + [mp.mpf(0)] * (len(a) - len(T[k - 2]))
        T.append([x - y for x, y in zip(a, b)])
    m = [mp.mpf(0)] * n
    for k in range(n):
        for i, x in enumerate(T[k]):
            m[i] += c[k] * x
    return m


def main():
    mp.mp.dps = 40
    c = chebyshev(q_of_u, NODES)
    m = to_monomial(c[:DEG + 1])
    coef = ",\n".join("    %s" % repr(float(x)) for x in m)
    print("""// gam_erfc.h -- erfc(z) and exp(-z^2) in FP64 for the kinetic fluxes.
// Generated by gen_erfc.py (same directory); do not edit by hand.
//
// a = |z|, t = 2/(2+a), u = 2t-1:  erfc(a) = t * exp(-a^2) * Q(u) with Q a
// degree-%d polynomial (monomial coefficients below), erfc(-a) = 2 - erfc(a).
// exp(-a^2) is formed from the exact split a^2 = hi + lo (one fma), so the
// pair is accurate to about 8e-16 relative for |z| <= 20.  Host and device
// compile the same code (the host build is what the CPU test checks) but
// for the reciprocal, see gam_math.h.
#pragma once
#include "gam_math.h"

static constexpr double GAM_ERFC_Q[%d] = {
%s};

// Returns erfc(z); e receives exp(-z^2).
GAM_HD inline double gam_erfc_exp(double z, double &e)
{
    const double a = std::fabs(z);
    const double t = 2.0 * gam_rcp(2.0 + std::fmin(a, 1.0e300));
    const double u = std::fma(2.0, t, -1.0);
    double q = GAM_ERFC_Q[%d];
#pragma unroll
    for (int n = %d; n >= 0; n--) q = std::fma(q, u, GAM_ERFC_Q[n]);
    const double hi = a * a;
    // 0 for a = inf; a NaN goes through here into both results (the fmin above
    // and gam_exp_neg drop it)
    const double lo = hi >= 1.0e300 ? 0.0 : std::fma(a, a, -hi);
    e = gam_exp_neg(-hi);
    e = std::fma(-e, lo, e);
    const double r = t * e * q;
    return z < 0.0 ? 2.0 - r : r;
}
""" % (DEG, DEG + 1, coef, DEG, DEG - 1))


if __name__ == "__main__":
    main()
