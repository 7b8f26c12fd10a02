// tanh in FP64 for the activations of the networks.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

namespace ptmc {

// tanh x = t / (t + 2), t = e^(2x) - 1 = 2^k q + (2^k - 1), q = e^r - 1 by its
// Taylor series, 2x = k ln 2 + r (Cody-Waite).  r, q, t and t + 2 carry the
// rounding of their last operation (2^k q takes up to half of 2^k - 1 away at k
// = 1: 2.5 ulp without), so that the value is within 0.7 ulp, small x included.
// rcp(d): 1 / d for d in [2, 2^59) to a few ulp; the quotient's remainder is put
// back.
template <typename Rcp>
__host__ __device__ inline double net_tanh(double x, Rcp rcp)
{
    const double y = fmin(fabs(x), 20.0) * 2.0;
    const double kd = rint(y * 1.4426950408889634);
    const double rh = fma(-kd, 6.93147180369123816490e-01, y), c = kd * 1.90821492927058770002e-10;
    const double r = rh - c, rl = (rh - r) - c;
    double s = 1.0 / 87178291200.0;
    s = fma(s, r, 1.0 / 6227020800.0);
    s = fma(s, r, 1.0 / 479001600.0);
    s = fma(s, r, 1.0 / 39916800.0);
    s = fma(s, r, 1.0 / 3628800.0);
    s = fma(s, r, 1.0 / 362880.0);
    s = fma(s, r, 1.0 / 40320.0);
    s = fma(s, r, 1.0 / 5040.0);
    s = fma(s, r, 1.0 / 720.0);
    s = fma(s, r, 1.0 / 120.0);
    s = fma(s, r, 1.0 / 24.0);
    s = fma(s, r, 1.0 / 6.0);
    const double r2 = r * r, h = 0.5 * r2, q0 = r + h;
    const double m = fma(r2 * r, s, (h - (q0 - r)) + fma(0.5, fma(r, r, -r2), rl));
    const double q = q0 + m, ql = m - (q - q0);
    const double p = ldexp(1.0, (int)kd), a = p - 1.0, b = p * q;
    const double t = a + b, tl = fma(p, ql, b - (t - a));  // |b| < a, or a = 0
    const double d = t + 2.0, dl = t >= 2.0 ? 2.0 - (d - t) : t - (d - 2.0);
    const double i = rcp(d), v = t * i;
    const double w = fma(fma(-v, d, t) + fma(-v, dl + tl, tl), i, v);
    return x != x ? x : copysign(w, x);
}

}  // namespace ptmc
