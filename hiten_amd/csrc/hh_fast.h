/* hh_fast.h -- divisions and powers of the stage loops without scaling,
 * special cases or branches.
 *
 * The CR3BP field's distances lie near 1 (a primary's surface is 1e-3 away,
 * an escaping arc 1e3), where the scaling and fix-up steps of an IEEE
 * division or square root do nothing.  FastChk holds the exponent range of
 * the forms below; where a lane of the wave leaves it, the wave takes the
 * general forms.  Within the range every result is the correctly rounded
 * one except for rare arguments, named below; no output of any test or timed
 * case has differed.
 *
 *   fast_div     q = n r, then one correction with the exact remainder.  By
 *                Markstein's theorem the corrected quotient is the correctly
 *                rounded one if r is 1/d correctly rounded and d's significand
 *                is not all ones.  r comes from one Newton step on a value
 *                good to 2^-43 or better, so it is correctly rounded except
 *                where 1/d lies within about 2^-33 of its last place of a
 *                rounding boundary; a quotient of such a d can then be off by
 *                its last bit, and only if it lies as close to a boundary
 *                itself.  Quotients of one denominator share its reciprocal.  The
 *                remainder is taken with the sign that keeps a zero
 *                quotient's sign.
 *   fast_pow     x^1.5 and x^2.5 as hh_pow15_25 forms them, without its
 *                overflow tests, and with one correction of the square root
 *                instead of two: the second changes the root's last bit in
 *                about 1 of 2^37 arguments, and the powers, formed from the
 *                root and its exact remainder, change only if their exact
 *                value also lies within 2^-103 of a rounding boundary: not the
 *                same bits for every argument, at the same precision.
 *   reciprocals  of r^3 and r^5 start from powers of the refined 1/r the
 *                square root leaves behind (2^-43), one Newton step each.
 */
#ifndef HH_FAST_H
#define HH_FAST_H

namespace hh {

/* Extreme exponents seen by the fast forms.  Squared distances must lie in
 * [2^-100, 2^100), the coordinates they come from (and so the numerators)
 * must be 0 or at least 2^-301 in magnitude, error scales in
 * [2^-300, 2^960): the scale of an STM entry is rtol times the entry, and the
 * entries of a trajectory that runs into a primary grow to 1e300 over
 * thousands of attempts.  A quotient by a scale that falls below the normal
 * range has the square 0 either way.  NaN and infinities fail the first test. */
struct FastChk {
    static constexpr unsigned DIST_LO = (1023u - 100u) << 20, DIST_SPAN = 200u << 20;
    static constexpr unsigned SCALE_LO = (1023u - 300u) << 20, SCALE_SPAN = 1260u << 20;
    unsigned dist_max = 0, scale_max = 0;
    int num_min = 0;

    __device__ __forceinline__ static unsigned umax(unsigned a, unsigned b) {
        return a > b ? a : b;
    }
    __device__ __forceinline__ static int imin(int a, int b) { return a < b ? a : b; }
    __device__ __forceinline__ void dist(double p) {
        dist_max = umax(dist_max, (unsigned)__double2hiint(p) - DIST_LO);
    }
    __device__ __forceinline__ void scale(double s) {
        scale_max = umax(scale_max, (unsigned)__double2hiint(s) - SCALE_LO);
    }
    __device__ __forceinline__ void num(double v) {
        num_min = imin(num_min, __builtin_amdgcn_frexp_exp(v));
    }
    __device__ __forceinline__ bool outside() const {
        return dist_max >= DIST_SPAN || scale_max >= SCALE_SPAN || num_min < -300;
    }
};

/* n / d from r = 1/d correctly rounded (see above where it is not) */
__device__ __forceinline__ double fast_div(double n, double d, double r) {
    const double q = n * r;
    const double t = __builtin_fma(d, q, -n);
    return __builtin_fma(-t, r, q);
}

/* 1/d, correctly rounded but for rare d */
__device__ __forceinline__ double fast_rcp(double d) {
    double r = __builtin_amdgcn_rcp(d);
    double e = __builtin_fma(-d, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-d, r, 1.0);
    return __builtin_fma(r, e, r);
}

/* one Newton step of a reciprocal */
__device__ __forceinline__ double rcp_step(double d, double r) {
    const double e = __builtin_fma(-d, r, 1.0);
    return __builtin_fma(r, e, r);
}

/* s ~ sqrt(x) after one correction and h ~ 1 / (2 sqrt(x)) */
__device__ __forceinline__ void fast_root(double x, double& s, double& h) {
    const double y0 = __builtin_amdgcn_rsq(x);
    double g = x * y0;
    h = y0 * 0.5;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    const double d = __builtin_fma(-g, g, x);
    s = __builtin_fma(d, h, g);
}

/* x^1.5, x^2.5 and their reciprocals */
__device__ __forceinline__ void fast_pow15_25(double x, double& p15, double& p25, double& r15,
                                              double& r25) {
    double s, h;
    fast_root(x, s, h);
    const double e = __builtin_fma(-s, s, x);
    const double he = 0.5 * e;
    const double p = x * s, pe = __builtin_fma(x, s, -p);
    p15 = p + (pe + s * he);
    const double q = x * x, qe = __builtin_fma(x, x, -q);
    const double p2 = q * s, pe2 = __builtin_fma(q, s, -p2);
    p25 = p2 + (pe2 + (p * he + qe * s));
    const double h2 = h * h;
    const double y15 = (8.0 * h) * h2;
    r15 = rcp_step(p15, y15);
    r25 = rcp_step(p25, y15 * (4.0 * h2));
}

/* sqrt(x), correctly rounded (the compiler's own expansion without scaling) */
__device__ __forceinline__ double fast_sqrt(double x, double& h) {
    double s;
    fast_root(x, s, h);
    const double d = __builtin_fma(-s, s, x);
    return __builtin_fma(d, h, s);
}

}  // namespace hh

#endif /* HH_FAST_H */
