/* hh_group6.h -- one 6-d CR3BP trajectory per aligned group of 8 or 16 lanes,
 * one component per lane: lanes 0..2 of the group hold x, y, z, lanes 4..6
 * vx, vy, vz; lanes 3 and 7 hold 0 and help, lanes 8..15 (of the 16-lane form)
 * are idle.  Every per-component expression is Lane6's (rhs6,
 * dop853_attempt, dense output: dynamics/rtbp.py:30-74, integrators/rk.py:
 * 1636-1699, 1836-1874, 2457-2484), so results are bit-identical; the group
 * shares out what Lane6 does serially:
 *   - the two primaries: the position lanes form r1^3 and the three
 *     quotients of the first primary, the velocity lanes r2^3 and those of
 *     the second, one quotient a lane; the first's move to the velocity
 *     lanes with one DPP move per dword;
 *   - the error-norm divisions (one pair per lane) and the three pow calls
 *     of the step controller (lanes 0..2).
 * Sums over the six components are formed in Lane6's order (from 0.0, d =
 * 0..5).
 *
 * What bounds it is one wave's instruction stream and the latency of the
 * dependent chain through a stage (position broadcast, square root, cube,
 * quotient, stage sum), so an attempt runs branch-free from end to end on the
 * unscaled forms of hh_fast.h and lanes exchange values by DPP, not through
 * LDS (about 7 cycles a dependent FP64 operation, 14 a DPP move, 61 a
 * ds_swizzle, 67 an IEEE division, 104 a square root).  An attempt that
 * leaves their range is evaluated again with the general forms.
 *
 * 8 or 16 lanes: in a group of 16 lanes (a DPP row) a broadcast is one
 * row_newbcast move instead of four moves and coefficients come from the row
 * (RowTab), but a wave holds four trajectories instead of eight.
 *
 * Measured against the form before (components in lanes 0..5, LDS swizzles,
 * IEEE divisions and branches): 1,024 x 2,000 RK8 steps 7.29 -> 3.73 ms (150
 * ns a stage, about 74 instructions of a wave alone on its SIMD), 500
 * manifold arcs 5.31 -> 3.36 ms (1.28 with group6_points), 32,768 event
 * searches 0.72 -> 0.59 ms.
 */
#ifndef HH_GROUP6_H
#define HH_GROUP6_H

#include "hh_device.h"

namespace hh {

__device__ __forceinline__ double bperm(double v, int addr) {
    const int lo = __builtin_amdgcn_ds_bpermute(addr, __double2loint(v));
    const int hi = __builtin_amdgcn_ds_bpermute(addr, __double2hiint(v));
    return __hiloint2double(hi, lo);
}

/* v, negated where s has bit 31 set */
__device__ __forceinline__ double xor_sign(double v, unsigned s) {
    return __hiloint2double((int)((unsigned)__double2hiint(v) ^ s), __double2loint(v));
}

/* lane K (0..15) of each row, in every lane of the row */
template <int K>
__device__ __forceinline__ double row_bcast(double v) {
    return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + K, 0xF, 0xF, true);
}

/* row_bcast of a lane that is a constant once loops are unrolled */
__device__ __forceinline__ double row_bcast_at(double v, int k) {
    switch (k) {
        case 0: return row_bcast<0>(v);
        case 1: return row_bcast<1>(v);
        case 2: return row_bcast<2>(v);
        case 3: return row_bcast<3>(v);
        case 4: return row_bcast<4>(v);
        case 5: return row_bcast<5>(v);
        case 6: return row_bcast<6>(v);
        case 7: return row_bcast<7>(v);
        case 8: return row_bcast<8>(v);
        case 9: return row_bcast<9>(v);
        case 10: return row_bcast<10>(v);
        case 11: return row_bcast<11>(v);
        case 12: return row_bcast<12>(v);
        case 13: return row_bcast<13>(v);
        case 14: return row_bcast<14>(v);
        default: return row_bcast<15>(v);
    }
}

/* Coefficients of a tableau spread over the lanes of each row: entry n lies in
 * lane n % 16 of register n / 16, and a product h * a_n is formed for sixteen
 * coefficients by one multiplication.  A stage's term then takes a broadcast,
 * a product and a sum, where a coefficient written into the instructions takes
 * two scalar moves and the product h * a as well: a wave that runs alone on
 * its SIMD issues one instruction at a time, scalar ones included.        */
template <int N>
struct RowTab {
    static constexpr int R = (N + 15) / 16;
    double c[R];
    __device__ __forceinline__ void put(int n, double a, int lane) {
        if (n % 16 == 0) c[n / 16] = 0.0;
        c[n / 16] = ((lane & 15) == n % 16) ? a : c[n / 16];
    }
    __device__ __forceinline__ double at(int n) const { return row_bcast_at(c[n / 16], n % 16); }
    __device__ __forceinline__ RowTab times(double h) const {
        RowTab t;
#pragma unroll
        for (int r = 0; r < R; ++r) t.c[r] = h * c[r];
        return t;
    }
};

/* DOP853's non-zero coefficients in the order an attempt takes them: 50 of the
 * stages, 8 of the solution; 8 and 8 of the error estimators               */
struct DopRow {
    RowTab<58> a;
    RowTab<16> e;
    __device__ __forceinline__ void fill(int lane) {
        int n = 0;
#pragma unroll
        for (int i = 1; i < DOP_S; ++i)
#pragma unroll
            for (int j = 0; j < i; ++j)
                if (HH_DOP_A[i][j] != 0.0) a.put(n++, HH_DOP_A[i][j], lane);
#pragma unroll
        for (int j = 0; j < DOP_S; ++j)
            if (HH_DOP_B[j] != 0.0) a.put(n++, HH_DOP_B[j], lane);
        n = 0;
#pragma unroll
        for (int j = 0; j < DOP_K; ++j)
            if (HH_DOP_E5[j] != 0.0) e.put(n++, HH_DOP_E5[j], lane);
#pragma unroll
        for (int j = 0; j < DOP_K; ++j)
            if (HH_DOP_E3[j] != 0.0) e.put(n++, HH_DOP_E3[j], lane);
    }
};

/* the same of a fixed-step tableau */
template <class M>
struct RkRow {
    static constexpr int N = M::ORDER == 4 ? 7 : (M::ORDER == 6 ? 25 : 68);
    RowTab<N> a;
    __device__ __forceinline__ void fill(int lane) {
        int n = 0;
#pragma unroll
        for (int i = 1; i < M::S; ++i)
#pragma unroll
            for (int j = 0; j < i; ++j)
                if (M::a(i, j) != 0.0) a.put(n++, M::a(i, j), lane);
#pragma unroll
        for (int j = 0; j < M::S; ++j)
            if (M::b(j) != 0.0) a.put(n++, M::b(j), lane);
    }
};

/* DPP move CTRL into the lanes of BANKS (banks of four lanes of each row);
 * the other lanes keep `old`                                              */
template <int CTRL, int BANKS>
__device__ __forceinline__ double dpp_into(double old, double v) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, 0xF,
                                               BANKS, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, 0xF,
                                               BANKS, false);
    return __hiloint2double(hi, lo);
}

/* lane i takes lane i - 4 of its row, 0 in lanes 0..3 */
__device__ __forceinline__ double row_shr4_zero(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x114, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x114, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

constexpr int DPP_SHL4 = 0x104, DPP_SHR4 = 0x114;   /* row shifts: lane i takes i + 4, i - 4 */
constexpr int BANKS_POS = 0x5, BANKS_VEL = 0xA;     /* banks 0 and 2, banks 1 and 3          */
constexpr int QUAD_SWAP01 = 0xF1;                   /* quad_perm [1, 0, 3, 3]                */

template <int LANES_>
struct Lanes6 {
    static_assert(LANES_ == 8 || LANES_ == 16, "a group is 8 or 16 lanes");
    static constexpr int LANES = LANES_;
    double mu, one_mu;
    int d;                    /* component 0..5 of this lane, 6 or 7 in the others */
    bool act;                 /* this lane holds a component                      */
    bool vel;                 /* a velocity lane's quad                           */
    bool xy;                  /* lane of vx or vy                                 */
    int base;                 /* the group's first lane as a bpermute byte address */
    double cl;                /* mu (position lanes) or -one_mu (velocity lanes)  */
    double b1, b2;            /* (w + b1) + b2: the distance component of the
                                 lane's quotient as the field writes it            */
    double c1;                /* the quotient's mass, 0 in lanes without one       */
    double c2;                /* factor of the velocity entry in the lane's row    */
    unsigned sign;            /* bit 31: this lane's derivative is negated         */
    const PowTab* pt;         /* hh_pow's tables (an LDS copy)                     */
    int lane;
    DopRow tab;               /* filled for the 16-lane form's attempts (dop_setup) */

    /* before the first attempt */
    __device__ __forceinline__ void dop_setup() {
        if constexpr (LANES == 16) tab.fill(lane);
    }

    __device__ __forceinline__ void setup(int lane_, double mu_, int fwd, unsigned long long flip,
                                          const PowTab* pt_) {
        lane = lane_;
        pt = pt_;
        const int l = lane & (LANES - 1);
        act = l < 7 && l != 3;
        vel = (l & 4) != 0;
        xy = l == 4 || l == 5;
        d = l < 3 ? l : (l == 3 ? 6 : (l < 7 ? l - 1 : 7));
        base = (lane & ~(LANES - 1)) << 2;
        mu = mu_;
        one_mu = 1.0 - mu_;
        cl = vel ? -one_mu : mu_;
        /* adding -0.0 leaves every value, signed zeros too, as it is */
        b1 = l == 0 ? mu_ : (l == 4 ? -1.0 : -0.0);
        b2 = l == 4 ? mu_ : -0.0;
        c1 = act ? (vel ? mu_ : one_mu) : 0.0;
        c2 = l < 3 ? 1.0 : (l == 4 ? 2.0 : (l == 5 ? -2.0 : (l == 6 ? -1.0 : 0.0)));
        sign = (act && fwd == -1 && ((flip >> d) & 1ULL)) ? 1u << 31 : 0u;
    }

    /* byte address of the lane of this group that holds component k */
    __device__ __forceinline__ int comp_addr(int k) const {
        return base + ((k < 3 ? k : k + 1) << 2);
    }

    /* component K of this lane's group */
    template <int K>
    __device__ __forceinline__ double get(double v) const {
        constexpr int L = K < 3 ? K : K + 1;
        if constexpr (LANES == 16) {
            return row_bcast<L>(v);
        } else if constexpr (L < 4) {
            /* the quad's lane L, then from the lower quad into the upper one */
            const double t = quad_get<L * 0x55>(v);
            return dpp_into<DPP_SHR4, BANKS_VEL>(t, t);
        } else {
            const double t = quad_get<(L - 4) * 0x55>(v);
            return dpp_into<DPP_SHL4, BANKS_POS>(t, t);
        }
    }

    /* derivative of this lane's component, v = its stage component:
     * rows 0..2  the velocity entry
     * row 3      ((2 vy + x) - (one_mu xm)/r1c) - (mu xm1)/r2c
     * row 4      ((-2 vx + y) - (one_mu y)/r1c) - (mu y)/r2c
     * row 5      ((-one_mu) z)/r1c - (mu z)/r2c
     * all as ((c2 pv + hz) - q1) - q2, with zeros of the sign that leaves
     * the other terms as they are where a row has no such term             */
    template <bool FAST>
    __device__ __forceinline__ double rhs_form(double v, FastChk& c) const {
        const double x = get<0>(v);
        const double y = get<1>(v);
        const double z = get<2>(v);
        /* the velocity entry of this lane's row: lanes 0..2 take lanes 4..6,
         * lane 4 vy, lane 5 vx, lane 6 lane 7's zero                       */
        const double pv = dpp_into<DPP_SHL4, BANKS_POS>(quad_get<QUAD_SWAP01>(v), v);
        /* the position entry of lanes 0..2 and 4..6 */
        const double w = dpp_into<DPP_SHR4, BANKS_VEL>(v, v);
        const double u = (w + b1) + b2;
        const double num = c1 * u;
        const double xo = x + cl;
        const double P = (xo * xo + y * y) + z * z;
        double q;
        if constexpr (FAST) {
            c.dist(P);
            c.num(u);
            double h;
            const double r = fast_sqrt(P, h);
            const double rc = r * (r * r);
            q = fast_div(num, rc, rcp_step(rc, (8.0 * h) * (h * h)));
        } else {
            const double r = __builtin_sqrt(P);
            q = num / (r * (r * r));
        }
        /* the first primary's quotient, 0 in the position lanes (of a 16-lane
         * group, which lie at the row's start, by the shift's zero fill)    */
        double q1;
        if constexpr (LANES == 16) q1 = row_shr4_zero(q);
        else q1 = dpp_into<DPP_SHR4, BANKS_VEL>(0.0, q);
        const double q2 = vel ? q : 0.0;
        const double head = c2 * pv + (xy ? w : -0.0);
        double o = (head - q1) - q2;
        if constexpr (!FAST) o = act ? o : 0.0;   /* 0/0 and the like in idle lanes */
        return xor_sign(o, sign);
    }

    __device__ __forceinline__ double rhs(double v) const {
        FastChk c;
        c.num(c1);
        const double o = rhs_form<true>(v, c);
        if (__builtin_expect(__any(c.outside()), 0)) return rhs_form<false>(v, c);
        return o;
    }

    /* sum over the group's six components of this lane's term, from 0.0 in
     * component order (all lanes of the group get the sum)                  */
    __device__ __forceinline__ double sum6(double term) const {
        const double g0 = get<0>(term);
        const double g1 = get<1>(term);
        const double g2 = get<2>(term);
        const double g3 = get<3>(term);
        const double g4 = get<4>(term);
        const double g5 = get<5>(term);
        return (((((0.0 + g0) + g1) + g2) + g3) + g4) + g5;
    }

    /* initial_step (rk.py:2443-2448) */
    __device__ __forceinline__ double initial_step(double y, double f0, double rtol, double atol,
                                                   double min_step, double max_step) const {
        const double sc = atol + rtol * __builtin_fabs(y);
        const double a = y / sc;
        const double b = f0 / sc;
        const double s0 = sum6(a * a);
        const double s1 = sum6(b * b);
        const double sn = __builtin_sqrt(6.0);
        const double d0 = __builtin_sqrt(s0) / sn;
        const double d1 = __builtin_sqrt(s1) / sn;
        return select_initial_step(d0, d1, min_step, max_step);
    }

    /* dop853_attempt, one component per lane */
    template <bool FAST>
    __device__ __forceinline__ double attempt_form(double y, double (&k)[DOP_K], double h,
                                                   double rtol, double atol, double& yh,
                                                   FastChk& c) const {
        /* h * a for every coefficient: from the row tables, or formed in place */
        RowTab<58> ha;
        if constexpr (LANES == 16) ha = tab.a.times(h);
        int n = 0;
#pragma unroll
        for (int i = 1; i < DOP_S; ++i) {
            double ys = y;
#pragma unroll
            for (int j = 0; j < i; ++j) {
                const double a = HH_DOP_A[i][j];
                if (a != 0.0) ys = ys + (LANES == 16 ? ha.at(n++) : h * a) * k[j];
            }
            k[i] = rhs_form<FAST>(ys, c);
        }
        yh = y;
#pragma unroll
        for (int j = 0; j < DOP_S; ++j) {
            const double bb = HH_DOP_B[j];
            if (bb != 0.0) yh = yh + (LANES == 16 ? ha.at(n++) : h * bb) * k[j];
        }
        k[DOP_S] = rhs_form<FAST>(yh, c);
        double e5 = 0.0, e3 = 0.0;
        n = 0;
#pragma unroll
        for (int j = 0; j < DOP_K; ++j) {
            const double c5 = HH_DOP_E5[j];
            if (c5 != 0.0) e5 = e5 + (LANES == 16 ? tab.e.at(n++) : c5) * k[j];
        }
#pragma unroll
        for (int j = 0; j < DOP_K; ++j) {
            const double c3 = HH_DOP_E3[j];
            if (c3 != 0.0) e3 = e3 + (LANES == 16 ? tab.e.at(n++) : c3) * k[j];
        }
        const double m = np_max(__builtin_fabs(y), __builtin_fabs(yh));
        const double sc = act ? atol + rtol * m : 1.0;
        const double n5 = act ? e5 * h : 0.0;
        const double n3 = act ? e3 * h : 0.0;
        double q5, q3;
        if constexpr (FAST) {
            c.scale(sc);
            c.num(n5);
            c.num(n3);
            const double r = fast_rcp(sc);
            q5 = fast_div(n5, sc, r);
            q3 = fast_div(n3, sc, r);
        } else {
            q5 = n5 / sc;
            q3 = n3 / sc;
        }
        const double s5 = sum6(q5 * q5);
        const double s3 = sum6(q3 * q3);
        const double denom = (s5 + 0.01 * s3) * 6.0;
        const double top = __builtin_fabs(h) * s5;
        if constexpr (FAST) {
            c.scale(denom);
            c.num(top);
            double g;
            const double r = fast_sqrt(denom, g);
            return fast_div(top, r, rcp_step(r, g + g));
        } else {
            if (s5 == 0.0 && s3 == 0.0) return 0.0;
            return top / __builtin_sqrt(denom);
        }
    }

    __device__ __forceinline__ double attempt(double y, double (&k)[DOP_K], double h, double rtol,
                                              double atol, double& yh) const {
        FastChk c;
        c.num(c1);
        double err = attempt_form<true>(y, k, h, rtol, atol, yh, c);
        if (__builtin_expect(__any(c.outside() || !(err < __builtin_inf())), 0)) {
            /* an h of its own: the products h*a above are not kept for this */
            asm volatile("" : "+v"(h));
            err = attempt_form<false>(y, k, h, rtol, atol, yh, c);
        }
        return err;
    }

    /* pi_accept_factor / pi_reject_factor with their pow calls in lanes 0..2 */
    __device__ __forceinline__ void step_factors(double err, double err_prev, double& f_acc,
                                                 double& f_rej) const {
        const double beta = 1.0 / (8.0 + 1.0);
        const double alpha = 0.4 * beta;
        const double err_exp = 1.0 / 8.0;
        const double px = (d == 1) ? err_prev : err;
        const double pe = (d == 0) ? -beta : ((d == 1) ? alpha : -err_exp);
        step_factors_from(pt, err, err_prev, px, pe, [this](double v, int i) {
            return i == 0 ? get<0>(v) : (i == 1 ? get<1>(v) : get<2>(v));
        }, f_acc, f_rej);
    }

    /* the three extension stages and the seven interpolant rows of this
     * lane's component (rk.py:1836-1874)                                    */
    __device__ __forceinline__ void dense_rows(double y_old, double y_new, const double (&k)[DOP_K],
                                               double hs, double (&row)[DOP_P]) const {
        double kx[DOP_SX - DOP_K];
#pragma unroll
        for (int sr = DOP_K; sr < DOP_SX; ++sr) {
            double acc = 0.0;
#pragma unroll
            for (int r = 0; r < sr; ++r) {
                const double a = HH_DOP_A[sr][r];
                if (a != 0.0) acc = acc + a * (r < DOP_K ? k[r] : kx[r - DOP_K]);
            }
            kx[sr - DOP_K] = rhs(y_old + hs * acc);
        }
        const double dy = y_new - y_old;
        row[0] = dy;
        row[1] = hs * k[0] - dy;
        row[2] = 2.0 * dy - hs * (k[DOP_S] + k[0]);
#pragma unroll
        for (int i = 3; i < DOP_P; ++i) {
            double acc = 0.0;
#pragma unroll
            for (int r = 0; r < DOP_SX; ++r) {
                const double c = HH_DOP_D[i - 3][r];
                if (c != 0.0) acc = acc + c * (r < DOP_K ? k[r] : kx[r - DOP_K]);
            }
            row[i] = hs * acc;
        }
    }
};

using Group6 = Lanes6<8>;
using Row6 = Lanes6<16>;

/* rk_step (rk.py:154-215) for this lane's component; k0 receives the first
 * stage (the derivative at the step's start)                              */
template <class M, bool FAST, class P>
__device__ __forceinline__ double rk_step_form(const P& p, const RkRow<M>& tab, double y, double h,
                                               double& k0, FastChk& c) {
    constexpr bool ROW = P::LANES == 16;
    RowTab<RkRow<M>::N> ha;
    if constexpr (ROW) ha = tab.a.times(h);
    int n = 0;
    double k[M::S];
    k[0] = p.template rhs_form<FAST>(y, c);
    k0 = k[0];
#pragma unroll
    for (int i = 1; i < M::S; ++i) {
        double ys = y;
#pragma unroll
        for (int j = 0; j < i; ++j) {
            const double a = M::a(i, j);
            if (a != 0.0) ys = ys + (ROW ? ha.at(n++) : h * a) * k[j];
        }
        k[i] = p.template rhs_form<FAST>(ys, c);
    }
#pragma unroll
    for (int j = 0; j < M::S; ++j) {
        const double b = M::b(j);
        if (b != 0.0) y = y + (ROW ? ha.at(n++) : h * b) * k[j];
    }
    return y;
}

template <class M, class P>
__device__ __forceinline__ void rk_step_group(const P& p, const RkRow<M>& tab, double& y, double h,
                                              double& k0) {
    FastChk c;
    c.num(p.c1);
    double yn = rk_step_form<M, true>(p, tab, y, h, k0, c);
    if (__builtin_expect(__any(c.outside()), 0)) {
        asm volatile("" : "+v"(h));
        yn = rk_step_form<M, false>(p, tab, y, h, k0, c);
    }
    y = yn;
}

/* dense_value of one component from its rows (rk.py:1989-2003) */
__device__ __forceinline__ double dense_from_rows(const double (&row)[DOP_P], double y_old,
                                                  double x) {
    const double omx = 1.0 - x;
    double v = 0.0;
#pragma unroll
    for (int i = DOP_P - 1; i >= 0; --i) {
        v = v + row[i];
        v = v * (((DOP_P - 1 - i) % 2 == 0) ? x : omx);
    }
    return v + y_old;
}

}  // namespace hh

#endif /* HH_GROUP6_H */
