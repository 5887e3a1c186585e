/* hh_wave.h -- one 42-d variational trajectory per wave (64 lanes), and the
 * lane layout it shares with the two-wave form (hh_pair.h).
 *
 * Lanes 0..15 (the wave's first DPP row) hold the state: x, y, z in lanes
 * 0..2, vx, vy, vz in lanes 4..6, the constant 1 in lane 3, 0 in lane 7.
 * Lanes 16 + 8 j .. hold STM column j (j = 0..5) the same way: entries 0..2,
 * 0, entries 3..5, 0.  Every per-component expression is Lane42's (and so the
 * reference's, dynamics/rtbp.py:115-141, 219-242 and integrators/rk.py:
 * 1636-1699, 1836-1874, 2457-2484), evaluated one component per lane instead
 * of six, so results are bit-identical to Lane42's:
 *   - the twelve quotients of the variational field are formed one per lane
 *     in lanes 4..15, each lane raising its own primary's distance to the
 *     power its quotient needs;
 *   - the state's rows take theirs by DPP; the columns read the other six and
 *     the coordinates from LDS, where the first row writes them;
 *   - the three pow calls of the step-size controller run in lanes 0..2;
 *   - the error-norm block sums are formed in Lane42's in-lane order and
 *     combined by the same block tree.
 *
 * What bounds a trajectory that runs alone on its SIMD is the length of its
 * wave's instruction stream (about 5 cycles an instruction) and the latency
 * of the state's chain, so an attempt is branch-free on the unscaled forms of
 * hh_fast.h and is evaluated again with the general ones if a value leaves
 * their range.
 */
#ifndef HH_WAVE_H
#define HH_WAVE_H

#include "hh_device.h"
#include "hh_group6.h"

namespace hh {

/* value of a double in lane l (l wave-uniform) */
__device__ __forceinline__ double rlane(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

/* What the state's row hands to the columns in one right-hand side: every
 * lane's quotient and distance component (those of lanes 4..15 are read).
 * Lanes whose row of F has no entries read a record of zeros.             */
struct StageRec {
    double q[64], u[64];
};

/* Keeps the compiler to the order in which LDS accesses are written: the one-wave
 * form issues the loads of its record before the state row's arithmetic, which
 * hides them (200 corrections 3.75 ms, 3.83 without).                       */
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

/* Lane layout, constants and the two halves of the field */
struct Var42 {
    double mu, mu2;
    int lane;
    int l;                    /* lane & 7                                        */
    int d;                    /* entry 0..5 of the block, 6 or 7 without one      */
    bool act;                 /* holds a component                               */
    bool st;                  /* in the state's row                              */
    bool vel;                 /* in a quad of velocity entries                   */
    bool xy;                  /* lane of vx or vy of the state                   */
    bool p5;                  /* this lane's quotient divides by r^5             */
    bool quot;                /* holds a quotient (lanes 4..15)                  */
    double cl;                /* x + cl: the lane's primary's x distance          */
    double b;                 /* w + b: the lane's distance component             */
    double cm, ca;            /* numerator cm (w + b) + ca                       */
    double cr;                /* 8 or, for a quotient by r^5, 32                 */
    double ka, kb;            /* mu2, mu in the state's velocity lanes, else 0   */
    double c2;                /* factor of the velocity entry: state rows         */
    double e2;                /* and column rows                                 */
    double diag;              /* 1, 1, 0: the constant of the Hessian's diagonal */
    unsigned sign;            /* bit 31: this lane's derivative is negated       */
    const PowTab* pt;         /* hh_pow's tables (an LDS copy)                   */
    DopRow tab;               /* tableau coefficients, one copy per row           */

    __device__ __forceinline__ void setup(int lane_, double mu_, int fwd,
                                          unsigned long long flip, const PowTab* pt_) {
        lane = lane_;
        pt = pt_;
        l = lane & 7;
        st = lane < 16;
        act = l != 3 && l != 7 && (lane < 8 || !st);
        vel = (l & 4) != 0;
        d = l < 3 ? l : (l == 3 ? 6 : (l < 7 ? l - 1 : 7));
        xy = lane == 4 || lane == 5;
        quot = st && lane >= 4;
        p5 = lane >= 8 && lane < 12;
        mu = mu_;
        mu2 = 1.0 - mu_;
        const bool second = lane >= 10 && st;
        cl = second ? -mu2 : mu_;
        /* lanes   4 xm/r3   5 y/r3        6 z/r3   7 mu2/r3
         *         8 mu2/r5  9 (mu2 xm)/r5 10 mu/R5 11 (mu xr)/R5
         *        12 xr/R3  13 y/R3       14 z/R3  15 mu/R3
         * from w = x, y, z, 1 in lanes 4..7 and 12..15, x in lanes 8..11;
         * adding -0.0 leaves every value, signed zeros too, as it is       */
        b = (lane == 4 || lane == 9) ? mu_ : ((lane == 11 || lane == 12) ? -mu2 : -0.0);
        const double m = second ? mu_ : mu2;
        cm = (lane == 7 || lane == 9 || lane == 11 || lane == 15)
                 ? m : ((quot && lane != 8 && lane != 10) ? 1.0 : 0.0);
        cr = p5 ? 32.0 : 8.0;
        ca = (lane == 8 || lane == 10) ? m : (lane < 4 ? 0.0 : -0.0);
        const bool sv = lane >= 4 && lane < 7;
        ka = sv ? mu2 : 0.0;
        kb = sv ? mu_ : 0.0;
        /* lane 6 multiplies lane 7's zero: -0.0, which adds nothing        */
        c2 = lane < 4 ? 1.0 : (lane == 4 ? 2.0 : (lane == 5 ? -2.0 : (lane == 6 ? -1.0 : 0.0)));
        e2 = l < 3 ? 1.0 : (l == 4 ? 2.0 : (l == 5 ? -2.0 : 0.0));
        diag = (l == 4 || l == 5) ? 1.0 : 0.0;
        sign = (act && fwd == -1 && ((flip >> comp()) & 1ULL)) ? 1u << 31 : 0u;
        tab.fill(lane);
    }

    /* Lane42's block (0 the state, 1..6 the columns) and the component's place
     * in the 42-vector, of a lane that holds one                            */
    __device__ __forceinline__ int block() const { return st ? 0 : (lane >> 3) - 1; }
    __device__ __forceinline__ int comp() const { return comp42(block(), d < 6 ? d : 0); }
    /* what lanes without a component hold */
    __device__ __forceinline__ double idle() const { return lane == 3 ? 1.0 : 0.0; }

    /* the velocity entry of this lane's row: lanes 0..2 of a half row take
     * lanes 4..6, lane 4 lane 5, lane 5 lane 4, lane 6 lane 7's zero        */
    __device__ __forceinline__ double vel_entry(double v) const {
        return dpp_into<DPP_SHL4, BANKS_POS>(quad_get<QUAD_SWAP01>(v), v);
    }

    /* This lane's quotient of the field, from the state in lanes 0..7 of v;
     * w and u as in setup's table; pos is any value that is not negative.   */
    template <bool FAST>
    __device__ __forceinline__ double quotient(double v, FastChk& c, double& w, double& u,
                                               double& pos) const {
        const double x = row_bcast<0>(v);
        const double y = row_bcast<1>(v);
        const double z = row_bcast<2>(v);
        w = dpp_into<0x11C, 0x8>(dpp_into<DPP_SHR4, 0x2>(x, v), v);   /* row_shr 12, 4 */
        u = w + b;
        const double num = __builtin_fma(cm, u, ca);
        const double xo = x + cl;
        const double P = (xo * xo + y * y) + z * z;
        if constexpr (FAST) {
            c.dist(P);
            c.num(u);
            /* fast_pow15_25 for the one power this lane needs:
             * base * s with base = P or P^2 (= base + be), t = s or P s      */
            double s, h;
            fast_root(P, s, h);
            const double e = __builtin_fma(-s, s, P);
            const double he = 0.5 * e;
            /* a factor P or 1 instead of a choice between powers: exact where it
             * is 1, and eight instructions of 88 fewer with the choice of the
             * scale in cr and pos in state_row (0.640 -> 0.606 ms a trajectory
             * on a pair, 0.902 -> 0.854 ms on one wave)                        */
            const double m = p5 ? P : 1.0;
            const double base = m * P, be = __builtin_fma(m, P, -base);
            const double t = m * s;
            const double p = base * s, pe = __builtin_fma(base, s, -p);
            const double D = p + (pe + (t * he + be * s));
            const double h2 = h * h;
            const double R = rcp_step(D, ((cr * h) * h2) * (p5 ? h2 : 1.0));
            pos = h2;
            return fast_div(num, D, R);
        } else {
            double P3, P5;
            hh_dev_pow15_25(P, &P3, &P5);
            const double q = num / (p5 ? P5 : P3);
            pos = 0.0;
            return quot ? q : 0.0;
        }
    }

    /* derivative of this lane's state component (rtbp.py:233-242):
     * rows 0..2  the velocity entry
     * row 3      ((x - mu2 xm/r3) - mu xr/R3) + 2 vy
     * row 4      ((y - mu2 y/r3) - mu y/R3) - 2 vx
     * row 5      (-mu2 z/r3) - mu z/R3
     * all as ((w0 - ka q) - kb q2) + c2 pv, where lanes with kb = 0 may have
     * any q2 that is not negative                                           */
    template <bool FAST>
    __device__ __forceinline__ double state_row(double v, double q, double w, double pos) const {
        const double pv = vel_entry(v);
        const double q2 = dpp_into<0x108, 0x2>(pos, q);   /* row_shl 8 into lanes 4..7 */
        const double w0 = xy ? w : -0.0;
        const double o = ((w0 - ka * q) - kb * q2) + c2 * pv;
        if constexpr (FAST) return o;
        return (act && st) ? o : 0.0;
    }

    /* What a column's lane reads of a stage's record: by value, since
     * column_row holds them in registers from one point on                  */
    struct Entries {
        double Q6, Q7, Q8, Q9, Q10, Q11, y, z, pa, pb;
    };
    __device__ __forceinline__ Entries entries(const StageRec& r) const {
        const int row = vel ? (l & 3) : 0;
        return {r.q[8], r.q[10], r.q[7], r.q[15], r.q[9], r.q[11], r.u[5], r.u[6],
                r.u[4 + row], r.u[12 + row]};   /* xm, y, z and xr, y, z */
    }

    /* derivative of this lane's column entry: row d of F @ Phi[:, j]
     * (rtbp.py:124-141, column_rhs); r: from the stage's record in velocity
     * lanes, zeros in the others                                              */
    template <bool FAST>
    __device__ __forceinline__ double column_row(double v, Entries r) const {
        double pv = vel_entry(v);
        const double t = dpp_into<DPP_SHR4, BANKS_VEL>(v, v);
        double p0 = quad_get<0x00>(t), p1 = quad_get<0x55>(t), p2 = quad_get<0xAA>(t);
        /* every operand is there before the arithmetic begins: left to itself the
         * compiler moves loads and DPP moves into the chain (STMs of 4,096
         * trajectories on pairs 11.1 ms, 12.2 without; one orbit's grid 0.67 and
         * 0.70; 262,144 uneven ones 84.7 and 87.3)                          */
        asm volatile(""
                     : "+v"(r.Q6), "+v"(r.Q7), "+v"(r.Q8), "+v"(r.Q9), "+v"(r.Q10), "+v"(r.Q11),
                       "+v"(r.y), "+v"(r.z), "+v"(r.pa), "+v"(r.pb), "+v"(pv), "+v"(p0),
                       "+v"(p1), "+v"(p2));
        const double a53 = r.Q6 * 3.0;
        const double b53 = r.Q7 * 3.0;
        const double c3 = r.Q8 + r.Q9;
        const double gx = r.Q10 + r.Q11;
        const double dd = ((diag + a53 * (r.pa * r.pa)) + b53 * (r.pb * r.pb)) - c3;
        const double uxy = (3.0 * r.y) * gx;
        const double uxz = (3.0 * r.z) * gx;
        const double uyz = ((3.0 * r.y) * r.z) * (r.Q6 + r.Q7);
        const double cA = (l == 4) ? dd : ((l == 5) ? uxy : uxz);
        const double cB = (l == 4) ? uxy : ((l == 5) ? dd : uyz);
        const double cC = (l == 4) ? uxz : ((l == 5) ? uyz : dd);
        const double acc = ((0.0 + cA * p0) + cB * p1) + cC * p2;
        const double o = acc + e2 * pv;
        if constexpr (FAST) return o;
        return vel ? (l == 7 ? 0.0 : o) : (l == 3 ? 0.0 : 0.0 + pv);
    }

    /* Lane42's in-lane sum over a block (entries 0..5 from 0.0), in the lane
     * of entry 5: the running sum moves from lane to lane                  */
    __device__ __forceinline__ static double block_sum(double term) {
        double s = 0.0 + term;
        s = row_shr<1>(s) + term;
        s = row_shr<1>(s) + term;
        s = row_shr<2>(s) + term;
        s = row_shr<1>(s) + term;
        return row_shr<1>(s) + term;
    }
    template <int N>
    __device__ __forceinline__ static double row_shr(double v) {
        return dpp_into<0x110 + N, 0xF>(v, v);
    }
    static constexpr int SUM_LANE0 = 6;                    /* the state's block sum */
    __device__ __forceinline__ static constexpr int sum_lane(int blk) { return 8 * blk + 14; }

    /* scaled errors of this lane's component (rk.py:2457-2463), 0 without one */
    template <bool FAST>
    __device__ __forceinline__ void scaled_errors(double y, double yh, const double (&k)[DOP_K],
                                                  double h, double rtol, double atol,
                                                  FastChk& c, double& q5, double& q3) const {
        double e5 = 0.0, e3 = 0.0;
        int n = 0;
#pragma unroll
        for (int j = 0; j < DOP_K; ++j)
            if (HH_DOP_E5[j] != 0.0) e5 = e5 + tab.e.at(n++) * k[j];
#pragma unroll
        for (int j = 0; j < DOP_K; ++j)
            if (HH_DOP_E3[j] != 0.0) e3 = e3 + tab.e.at(n++) * k[j];
        const double m = np_max(__builtin_fabs(y), __builtin_fabs(yh));
        const double sc = act ? atol + rtol * m : 1.0;
        const double n5 = act ? e5 * h : 0.0;
        const double n3 = act ? e3 * h : 0.0;
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
    }

    /* error norm from the two sums of squares (rk.py:2464-2467) */
    template <bool FAST>
    __device__ __forceinline__ static double error_norm(double s5, double s3, double h,
                                                        FastChk& c) {
        const double denom = (s5 + 0.01 * s3) * 42.0;
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

    /* pi_accept_factor(err, err_prev) and pi_reject_factor(err) with their
     * three pow calls in lanes 0..2                                         */
    __device__ __forceinline__ void step_factors(double err, double err_prev, double& f_acc,
                                                 double& f_rej) const {
        const double beta = 1.0 / (8.0 + 1.0);
        const double alpha = 0.4 * beta;
        const double err_exp = 1.0 / 8.0;
        const double px = (lane == 1) ? err_prev : err;
        const double pe = (lane == 0) ? -beta : ((lane == 1) ? alpha : -err_exp);
        step_factors_from(pt, err, err_prev, px, pe,
                          [](double v, int i) { return rlane(v, i); }, f_acc, f_rej);
    }
};

/* dop853_attempt's stages and solution, one component per lane; W supplies
 * the right-hand side; its last argument numbers those of an integration
 * between two norms: 0..11 an attempt's, 12..14 the extension stages',
 * RHS_START the start's                                                     */
constexpr int RHS_START = 15;

template <bool FAST, class W>
__device__ __forceinline__ double dop853_stages(const W& w, double y, double (&k)[DOP_K], double h,
                                                FastChk& c) {
    const RowTab<58> ha = w.tab.a.times(h);
    int n = 0;
#pragma unroll
    for (int i = 1; i < DOP_S; ++i) {
        double ys = y;
#pragma unroll
        for (int j = 0; j < i; ++j)
            if (HH_DOP_A[i][j] != 0.0) ys = ys + ha.at(n++) * k[j];
        k[i] = w.template rhs_form<FAST>(ys, c, i - 1);
    }
    double yh = y;
#pragma unroll
    for (int j = 0; j < DOP_S; ++j)
        if (HH_DOP_B[j] != 0.0) yh = yh + ha.at(n++) * k[j];
    k[DOP_S] = w.template rhs_form<FAST>(yh, c, DOP_S - 1);
    return yh;
}

/* The three extension stages and the seven interpolant rows of this lane's
 * component (rk.py:1836-1874)                                              */
template <class W>
__device__ __forceinline__ void dop853_rows(const W& w, double y_old, double y_new,
                                            const double (&k)[DOP_K], double hs,
                                            double (&row)[DOP_P]) {
    double kx[DOP_SX - DOP_K];
#pragma unroll
    for (int sr = DOP_K; sr < DOP_SX; ++sr) {
        double acc = 0.0;
#pragma unroll
        for (int r = 0; r < sr; ++r) {
            const double a = HH_DOP_A[sr][r];
            if (a != 0.0) acc = acc + a * (r < DOP_K ? k[r] : kx[r - DOP_K]);
        }
        kx[sr - DOP_K] = w.rhs(y_old + hs * acc, sr - 1);
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

/* zeros for the lanes that read none of the field's entries; a barrier of the
 * workgroup must follow                                                     */
__device__ __forceinline__ void wave_lds_clear(StageRec& zero) {
    for (int i = (int)threadIdx.x; i < 64; i += (int)blockDim.x) {
        zero.q[i] = 0.0;
        zero.u[i] = 0.0;
    }
}

struct Wave42 : Var42 {
    StageRec* rec;            /* this wave's record                              */
    const StageRec* mine;     /* what this lane reads: rec or the zeros          */

    __device__ __forceinline__ void setup(int lane_, double mu_, int fwd,
                                          unsigned long long flip, const PowTab* pt_,
                                          StageRec* rec_, const StageRec* zero) {
        Var42::setup(lane_, mu_, fwd, flip, pt_);
        rec = rec_;
        mine = (vel && l != 7) ? rec_ : zero;
    }

    /* accessors shared with the pair layout */
    __device__ __forceinline__ bool holds() const { return act; }
    __device__ __forceinline__ bool leader() const { return lane == 0; }

    /* derivative of this lane's component; v = this lane's component of the
     * stage state (idle() in lanes without one)                             */
    template <bool FAST>
    __device__ __forceinline__ double rhs_form(double v, FastChk& c, int = 0) const {
        double w, u, pos;
        const double q = quotient<FAST>(v, c, w, u, pos);
        rec->q[lane] = q;
        rec->u[lane] = u;
        /* the wave's own stores before its loads */
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const Entries e = entries(*mine);
        lds_order();
        const double os = state_row<FAST>(v, q, w, pos);
        const double oc = column_row<FAST>(v, e);
        __builtin_amdgcn_wave_barrier();
        return xor_sign(st ? os : oc, sign);
    }

    /* whether the state's lanes left the range of the unscaled forms */
    __device__ __forceinline__ bool left_range(const FastChk& c) const {
        return st && c.outside();
    }

    __device__ __forceinline__ double rhs(double v, int = 0) const {
        FastChk c;
        c.num(mu);
        c.num(mu2);
        const double o = rhs_form<true>(v, c);
        if (__builtin_expect(__any(left_range(c)), 0)) return rhs_form<false>(v, c);
        return o;
    }

    /* Lane42::reduce of in-lane sums over a block: sq = this lane's term */
    __device__ __forceinline__ double block_tree(double sq) const {
        const double s = block_sum(sq);
        const double B0 = rlane(s, SUM_LANE0), B1 = rlane(s, sum_lane(1)), B2 = rlane(s, sum_lane(2));
        const double B3 = rlane(s, sum_lane(3)), B4 = rlane(s, sum_lane(4));
        const double B5 = rlane(s, sum_lane(5)), B6 = rlane(s, sum_lane(6));
        return ((B0 + B1) + (B2 + B3)) + ((B4 + B5) + (B6 + 0.0));
    }

    /* initial_step (rk.py:2443-2448) with the block-tree sums of Lane42 */
    __device__ __forceinline__ double initial_step(double y, double f0,
                                                   const StepParams& sp) const {
        const double sc = sp.atol + sp.rtol * __builtin_fabs(y);
        const double ua = y / sc;
        const double ub = f0 / sc;
        const double s0 = block_tree(act ? ua * ua : 0.0);
        const double s1 = block_tree(act ? ub * ub : 0.0);
        const double sn = __builtin_sqrt(42.0);
        return select_initial_step(__builtin_sqrt(s0) / sn, __builtin_sqrt(s1) / sn, sp.min_step,
                                   sp.max_step);
    }

    template <bool FAST>
    __device__ __forceinline__ double attempt_form(double y, double (&k)[DOP_K], double h,
                                                   double rtol, double atol, double& yh,
                                                   FastChk& cs, FastChk& ce) const {
        yh = dop853_stages<FAST>(*this, y, k, h, cs);
        double q5, q3;
        scaled_errors<FAST>(y, yh, k, h, rtol, atol, ce, q5, q3);
        const double s5 = block_tree(q5 * q5);
        const double s3 = block_tree(q3 * q3);
        return error_norm<FAST>(s5, s3, h, ce);
    }

    /* dop853_attempt, one component per lane */
    __device__ __forceinline__ double attempt(double y, double (&k)[DOP_K], double h, double rtol,
                                              double atol, double& yh) const {
        FastChk cs, ce;
        cs.num(mu);
        cs.num(mu2);
        double err = attempt_form<true>(y, k, h, rtol, atol, yh, cs, ce);
        if (__builtin_expect(__any(left_range(cs) || ce.outside() || !(err < __builtin_inf())),
                             0)) {
            asm volatile("" : "+v"(h));
            err = attempt_form<false>(y, k, h, rtol, atol, yh, cs, ce);
        }
        return err;
    }
};

/* dense_from_rows of the last step of an integration (FinalOut::accepted) */
template <class W>
__device__ __forceinline__ double dop853_dense_at(const W& w, double y_old, double y_new,
                                                  const double (&k)[DOP_K], double hs,
                                                  double xq) {
    double row[DOP_P];
    dop853_rows(w, y_old, y_new, k, hs, row);
    return dense_from_rows(row, y_old, xq);
}

}  // namespace hh

#endif /* HH_WAVE_H */
