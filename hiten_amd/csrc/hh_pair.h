/* hh_pair.h -- one 42-d variational trajectory per pair of waves.
 *
 * The two waves of a 128-thread workgroup share one trajectory in the lane
 * layout of hh_wave.h:
 *   - the state wave (wave 0) holds the state in its first row and forms
 *     per stage the field's quotients and the state rows;
 *   - the STM wave (wave 1) holds the six STM columns and forms the Hessian
 *     of the effective potential from the quotients of the same stage, then
 *     the rows of F @ Phi.
 * The state of a stage does not depend on Phi, so the two instruction
 * streams run side by side on two SIMDs: per right-hand side the state wave
 * writes the stage's quotients and coordinates to LDS and both waves meet at
 * one barrier; the STM wave then forms its rows from them while the state
 * wave goes on to its state rows and the next stage.  Norms over all 42
 * components take one more barrier.  Each wave evaluates exactly Wave42's
 * expressions for its lanes, so results are bit-identical to Wave42's (and
 * so to Lane42's and the reference's).  Error-norm and initial-step sums
 * exchange their block sums through LDS and are combined in Wave42's
 * block-tree order by both waves, which then take the same step-size
 * decisions -- and the same decision to evaluate an attempt again with the
 * general forms, from the flags both waves write beside the sums.
 *
 * Bound by the longer of the two instruction streams and the LDS round trip
 * and barrier of every stage.  One trajectory alone: 3.4 us an attempt (5.83
 * us with twelve quotients read back by readlane, IEEE divisions and both
 * roles in one stream; 4.22 us before each role had a stream of its own, 3.94
 * us before the state row hid the record's stores, 3.74 us before the step
 * controller lost its branches), 4.8 us in the one-wave form (6.75 us).
 * 262,144 uneven trajectories on the persistent kernel, whose heaviest ones
 * end in this form: 94 -> 59 ms.
 */
#ifndef HH_PAIR_H
#define HH_PAIR_H

#include "hh_wave.h"

namespace hh {

/* LDS of one pair.  A record is read by the STM wave before the barrier of the
 * next right-hand side, so consecutive right-hand sides take different
 * records: the stages of an attempt alternate between 1 and 0 (starting at 1,
 * ending at 0), the extension stages take 1, 0 and 2.                       */
struct PairLds {
    StageRec rec[3], zero[3];
    double bsum[2][8];     /* block sums of two norms, blocks 0..6      */
    int left[2];           /* a wave's lanes left the unscaled forms    */
};

__device__ __forceinline__ void pair_lds_clear(PairLds& p) {
    for (int b = 0; b < 3; ++b) wave_lds_clear(p.zero[b]);
}

/* ROLE 0: the state wave, 1: the STM wave.  The role is a template parameter so
 * that each wave runs an instruction stream of its own, without the other's
 * half of every right-hand side between its own                            */
template <int ROLE>
struct Pair42 : Var42 {
    PairLds* lds;
    const StageRec* mine;   /* the records this lane reads: rec or zero    */

    __device__ __forceinline__ void setup(int lane_, double mu_, int fwd,
                                          unsigned long long flip, PairLds* p,
                                          const PowTab* pt_) {
        Var42::setup(lane_, mu_, fwd, flip, pt_);
        lds = p;
        mine = (vel && l != 7) ? p->rec : p->zero;
        /* the state wave holds the state only, the STM wave the columns */
        act = act && ((ROLE == 0) == st);
    }

    __device__ __forceinline__ bool holds() const { return act; }
    __device__ __forceinline__ bool leader() const { return ROLE == 0 && lane == 0; }

    __device__ __forceinline__ bool left_range(const FastChk& c) const {
        return ROLE == 0 && st && c.outside();
    }

    /* record of right-hand side n (a constant once loops are unrolled) */
    __device__ __forceinline__ static constexpr int buf(int n) {
        return n == 14 ? 2 : (n + 1) % 2;
    }

    /* derivative of this lane's component; v = this lane's component of the
     * stage state.  One barrier per call, in both waves: the state wave
     * writes the stage record before it, the STM wave reads it after.       */
    template <bool FAST>
    __device__ __forceinline__ double rhs_form(double v, FastChk& c, int n) const {
        const int b = buf(n);
        if constexpr (ROLE == 0) {
            double w, u, pos;
            const double q = quotient<FAST>(v, c, w, u, pos);
            lds->rec[b].q[lane] = q;
            lds->rec[b].u[lane] = u;
            /* the state row while the stores are on their way: the barrier
             * waits for them                                               */
            double o = xor_sign(state_row<FAST>(v, q, w, pos), sign);
            asm volatile("" : "+v"(o));
            __syncthreads();
            return o;
        } else {
            __syncthreads();
            return xor_sign(column_row<FAST>(v, entries(mine[b])), sign);
        }
    }

    /* the state wave alone decides which form its quotients take */
    __device__ __forceinline__ double rhs(double v, int n = RHS_START) const {
        const int b = buf(n);
        if constexpr (ROLE == 0) {
            FastChk c;
            c.num(mu);
            c.num(mu2);
            double w, u, pos;
            double q = quotient<true>(v, c, w, u, pos);
            const bool general = __any(left_range(c));
            if (__builtin_expect(general, 0)) q = quotient<false>(v, c, w, u, pos);
            lds->rec[b].q[lane] = q;
            lds->rec[b].u[lane] = u;
            __syncthreads();
            return xor_sign(state_row<false>(v, q, w, pos), sign);
        } else {
            __syncthreads();
            return xor_sign(column_row<false>(v, entries(mine[b])), sign);
        }
    }

    /* Wave42::block_tree of two sums at once over both waves: each wave
     * contributes the block sums of its own blocks, and whether its lanes
     * left the unscaled forms.  One barrier.                                */
    __device__ __forceinline__ bool pair_tree(double sa, double sb, bool left, double& ra,
                                              double& rb) const {
        const double ga = block_sum(sa);
        const double gb = block_sum(sb);
        if (l == 6 && (ROLE == 0 ? lane == 6 : !st)) {
            lds->bsum[0][block()] = ga;
            lds->bsum[1][block()] = gb;
        }
        const int any = __any(left) ? 1 : 0;
        if (lane == 0) lds->left[ROLE] = any;
        __syncthreads();
        const double* A = lds->bsum[0];
        const double* B = lds->bsum[1];
        ra = ((A[0] + A[1]) + (A[2] + A[3])) + ((A[4] + A[5]) + (A[6] + 0.0));
        rb = ((B[0] + B[1]) + (B[2] + B[3])) + ((B[4] + B[5]) + (B[6] + 0.0));
        return (lds->left[0] | lds->left[1]) != 0;
    }

    /* Wave42::initial_step */
    __device__ __forceinline__ double initial_step(double y, double f0,
                                                   const StepParams& sp) const {
        const double sc = sp.atol + sp.rtol * __builtin_fabs(y);
        const double ua = y / sc;
        const double ub = f0 / sc;
        double s0, s1;
        pair_tree(act ? ua * ua : 0.0, act ? ub * ub : 0.0, false, s0, s1);
        const double sn = __builtin_sqrt(42.0);
        return select_initial_step(__builtin_sqrt(s0) / sn, __builtin_sqrt(s1) / sn, sp.min_step,
                                   sp.max_step);
    }

    template <bool FAST>
    __device__ __forceinline__ double attempt_form(double y, double (&k)[DOP_K], double h,
                                                   double rtol, double atol, double& yh,
                                                   bool& left) const {
        FastChk cs, ce;
        cs.num(mu);
        cs.num(mu2);
        yh = dop853_stages<FAST>(*this, y, k, h, cs);
        double q5, q3, s5, s3;
        scaled_errors<FAST>(y, yh, k, h, rtol, atol, ce, q5, q3);
        left = pair_tree(q5 * q5, q3 * q3, left_range(cs) || ce.outside(), s5, s3);
        FastChk cn;
        const double err = error_norm<FAST>(s5, s3, h, cn);
        left = left || cn.outside() || !(err < __builtin_inf());
        return err;
    }

    /* Wave42::attempt with the pair's right-hand side and norm */
    __device__ __forceinline__ double attempt(double y, double (&k)[DOP_K], double h, double rtol,
                                              double atol, double& yh) const {
        bool left;
        double err = attempt_form<true>(y, k, h, rtol, atol, yh, left);
        /* the same in both waves and all lanes: every branch around a barrier
         * is on a scalar                                                    */
        if (__builtin_expect(__builtin_amdgcn_readfirstlane(left ? 1 : 0), 0)) {
            asm volatile("" : "+v"(h));
            err = attempt_form<false>(y, k, h, rtol, atol, yh, left);
        }
        return err;
    }
};

}  // namespace hh

#endif /* HH_PAIR_H */
