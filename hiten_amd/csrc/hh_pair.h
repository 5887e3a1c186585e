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
 * writes a record of the stage's quotients and coordinates to LDS, then the
 * record's tag, and goes on without waiting; the STM wave reads tag and record
 * together until the tag is there, then forms its rows.  Norms over all 42
 * components are exchanged the same way, each wave waiting for the other's
 * part.  There is no barrier of the workgroup in this, so other waves of the
 * workgroup may do other work meanwhile.  Each wave evaluates exactly Wave42's
 * expressions for its lanes, so results are bit-identical to Wave42's (and
 * so to Lane42's and the reference's).  Error-norm and initial-step sums
 * exchange their block sums through LDS and are combined in Wave42's
 * block-tree order by both waves, which then take the same step-size
 * decisions -- and the same decision to evaluate an attempt again with the
 * general forms, from the flags both waves write beside the sums.
 *
 * Bound by the two instruction streams, which are about equally long: of the
 * 8,400 cycles of an attempt the state wave waits 950 for the other's last
 * stage and sums, the STM wave 550 for records.  One trajectory alone: 3.42 us
 * an attempt (5.83 us with twelve quotients read back by readlane, IEEE
 * divisions, both roles in one stream and a barrier a stage; a barrier a stage
 * alone costs what the tags do; 3.59 us with selected powers, see quotient), 4.8
 * us in the one-wave form (6.75
 * us).  262,144 uneven trajectories on the persistent kernel, whose heaviest
 * ones end in this form: 94 -> 59 ms.
 */
#ifndef HH_PAIR_H
#define HH_PAIR_H

#include "hh_wave.h"

namespace hh {

/* What the state wave hands to the STM wave in one right-hand side: entries
 * 0..15 are the first row's quotients and distance components, 16..31 zeros for
 * the lanes whose row of F has no entries (they read 16 further on), 32..47
 * take what the state wave's other lanes write.                             */
struct PairRec {
    double q[48], u[48];
};

/* LDS of one pair.  Every right-hand side between two norms has a record of its
 * own, so a record is written again only after both waves have met in the norm
 * that follows its reading; the sums of consecutive norms alternate between two
 * sets.  Tags hold the number of the norm that comes next.                   */
constexpr int PAIR_RECS = 16;
struct PairLds {
    PairRec rec[PAIR_RECS];
    unsigned tag[PAIR_RECS + 64 + PAIR_RECS];   /* a record's tag, and what lanes 1..63 write */
    unsigned met[2];           /* the last norm each wave has written its part of  */
    unsigned next;             /* the next norm, while the pair has no trajectory  */
    int left[2][2];            /* a wave's lanes left the unscaled forms           */
    double bsum[2][2][8];      /* block sums of a norm's two sums, blocks 0..6     */
};

/* a barrier of the workgroup must follow */
__device__ __forceinline__ void pair_lds_clear(PairLds& p) {
    for (int i = (int)threadIdx.x; i < PAIR_RECS * 48; i += (int)blockDim.x) {
        p.rec[i / 48].q[i % 48] = 0.0;
        p.rec[i / 48].u[i % 48] = 0.0;
    }
    if (threadIdx.x < PAIR_RECS) p.tag[threadIdx.x] = 0;
    if (threadIdx.x < 2) p.met[threadIdx.x] = 0;
    if (threadIdx.x == 0) p.next = 1;
}

/* Tags: the LDS carries out one wave's accesses in order, so data written before
 * a tag are there for a wave that reads the tag before the data.            */
__device__ __forceinline__ unsigned lds_tag(const unsigned* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

/* ROLE 0: the state wave, 1: the STM wave.  The role is a template parameter so
 * that each wave runs an instruction stream of its own, without the other's
 * half of every right-hand side between its own                            */
template <int ROLE, bool WATCH = false>
struct Pair42 : Var42 {
    PairLds* lds;
    const PairRec* mine;    /* where this lane reads, from the first record on   */
    double *wq, *wu;        /* where it writes, in the first record              */
    unsigned* wt;           /* and its tag                                       */
    mutable unsigned next;  /* number of the next norm                           */
    const int* watch;       /* WATCH: a flag in LDS                              */
    mutable bool seen;      /* and whether the state wave found it set before the
                               last norm, the same in both waves                 */

    /* after a barrier of the workgroup that both waves have passed since
     * pair_lds_clear or the finish of the trajectory before                  */
    __device__ __forceinline__ void setup(int lane_, double mu_, int fwd,
                                          unsigned long long flip, PairLds* p,
                                          const PowTab* pt_) {
        Var42::setup(lane_, mu_, fwd, flip, pt_);
        lds = p;
        const double* z = p->rec[0].q + ((vel && l != 7) ? 0 : 16);
        mine = (const PairRec*)z;
        const int at = st ? lane : 32 + (lane & 15);
        wq = p->rec[0].q + at;
        wu = p->rec[0].u + at;
        wt = p->tag + (lane == 0 ? 0 : PAIR_RECS + lane);
        next = p->next;
        watch = nullptr;
        seen = false;
        /* the state wave holds the state only, the STM wave the columns */
        act = act && ((ROLE == 0) == st);
    }

    /* before the barrier that ends a trajectory another one may follow */
    __device__ __forceinline__ void finish() const {
        if (leader()) lds->next = next;
    }

    __device__ __forceinline__ bool holds() const { return act; }
    __device__ __forceinline__ bool leader() const { return ROLE == 0 && lane == 0; }

    __device__ __forceinline__ bool left_range(const FastChk& c) const {
        return ROLE == 0 && st && c.outside();
    }

    /* the state wave's half: record n, then its tag */
    __device__ __forceinline__ void hand_over(int n, double q, double u) const {
        constexpr int R = sizeof(PairRec) / sizeof(double);
        wq[n * R] = q;
        wu[n * R] = u;
        lds_order();
        __hip_atomic_store(wt + n, next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    /* the STM wave's half: its rows once the tag of record n is there.  The
     * record is read along with the tag, and again until the tag was there
     * first; the state wave writes it without waiting for this wave.        */
    template <bool FAST>
    __device__ __forceinline__ double column(double v, int n) const {
        unsigned t;
        Entries e;
        auto look = [&]() {
            lds_order();
            t = lds_tag(lds->tag + n);
            lds_order();
            e = entries(mine[n]);
            lds_order();
            return __builtin_amdgcn_readfirstlane(t) == next;
        };
        /* the first look by itself: the loop's waits are not in its way */
        if (__builtin_expect(!look(), 0))
            while (!look()) {}
        return column_row<FAST>(v, e);
    }

    /* derivative of this lane's component, right-hand side n; v = this lane's
     * component of the stage state                                          */
    template <bool FAST>
    __device__ __forceinline__ double rhs_form(double v, FastChk& c, int n) const {
        if constexpr (ROLE == 0) {
            double w, u, pos;
            const double q = quotient<FAST>(v, c, w, u, pos);
            hand_over(n, q, u);
            double o = xor_sign(state_row<FAST>(v, q, w, pos), sign);
            /* the stores leave before the next stage begins */
            asm volatile("" : "+v"(o) : : "memory");
            return o;
        } else {
            return xor_sign(column<FAST>(v, n), sign);
        }
    }

    /* the state wave alone decides which form its quotients take */
    __device__ __forceinline__ double rhs(double v, int n = RHS_START) const {
        if constexpr (ROLE == 0) {
            FastChk c;
            c.num(mu);
            c.num(mu2);
            double w, u, pos;
            double q = quotient<true>(v, c, w, u, pos);
            const bool general = __any(left_range(c));
            if (__builtin_expect(general, 0)) q = quotient<false>(v, c, w, u, pos);
            hand_over(n, q, u);
            return xor_sign(state_row<false>(v, q, w, pos), sign);
        } else {
            return xor_sign(column<false>(v, n), sign);
        }
    }

    /* Wave42::block_tree of two sums at once over both waves: each wave
     * contributes the block sums of its own blocks, and whether its lanes
     * left the unscaled forms, and waits for the other's.  Neither can be more
     * than one norm ahead: it needs the other's part of each.               */
    __device__ __forceinline__ bool pair_tree(double sa, double sb, bool left, double& ra,
                                              double& rb) const {
        const double ga = block_sum(sa);
        const double gb = block_sum(sb);
        const int set = next & 1;
        double(*sum)[8] = lds->bsum[set];
        if (l == 6 && (ROLE == 0 ? lane == 6 : !st)) {
            sum[0][block()] = ga;
            sum[1][block()] = gb;
        }
        int any = __any(left) ? 1 : 0;
        if constexpr (WATCH && ROLE == 0)
            any |= __builtin_amdgcn_readfirstlane(__hip_atomic_load(
                       watch, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP)) ? 2 : 0;
        if (lane == 0) lds->left[set][ROLE] = any;
        lds_order();
        if (lane == 0)
            __hip_atomic_store(&lds->met[ROLE], next, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        unsigned t;
        int other;
        do {
            lds_order();
            t = lds_tag(&lds->met[1 - ROLE]);
            lds_order();
            const double* A = sum[0];
            const double* B = sum[1];
            ra = ((A[0] + A[1]) + (A[2] + A[3])) + ((A[4] + A[5]) + (A[6] + 0.0));
            rb = ((B[0] + B[1]) + (B[2] + B[3])) + ((B[4] + B[5]) + (B[6] + 0.0));
            other = lds->left[set][1 - ROLE];
            lds_order();
        } while ((int)(__builtin_amdgcn_readfirstlane(t) - next) < 0);
        ++next;
        if constexpr (WATCH)
            seen = __builtin_amdgcn_readfirstlane((ROLE == 0 ? any : other) & 2) != 0;
        return ((any | other) & 1) != 0;
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
