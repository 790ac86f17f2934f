/* radix.h - the radix step of a group of slots held in registers: butterflies of up to 4 levels with lazy reduction (device code,
 * and host code for the tests of its bounds).
 *
 * Lazy reduction.  For |x| <= k p, k <= 4, mul_shoup gives at most (1/2 + k/16) p, reduce p/2 + 1; sums are exact below 8p.
 * The DIF follows every slot's bound from inputs within p (DifRed): a sum is reduced where it would take the next
 * level's difference past 4p (above 2p), or at the last level above p.  13 reductions for 16 points in 4 levels, where one of
 * every sum at odd levels took 16.  The DIT's outputs grow by less than 0.71 p a level: from inputs within p (and a trivial first
 * level) 2, 2.625, 3.29, 3.995 p.  Rounds with another one after them leave their outputs so; that one reduces the half of
 * its inputs that its first level does not multiply (then 1.25, 1.83, 2.45, 3.10 p), and a pass's last round reduces all
 * outputs.  (Reducing all outputs of every round: 16 a round in place of 0, 8 and 24.)  Both together, ms:
 * 2^27 x 2^27 limbs 22.16 to 21.98, 2^25 x 2^25 5.38 to 5.28, 4096 leaves as a plan 4.89 to 4.80.
 * Where the round's low row bits are known to be zero at compile time, twiddles w^0 = 1 are not multiplied: the DIF
 * difference then follows the sum path's rule, the DIT skips them at its first level (where all of them are 1). */
#ifndef NTTM_RADIX_H
#define NTTM_RADIX_H
#include "arith.h"

/* rlow == 0 known at compile time (the round over the lowest bits of a fixed-shape tile): the butterflies with
 * jj = 0 then have the twiddle w^0 = 1 */
#ifndef NTTM_TRIVIAL_W
#define NTTM_TRIVIAL_W(rlow, jj) ((jj) == 0 && __builtin_constant_p(rlow) && (rlow) == 0)
#endif

/* which outputs of each DIF level are reduced, from the slots' bounds in units of p (TRIV: the twiddles of slot 0 of every
 * block are 1 and not multiplied) */
template <int LOGR, bool TRIV> struct DifRed {
    uint32_t mask[LOGR];
    constexpr DifRed() : mask{}
    {
        constexpr int R = 1 << LOGR;
        double b[R] = {};
        for (int j = 0; j < R; j++) b[j] = 1.0;
        for (int lev = 0; lev < LOGR; lev++) {
            const int h = R >> (lev + 1);
            const double most = lev == LOGR - 1 ? 1.0 : 2.0;
            for (int jj = 0; jj < h; jj++)
                for (int j = jj; j < R; j += 2 * h) {
                    const double sm = b[j] + b[j + h];
                    const bool one = TRIV && jj == 0;
                    b[j] = sm; b[j + h] = one ? sm : 0.5 + sm / 16;
                    for (int e = j; e <= j + h; e += h)
                        if (b[e] > most) { mask[lev] |= 1u << e; b[e] = 0.5; }
                }
        }
    }
};

template <int LOGR, typename TW>
NTTM_HD void dif_group(double *v, int s_lo, uint32_t rlow, TW tw, double p, double pinv)
{
    constexpr int R = 1 << LOGR;
    constexpr DifRed<LOGR, false> rn{};
    constexpr DifRed<LOGR, true> rt{};
#pragma unroll
    for (int lev = 0; lev < LOGR; lev++) {
        const int k = LOGR - 1 - lev, h = 1 << k;
        const uint32_t red = NTTM_TRIVIAL_W(rlow, 0) ? rt.mask[lev] : rn.mask[lev];
#pragma unroll
        for (int jj = 0; jj < h; jj++) {
            const bool one = NTTM_TRIVIAL_W(rlow, jj);
            const double2 w = one ? make_double2(1.0, 0.0) : tw_at(tw, rlow, (1u << (s_lo + k)) + ((uint32_t)jj << s_lo));
#pragma unroll
            for (int j = jj; j < R; j += 2 * h) {
                const double u = v[j], x = v[j + h];
                const double sm = u + x, df = u - x;
                v[j] = (red >> j) & 1 ? reduce(sm, p, pinv) : sm;
                v[j + h] = !one ? mul_shoup(df, w.x, w.y, p) : (red >> (j + h)) & 1 ? reduce(df, p, pinv) : df;
            }
        }
    }
}

/* one DIT butterfly level's inputs: wide: within 4p (at the round's first level), so u, and an x that is not multiplied, are
 * reduced */
NTTM_HD double dit_u(double u, bool wide, double p, double pinv) { return wide ? reduce(u, p, pinv) : u; }
/* wide_in: the inputs are within 4p, else p; wide_out: the outputs may be left within 4p, else they are reduced */
template <int LOGR, typename TW>
NTTM_HD void dit_group(double *v, int s_lo, uint32_t rlow, TW tw, double p, double pinv, bool wide_in = false,
                                          bool wide_out = false)
{
    constexpr int R = 1 << LOGR;
#pragma unroll
    for (int lev = 0; lev < LOGR; lev++) {
        const int k = lev, h = 1 << k;
        const bool red = lev == LOGR - 1 && !wide_out, wide = lev == 0 && wide_in;
#pragma unroll
        for (int jj = 0; jj < h; jj++) {
            const bool one = lev == 0 && NTTM_TRIVIAL_W(rlow, jj);
            const double2 w = one ? make_double2(1.0, 0.0) : tw_at(tw, rlow, (1u << (s_lo + k)) + ((uint32_t)jj << s_lo));
#pragma unroll
            for (int j = jj; j < R; j += 2 * h) {
                const double u = dit_u(v[j], wide, p, pinv);
                const double x = one ? dit_u(v[j + h], wide, p, pinv) : mul_shoup(v[j + h], w.x, w.y, p);
                const double s1 = u + x, s2 = u - x;
                v[j] = red ? reduce(s1, p, pinv) : s1;
                v[j + h] = red ? reduce(s2, p, pinv) : s2;
            }
        }
    }
}

/* dit_group with the inverse twiddles taken from the FORWARD stage table: w^-j of stage s is the mirrored forward entry
 * negated, w^-j = -w^(2^s - j) (w^(2^s) = -1), the negation folded into the butterfly (the product's sign flipped), and
 * w^0 = 1 taken from entry 1 (stage 0).  Lets a kernel keep one small table in LDS for both directions. */
template <int LOGR>
NTTM_HD void dit_group_mirror(double *v, int s_lo, uint32_t rlow, const double2 *tw, double p,
                                                 double pinv, bool wide_in, bool wide_out)
{
    constexpr int R = 1 << LOGR;
#pragma unroll
    for (int lev = 0; lev < LOGR; lev++) {
        const int k = lev, h = 1 << k, s = s_lo + k;
        const bool red = lev == LOGR - 1 && !wide_out, wide = lev == 0 && wide_in;
#pragma unroll
        for (int jj = 0; jj < h; jj++) {
            const bool one = lev == 0 && NTTM_TRIVIAL_W(rlow, jj);
            const uint32_t j = rlow + ((uint32_t)jj << s_lo);
            double2 w;                                   /* (w, wq) negated for a mirrored entry */
            if (jj == 0) {
                const bool z = rlow == 0;
                const double2 t = tw[z ? 1u : (2u << s) - j];
                w = z ? t : make_double2(-t.x, -t.y);
            } else {
                const double2 t = tw[(2u << s) - j];
                w = make_double2(-t.x, -t.y);
            }
#pragma unroll
            for (int i = jj; i < R; i += 2 * h) {
                const double u = dit_u(v[i], wide, p, pinv);
                const double x = one ? dit_u(v[i + h], wide, p, pinv) : mul_shoup(v[i + h], w.x, w.y, p);
                const double s1 = u + x, s2 = u - x;
                v[i] = red ? reduce(s1, p, pinv) : s1;
                v[i + h] = red ? reduce(s2, p, pinv) : s2;
            }
        }
    }
}
#endif
