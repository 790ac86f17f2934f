/* rounds.h - the radix rounds of the transform kernels on a tile held in registers and LDS (device code): slots and
 * groups of a thread, butterflies with lazy reduction, stage tables in global memory or LDS, the padded LDS layout. */
#ifndef NTTM_ROUNDS_H
#define NTTM_ROUNDS_H
#include "internal.h"

/* ---- rounds of a tile -------------------------------------------------------------------------------------------------
 * A tile of T = W x 2^m x H points (T <= 2^13) is handled by T / 16 threads holding 16 points each in registers.  The m
 * stages run in rounds of up to 4 stages (radix 2..16 in registers); between rounds the tile goes through LDS once.
 * In a round over row bits [s_lo, s_lo + logR) (L = logw + s_lo), thread t owns G = 16 / R groups of R points; group g
 * has the base element
 *     eb = (tau mod 2^L) | (tau div 2^L) << (L + logR),   tau = g * nthr + t,
 * and point j of the group is element eb + j 2^L.  For every point the lanes of a wave touch consecutive LDS words
 * (and, in the first and last round, consecutive global addresses of a row).  Since the round's bits lie inside the
 * row field, point j sits at global offset ob + j 2^(s_lo + lo) and at bit-reversed row kb + brev(j) 2^(m - s_lo - logR):
 * addresses and boundary-twiddle exponents of a group are a base plus compile-time multiples.  Each thread reads and
 * writes exactly the elements of its groups within a round, so one barrier separates consecutive rounds.
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
#define PASS_PTS 16               /* points per thread of full tiles; tiles below 16 points use one thread */

template <int BITS>
__device__ __forceinline__ constexpr uint32_t brev_c(uint32_t j)
{
    uint32_t r = 0;
    for (int i = 0; i < BITS; i++) r |= ((j >> i) & 1u) << (BITS - 1 - i);
    return r;
}

/* rlow == 0 known at compile time (the round over the lowest bits of a fixed-shape tile): the butterflies with
 * jj = 0 then have the twiddle w^0 = 1 */
#define NTTM_TRIVIAL_W(rlow, jj) ((jj) == 0 && __builtin_constant_p(rlow) && (rlow) == 0)

/* a stage table in global memory, read through a buffer resource: the table's base in scalar registers, the lane's
 * part of an index as the 32-bit vector offset and its compile-time part as the scalar offset, so a twiddle's address
 * costs no vector instruction (a 64-bit pointer sum costs two, in kernels bound by vector issue) */
struct GTab {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ explicit GTab(const double2 *p)
        : r(__builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, 0x7fffffff, 0x00020000)) {}
};
/* a stage table in LDS (or any pointer): restrict, so that its loads move freely around the tile's LDS stores */
typedef const double2 *__restrict__ LTab;
/* entry lane + fixed of a stage table (lane: the part that varies across lanes; fixed: a compile-time part) */
__device__ __forceinline__ double2 tw_at(LTab tw, uint32_t lane, uint32_t fixed) { return tw[lane + fixed]; }
__device__ __forceinline__ double2 tw_at(const GTab &tw, uint32_t lane, uint32_t fixed)
{
    typedef int v4i __attribute__((ext_vector_type(4)));
    const v4i x = __builtin_amdgcn_raw_buffer_load_b128(tw.r, (int)(lane * 16u), (int)(fixed * 16u), 0);
    double2 d;
    __builtin_memcpy(&d, &x, 16);
    return d;
}

/* a stage table read at compile-time indices only (uniform): through the scalar unit */
struct CTab {
    const __attribute__((address_space(4))) double2 *p;
    __device__ __forceinline__ explicit CTab(const double2 *q) : p((const __attribute__((address_space(4))) double2 *)q) {}
};
__device__ __forceinline__ double2 tw_at(const CTab &tw, uint32_t, uint32_t fixed)
{
    typedef double v2d __attribute__((ext_vector_type(2)));
    const v2d x = ((const __attribute__((address_space(4))) v2d *)tw.p)[fixed];
    return make_double2(x[0], x[1]);
}

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
__device__ __forceinline__ void dif_group(double *v, int s_lo, uint32_t rlow, TW tw, double p, double pinv)
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
__device__ __forceinline__ double dit_u(double u, bool wide, double p, double pinv) { return wide ? reduce(u, p, pinv) : u; }
/* wide_in: the inputs are within 4p, else p; wide_out: the outputs may be left within 4p, else they are reduced */
template <int LOGR, typename TW>
__device__ __forceinline__ void dit_group(double *v, int s_lo, uint32_t rlow, TW tw, double p, double pinv, bool wide_in = false,
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

/* geometry of the pass seen by one thread */
struct PassPos {
    int m, logw, lo, nthr, t;
};

/* f(slot, e, o, c, k) for every slot of a round: e the LDS index, o the global offset in the tile, c the column inside
 * the tile, k the bit-reversed row */
/* PAD: e is the padded LDS index (SwzLds below) of the element; eb and the slot offsets j 2^L have disjoint bits, so
 * pad(eb + j 2^L) = pad(eb) + pad(j 2^L), the second term a compile-time constant in the fixed-shape kernels */
template <int LOGR, int PTS, bool PAD = false, typename F>
__device__ __forceinline__ void for_slots(const PassPos &pp, int s_lo, F f)
{
    constexpr int R = 1 << LOGR, G = PTS / R;
    const int L = pp.logw + s_lo;
#pragma unroll
    for (int g = 0; g < G; g++) {
        const uint32_t tau = (uint32_t)(g * pp.nthr + pp.t);
        const uint32_t eb = (tau & ((1u << L) - 1)) | ((tau >> L) << (L + LOGR));
        const uint32_t pe = PAD ? eb + (eb >> 5) : eb;
        const uint32_t c = eb & ((1u << pp.logw) - 1), r = (eb >> pp.logw) & ((1u << pp.m) - 1);
        const uint32_t h = eb >> (pp.logw + pp.m);
        /* h << (lo + m) in 64 bits: a tile of the first pass of a 2^32-point transform has lo + m = 32 (and h = 0) */
        const uint32_t ob = (uint32_t)((uint64_t)h << (pp.lo + pp.m)) + (r << pp.lo) + c;
        const uint32_t kb = pp.m ? (__brev(r) >> (32 - pp.m)) : 0u;
        const int ksh = pp.m - s_lo - LOGR;
#pragma unroll
        for (int j = 0; j < R; j++) {
            const uint32_t dj = (uint32_t)j << L;
            f(g * R + j, pe + (PAD ? dj + (dj >> 5) : dj), ob + ((uint32_t)j << (s_lo + pp.lo)), c,
              kb + (brev_c<LOGR>(j) << ksh));
        }
    }
}

/* the radix step of one round on all PTS slots: PTS / R groups of R points */
/* TW: GTab (a global stage table) or LTab (a table in LDS, named explicitly so that it stays restrict) */
template <int LOGR, bool INV, int PTS, typename TW>
__device__ __forceinline__ void round_compute(double *v, const PassPos &pp, int s_lo, TW tw, double p, double pinv, bool wide_in = false,
                                              bool wide_out = false)
{
    constexpr int R = 1 << LOGR, G = PTS / R;
    const int L = pp.logw + s_lo;
#pragma unroll
    for (int g = 0; g < G; g++) {
        const uint32_t tau = (uint32_t)(g * pp.nthr + pp.t);
        const uint32_t rlow = (tau & ((1u << L) - 1)) >> pp.logw;      /* row bits below s_lo */
        if (INV) dit_group<LOGR, TW>(v + g * R, s_lo, rlow, tw, p, pinv, wide_in, wide_out);
        else dif_group<LOGR, TW>(v + g * R, s_lo, rlow, tw, p, pinv);
    }
}

/* dit_group with the inverse twiddles taken from the FORWARD stage table: w^-j of stage s is the mirrored forward entry
 * negated, w^-j = -w^(2^s - j) (w^(2^s) = -1), the negation folded into the butterfly (the product's sign flipped), and
 * w^0 = 1 taken from entry 1 (stage 0).  Lets a kernel keep one small table in LDS for both directions. */
template <int LOGR>
__device__ __forceinline__ void dit_group_mirror(double *v, int s_lo, uint32_t rlow, const double2 *tw, double p,
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
template <int LOGR, int PTS>
__device__ __forceinline__ void round_compute_mirror(double *v, const PassPos &pp, int s_lo, const double2 *tw, double p,
                                                     double pinv, bool wide_in = false, bool wide_out = false)
{
    constexpr int R = 1 << LOGR, G = PTS / R;
    const int L = pp.logw + s_lo;
#pragma unroll
    for (int g = 0; g < G; g++) {
        const uint32_t tau = (uint32_t)(g * pp.nthr + pp.t);
        const uint32_t rlow = (tau & ((1u << L) - 1)) >> pp.logw;
        dit_group_mirror<LOGR>(v + g * R, s_lo, rlow, tw, p, pinv, wide_in, wide_out);
    }
}

/* rounds of a pass: sizes of at most maxr bits (the log2 of the points per thread, at most 4), balanced; forward from
 * the top bits down, inverse from bit 0 up */
__device__ __forceinline__ int round_count(int m, int maxr) { return (m + maxr - 1) / maxr; }
__device__ __forceinline__ void round_split(int m, int i, int *s_lo, int *logR, bool inv, int maxr)
{
    const int nr = round_count(m, maxr), q = m / nr, rem = m % nr;
    int lo = 0;                                     /* rounds in ascending bit order: sizes q+1 first (rem of them) */
    int k = inv ? i : nr - 1 - i;
    for (int r = 0; r < k; r++) lo += q + (r < rem ? 1 : 0);
    *s_lo = lo; *logR = q + (k < rem ? 1 : 0);
}

/* call body.template operator()<LOGR>() with the runtime round size */
#define ROUND_SWITCH(logR, ...) \
    switch (logR) { \
    case 4: { constexpr int LR = 4; __VA_ARGS__ } break; \
    case 3: { constexpr int LR = 3; __VA_ARGS__ } break; \
    case 2: { constexpr int LR = 2; __VA_ARGS__ } break; \
    default: { constexpr int LR = 1; __VA_ARGS__ } break; }

/* limbs and planes as global-space pointers: an address read from memory is generic to the compiler, and a generic
 * (flat) access counts against the LDS counter too */
typedef const __attribute__((address_space(1))) uint64_t *GLimb;
typedef __attribute__((address_space(1))) double *GPlane;

/* The tile in LDS, padded: element e at word e + e / 32 (LDS_WORDS(T) words for T elements).  A round over the lowest
 * row bits of a contiguous tile has lanes 16 elements apart, which unpadded all hit the same bank pair; padded, every
 * round, the linear staging and the strided tiles' rounds spread over all banks.  For a group's slots
 * e = eb + j 2^L the padded index is pad(eb) + a compile-time multiple of j (L >= 5, or the slot bits below bit 5 with
 * eb's bits clear), so the offsets stay immediate. */
#define LDS_WORDS(T) ((T) + ((T) >> 5))
struct SwzLds {
    double *p;
    __device__ __forceinline__ double &operator[](uint32_t e) const { return p[e + (e >> 5)]; }
    __device__ __forceinline__ double &at(uint32_t pe) const { return p[pe]; }   /* an index padded already */
};

/* w^E for a 32-bit exponent fraction E from the four-level table (bq[k 2^8 + x] = w32^(x 2^(8k))), balanced
 * (|result| <= p/2 + 1) */
__device__ __forceinline__ double bq_twiddle(const double2 *bq, uint32_t E, double p, double pinv)
{
    constexpr uint32_t M = (1u << NTTM_BQ_LOG) - 1;
    double x = bq[(3 << NTTM_BQ_LOG) + (E >> 24)].x;
    const double2 t2 = bq[(2 << NTTM_BQ_LOG) + ((E >> 16) & M)];
    const double2 t1 = bq[(1 << NTTM_BQ_LOG) + ((E >> 8) & M)];
    const double2 t0 = bq[E & M];
    x = mul_shoup(x, t2.x, t2.y, p);
    x = mul_shoup(x, t1.x, t1.y, p);
    x = mul_shoup(x, t0.x, t0.y, p);
    return reduce(x, p, pinv);
}
#endif
