/* rounds.h - the radix rounds of the transform kernels on a tile held in registers and LDS (device code): slots and
 * groups of a thread, butterflies with lazy reduction, stage tables in global memory or LDS, the padded LDS layout. */
#ifndef NTTM_ROUNDS_H
#define NTTM_ROUNDS_H
#include "internal.h"
#include "radix.h"

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
 * The radix step of a group, and what of it is reduced: radix.h. */
#define PASS_PTS 16               /* points per thread of full tiles; tiles below 16 points use one thread */

template <int BITS>
__device__ __forceinline__ constexpr uint32_t brev_c(uint32_t j)
{
    uint32_t r = 0;
    for (int i = 0; i < BITS; i++) r |= ((j >> i) & 1u) << (BITS - 1 - i);
    return r;
}

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
