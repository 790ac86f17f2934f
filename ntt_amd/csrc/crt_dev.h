/* crt_dev.h - device code of the CRT that more than one kernel uses: one-bit carry maps, the 64-limb adder's carry out
 * and the base-10^18 digits of a coefficient. */
#ifndef NTTM_CRT_DEV_H
#define NTTM_CRT_DEV_H
#include "internal.h"

#define CRT_CTL_WORDS 4                  /* control words before the block status words (16-byte aligned) */
/* block status word: map (2 bits) | error for cin 0 << 2 | error for cin 1 << 3 | first of product << 5 */
#define CRT_ST_E0 (1u << 2)
#define CRT_ST_E1 (1u << 3)
#define CRT_ST_FIRST (1u << 5)

__device__ __forceinline__ uint32_t map_apply(uint32_t f, uint32_t c) { return (f >> c) & 1u; }
/* (g o f)(c) = g(f(c)) for maps {0,1} -> {0,1} */
__device__ __forceinline__ uint32_t map_compose(uint32_t g, uint32_t f)
{
    return map_apply(g, f & 1u) | (map_apply(g, (f >> 1) & 1u) << 1);
}
/* carry out of X + Y + cin over 64 bits */
__device__ __forceinline__ uint32_t add_cout(uint64_t X, uint64_t Y, uint32_t cin)
{
    const uint64_t s = X + Y;
    const uint32_t c1 = s < X;
    const uint64_t s2 = s + cin;
    return c1 | (uint32_t)(s2 < s);
}

template <int NP>
__device__ __forceinline__ void crt_digits(const CrtConst &cc, const double *r, uint64_t *d)
{
    /* Garner's digits t_i in [0, p_i), for residues |r_i| < p_i (balanced or canonical):
     *   t_0 = r_0 mod p_0;  t_i = (r_i - t_0 - sum_{0<j<i} t_j (p_0 ... p_{j-1})) (p_0 ... p_{i-1})^-1 mod p_i.
     * The primes differ by less than 2^40, so t_j < p_j <= 1.0007 p_i: each t_j m_ij (|m_ij| <= p_i / 2) stays within
     * the Barrett product's bound (|result| < 0.63 p_i), the sum r_i - acc within 4 p_i (one reduce), and no
     * intermediate reduction of t_j mod p_i is needed. */
    uint64_t t[NP];
    double td[NP];                                       /* the same digits as doubles (exact, below 2^50) */
    const double p0 = cc.pk[0].p;
    { const double v = r[0] < 0.0 ? r[0] + p0 : r[0]; td[0] = v; t[0] = f64_to_u52(v); }
#pragma unroll
    for (int i = 1; i < NP; i++) {
        const double p = cc.pk[i].p, pinv = cc.pk[i].pinv;
        double acc = td[0];
#pragma unroll
        for (int j = 1; j < i; j++) acc += mul_barrett(td[j], cc.mmod[i][j], p, pinv);
        const double dd = reduce(r[i] - acc, p, pinv);
        double ti = mul_barrett(dd, cc.cinv[i], p, pinv);
        ti = ti < 0.0 ? ti + p : ti;
        td[i] = ti; t[i] = f64_to_u52(ti);
    }
    /* X = sum_i t_i M_i with M_i = p_0 ... p_{i-1} = sum_j m_ij B^j: every t_i m_ij = a_ij B + b_ij (mulmod_b), then
     * base-B columns col_j = sum_i b_ij + sum_i a_i(j-1) (+ t_0 in column 0) with their small carries.  Column sums
     * stay below NP B + NP 2^50 < 2^62; X < 2^(50 NP) bounds the top digit (NP = 3: < 2^31, NP = 4: < 2^21). */
    uint64_t acc[NP + 1];
#pragma unroll
    for (int j = 0; j <= NP; j++) acc[j] = 0;
    acc[0] = t[0];
#pragma unroll
    for (int i = 1; i < NP; i++)
#pragma unroll
        for (int j = 0; j < i; j++) {
            uint64_t ah, bl;
            mulmod_b(t[i], cc.mb[i][j], cc.mbp[i][j], &ah, &bl);
            acc[j] += bl; acc[j + 1] += ah;
        }
    uint64_t c = 0;
#pragma unroll
    for (int j = 0; j < NP - 1; j++) {
        /* column j holds NP - 1 - j terms below B, the rest (a's, t_0, the carry in) below 2^52 < B: its carry is at
         * most NP - 1 - j */
        uint64_t v = acc[j] + c;
        c = 0;
#pragma unroll
        for (int k = 0; k < NP - 1 - j; k++) { const int ge = v >= NTTM_B; v = ge ? v - NTTM_B : v; c += (uint64_t)ge; }
        d[j] = v;
    }
    d[NP - 1] = acc[NP - 1] + c;
}
#endif
