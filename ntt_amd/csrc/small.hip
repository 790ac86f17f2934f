/* small.hip - whole products in one kernel: every transform of up to 2^12 points, the pointwise product, the CRT and
 * the carries of a product inside one workgroup.
 *
 * A product of up to 4096 coefficients is three transforms per prime over at most 32 KiB of LDS per prime: the residues
 * of every prime fit a workgroup's LDS at once, so nothing but the operands' limbs and the product's own limbs crosses
 * HBM and no other launch follows.  (In separate launches a product of this size took three: the double-fused pass,
 * the CRT with its planes through HBM, the carry scan and its fix.)
 *
 * A block holds a tile of T points per prime, H = T / n products of n points, PTS points per thread: T / PTS threads per
 * prime, at least 64, so a wave works for one prime (64: exactly one, whose rounds then need no barrier).
 *   - transforms: the rounds of k_fused2 on each prime's tile; B's transform stays in registers; the inverse ends in LDS in
 *     natural order;
 *   - digits: each coefficient's residues are replaced in place by its base-10^18 digits (crt_digits);
 *   - limbs: words of 64 limbs, one per wave and step.  Product limbs run to n + 2 (n coefficients, two digits more), so
 *     a product has W = n / 64 + 1 words: 65 at most, and a block's 66 at most (two products of 2^11 points).  A word's
 *     carry chain is one addition of its ballot masks (crt.hip), and the chain over up to 65 words the same once more:
 *     lane l holds word l's carry out for either carry in, a product's last word passes nothing on.  Blocks of more words
 *     have a chain per product.
 * Bound by vector issue and, with one block a CU at n = 4096, by latency: 4606 vector instructions a wave at 69% of the issue
 * rate there (three primes, 8192 products 1.23 ms), 4323 at 87% at n = 1024 (32768 products 0.94 ms). */
#include <string.h>
#include "internal.h"
#include "rounds.h"
#include "crt_dev.h"
#include "segrule.h"

int nttm_ncu(void);

#define SMALL_LOG_MIN 7
#define SMALL_LOG_MAX 12

struct SmallArgs {
    const LoadDesc *ld; const CrtDesc *cd;      /* cnt products in device memory, or null: the one product below */
    LoadDesc ld1; CrtDesc cd1;
    uint64_t cnt;
    uint64_t *ncn;                              /* or null: the normalized lengths, bit 63 set for a carry beyond the top */
    uint32_t *ctl;                              /* one product: words 0, 1 written (1: the error); else word 1 gets it or-ed in */
    uint64_t *stamps;                           /* or null: the device clock at the four phase boundaries */
    const double2 *stage[NTTM_MAX_PRIMES], *istage[NTTM_MAX_PRIMES];
    double2 ninv[NTTM_MAX_PRIMES];
    CrtConst cc;
};

/* a barrier between the threads of one prime: the whole block's, or (one wave per prime) none but the compiler's, since a
 * wave's LDS operations complete in order */
template <bool WAVE> __device__ __forceinline__ void prime_barrier()
{
    if (WAVE) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else __syncthreads();
}

template <int LOGN, int NP, int TL = (LOGN > 10 ? LOGN : 10), int PTS = 16>
__global__ __launch_bounds__((NP << TL) / PTS) void k_small(SmallArgs a)
{
    constexpr int T = 1 << TL, N = 1 << LOGN, H = T / N;
    constexpr int NT = T / PTS, NTH = NP * NT, NW = NTH / 64;        /* threads per prime and block, waves */
    constexpr int SW = LOGN < 8 ? LOGN : LOGN == 11 && PTS == 8 ? 9 : 8;   /* stages whose twiddles are kept in LDS */
    constexpr int WPP = N / 64 + 1, NWORD = H * WPP, IT = (NWORD + NW - 1) / NW;
    constexpr bool WAVE = NT == 64;
    constexpr int MAXR = PTS == 16 ? 4 : PTS == 8 ? 3 : 2, NR = (LOGN + MAXR - 1) / MAXR;   /* rounds, of at most MAXR bits */
    constexpr int CH = NWORD <= 65 ? 1 : H;                          /* word chains: all products in one, or one each */
    static_assert(NWORD <= 65 || WPP <= 65, "a word chain is one 64-bit addition and its carry out");
    static_assert(PTS == 16 || PTS == 8 || PTS == 4, "rounds of 4, 3 or 2 bits");
    static_assert(LOGN <= SW || LOGN - LOGN / NR <= SW, "only the top round's stages lie above the LDS table");
    static_assert(NT % 64 == 0, "a wave works for one prime");
    typedef __attribute__((address_space(1))) uint64_t *GOut;
    struct Prod { const uint64_t *a, *b, *x; uint64_t *c; uint32_t na, nb, nx, nc, ncoef, trunc; };
    __shared__ double pl[NP][LDS_WORDS(T)];
    __shared__ double2 stw[NP][1 << SW];
    __shared__ Prod sp[H];
    __shared__ uint64_t sgx[NWORD], sgy[NWORD];
    __shared__ uint32_t slen[H], serr[H];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t pi = __builtin_amdgcn_readfirstlane((uint32_t)tid / NT);
    const int t = tid & (NT - 1);
    const uint64_t prod0 = (uint64_t)blockIdx.x * H;
    if (a.stamps) stamp_clock(a.stamps);

    const double2 *gst = a.stage[pi];
#pragma unroll
    for (int i = 0; i < ((1 << SW) + NT - 1) / NT; i++) {
        const int e = i * NT + t;
        if (e < (1 << SW)) stw[pi][e] = gst[e];
    }
    if (tid < H) {
        Prod q; q.a = q.b = q.x = (const uint64_t *)gst; q.c = nullptr;      /* a dead product reads no limb: any address */
        q.na = q.nb = q.nx = q.nc = q.ncoef = q.trunc = 0;
        const uint64_t i = prod0 + tid;
        if (i < a.cnt) {
            LoadDesc l = a.ld1; CrtDesc c = a.cd1;
            if (a.ld) { l = a.ld[i]; c = a.cd[i]; }
            q.a = l.a; q.b = l.b; q.na = (uint32_t)l.na; q.nb = (uint32_t)l.nb;
            if (c.x && c.nx) { q.x = c.x; q.nx = (uint32_t)c.nx; }
            q.c = c.c; q.nc = (uint32_t)c.nc; q.ncoef = (uint32_t)c.ncoef; q.trunc = c.trunc != 0;
        }
        sp[tid] = q; slen[tid] = 0; serr[tid] = 0;
    }
    __syncthreads();

    /* ---- the cyclic convolution modulo this wave's prime, into pl[pi] in natural order */
    const double p = a.cc.pk[pi].p, pinv = a.cc.pk[pi].pinv;
    {
        const SwzLds xs{pl[pi]};
        const double2 *lt = stw[pi];
        const GTab gf(a.stage[pi]), gi(a.istage[pi]);
        PassPos pp; pp.m = LOGN; pp.logw = 0; pp.lo = 0; pp.nthr = NT; pp.t = t;
        int s_lo, logR;
        round_split(LOGN, 0, &s_lo, &logR, false, MAXR);
        uint64_t raw[2][PTS];
        uint32_t in[2] = {0, 0};                                     /* bit sl: the slot lies inside the operand */
#pragma unroll
        for (int w = 0; w < 2; w++)                                  /* B's limbs, then A's: all requested at once */
            ROUND_SWITCH(logR, for_slots<LR, PTS>(pp, s_lo, [&](int sl, uint32_t, uint32_t o, uint32_t, uint32_t) {
                const Prod &q = sp[H > 1 ? o >> LOGN : 0];
                const uint32_t k = o & (N - 1), nl = w ? q.na : q.nb;
                const bool inside = k < nl;
                raw[w][sl] = ((GLimb)(w ? q.a : q.b))[inside ? k : 0];
                in[w] |= (uint32_t)inside << sl;
            });)
        double v[PTS], bv[PTS];
        const double2 ninv = a.ninv[pi];
#pragma unroll
        for (int w = 0; w < 2; w++) {
            if (w) prime_barrier<WAVE>();                            /* B's last LDS reads before A's first writes */
#pragma unroll
            for (int sl = 0; sl < PTS; sl++) {
                double x = (in[w] >> sl) & 1 ? limb_to_res(raw[w][sl], p, pinv) : 0.0;
                if (w == 0) x = mul_shoup(x, ninv.x, ninv.y, p);
                v[sl] = x;
            }
#pragma unroll
            for (int i = 0; i < NR; i++) {                           /* top bits first; the last round stays in registers */
                round_split(LOGN, i, &s_lo, &logR, false, MAXR);
                if (i > 0) {
                    prime_barrier<WAVE>();
                    ROUND_SWITCH(logR, for_slots<LR, PTS, true>(pp, s_lo, [&](int sl, uint32_t e, uint32_t, uint32_t, uint32_t) {
                        v[sl] = xs.at(e); });)
                }
                if (i == 0 && LOGN > SW) { ROUND_SWITCH(logR, round_compute<LR, false, PTS>(v, pp, s_lo, gf, p, pinv);) }
                else { ROUND_SWITCH(logR, round_compute<LR, false, PTS, LTab>(v, pp, s_lo, lt, p, pinv);) }
                if (i + 1 < NR)
                    ROUND_SWITCH(logR, for_slots<LR, PTS, true>(pp, s_lo, [&](int sl, uint32_t e, uint32_t, uint32_t, uint32_t) {
                        xs.at(e) = v[sl]; });)
            }
            if (w == 0) {
#pragma unroll
                for (int sl = 0; sl < PTS; sl++) bv[sl] = v[sl];
            }
        }
        if (a.stamps) stamp_clock(a.stamps + 1);
#pragma unroll
        for (int sl = 0; sl < PTS; sl++) v[sl] = mul_barrett(v[sl], bv[sl], p, pinv);
#pragma unroll
        for (int i = 0; i < NR; i++) {                               /* bit 0 first; round 0 has the layout in v */
            round_split(LOGN, i, &s_lo, &logR, true, MAXR);
            if (i > 0) {
                prime_barrier<WAVE>();
                ROUND_SWITCH(logR, for_slots<LR, PTS, true>(pp, s_lo, [&](int sl, uint32_t e, uint32_t, uint32_t, uint32_t) {
                    v[sl] = xs.at(e); });)
            }
            if (i == NR - 1 && LOGN > SW) { ROUND_SWITCH(logR, round_compute<LR, true, PTS>(v, pp, s_lo, gi, p, pinv, i > 0, i + 1 < NR);) }
            else { ROUND_SWITCH(logR, round_compute_mirror<LR, PTS>(v, pp, s_lo, lt, p, pinv, i > 0, i + 1 < NR);) }
            ROUND_SWITCH(logR, for_slots<LR, PTS, true>(pp, s_lo, [&](int sl, uint32_t e, uint32_t, uint32_t, uint32_t) {
                xs.at(e) = v[sl]; });)
        }
    }

    /* ---- the product's x limbs are requested; the residues become digits in place */
    uint64_t xk[IT], xp[IT];
#pragma unroll
    for (int i = 0; i < IT; i++) {
        const int w = wave + i * NW;
        const int h = w / WPP;
        const uint32_t k = (uint32_t)(w - h * WPP) * 64 + lane;
        xk[i] = xp[i] = 0;
        if (w < NWORD) {
            const Prod &q = sp[h];
            if (k < q.nx && k < q.nc) xk[i] = ((GLimb)q.x)[k];
            if (lane == 0 && k >= 1 && k - 1 < q.nx) xp[i] = ((GLimb)q.x)[k - 1];
        }
    }
    __syncthreads();
    if (a.stamps) stamp_clock(a.stamps + 2);
    for (int e = tid; e < T; e += NTH) {
        const bool live = (uint32_t)(e & (N - 1)) < sp[H > 1 ? e >> LOGN : 0].ncoef;
        double r[NP];
        uint64_t d[NP];
#pragma unroll
        for (int j = 0; j < NP; j++) r[j] = live ? pl[j][e + (e >> 5)] : 0.0;
        crt_digits<NP>(a.cc, r, d);
#pragma unroll
        for (int j = 0; j < NP; j++) pl[j][e + (e >> 5)] = __longlong_as_double((long long)d[j]);
    }
    __syncthreads();

    /* ---- limbs: v_k = sum_j d_j[k - j] + x_k < NP B + 2^31, w_k = v_k - q_k B + q_(k-1) */
    auto digit = [&](int h, int j, int k) -> uint64_t {              /* d_j of coefficient k of product h */
        const int e = h * N + k;
        return k >= 0 && k < N ? (uint64_t)__double_as_longlong(pl[j][e + (e >> 5)]) : 0;
    };
    auto vsum = [&](int h, int k, uint64_t x) -> uint64_t {
        uint64_t v = x;
#pragma unroll
        for (int j = 0; j < NP; j++) v += digit(h, j, k - j);
        return v;
    };
    auto quot = [](uint64_t v) -> uint32_t {
        uint32_t q = 0;
#pragma unroll
        for (int c = 1; c <= NP; c++) q += v >= (uint64_t)c * NTTM_B;
        return q;
    };
    uint64_t wv[IT], GX[IT], GY[IT];
    uint32_t ql[IT];
#pragma unroll
    for (int i = 0; i < IT; i++) {
        const int w = wave + i * NW;
        wv[i] = GX[i] = GY[i] = 0; ql[i] = 0;
        if (w < NWORD) {
            const int h = w / WPP, k = (w - h * WPP) * 64 + lane;
            const int nc = (int)sp[h].nc;
            const uint64_t v = k < nc ? vsum(h, k, xk[i]) : 0;
            const uint32_t q = quot(v);
            uint32_t qp = __shfl_up(q, 1, 64);
            if (lane == 0) qp = k >= 1 && k <= nc ? quot(vsum(h, k - 1, xp[i])) : 0u;
            wv[i] = v - (uint64_t)q * NTTM_B + qp;
            if (k >= nc) wv[i] = 0;
            ql[i] = q;
            const uint64_t g = __ballot(wv[i] >= NTTM_B), pr = __ballot(wv[i] == NTTM_B - 1);
            GX[i] = g; GY[i] = g | pr;
            if (lane == 0) { sgx[w] = g; sgy[w] = g | pr; }
        }
    }
    __syncthreads();
    /* the carry into every word of the block: bit w of its chain's CI (word 64: cout) */
    uint64_t CI[CH]; uint32_t cout64[CH];
#pragma unroll
    for (int h = 0; h < CH; h++) {
        constexpr int CW = CH == 1 ? NWORD : WPP;                    /* words of a chain */
        uint32_t f0 = 0, f1 = 0;
        if (lane < CW && lane % WPP != WPP - 1) {
            f0 = add_cout(sgx[h * CW + lane], sgy[h * CW + lane], 0); f1 = add_cout(sgx[h * CW + lane], sgy[h * CW + lane], 1);
        }
        const uint64_t G = __ballot(f0 != 0), GP = __ballot(f1 != 0), S = G + GP;
        CI[h] = S ^ G ^ GP; cout64[h] = S < G;
    }
#pragma unroll
    for (int i = 0; i < IT; i++) {
        const int w = wave + i * NW;
        if (w < NWORD) {
            const int h = w / WPP, k = (w - h * WPP) * 64 + lane;
            const int nc = (int)sp[h].nc;
            uint64_t ci = CI[0]; uint32_t co = cout64[0];
#pragma unroll
            for (int j = 1; j < CH; j++) if (h == j) { ci = CI[j]; co = cout64[j]; }
            const int cw = CH == 1 ? w : w - h * WPP;
            const uint32_t c = cw < 64 ? (uint32_t)(ci >> cw) & 1u : co;
            const uint64_t S = GX[i] + GY[i] + c, CB = S ^ GX[i] ^ GY[i];      /* bit b: the carry into bit b */
            const uint32_t oin = (uint32_t)(CB >> lane) & 1u;
            const uint32_t oout = lane == 63 ? add_cout(GX[i], GY[i], c) : (uint32_t)(CB >> (lane + 1)) & 1u;
            const uint64_t limb = wv[i] + oin - (oout ? NTTM_B : 0);
            if (k < nc) ((GOut)sp[h].c)[k] = limb;
            const uint64_t nz = __ballot(k < nc && limb != 0);
            if (nz && lane == 0) atomicMax(&slen[h], (uint32_t)(k + 64 - __clzll((long long)nz)));
            if (k + 1 == nc && !sp[h].trunc) {                       /* the last limb: nothing may remain beyond it */
                uint64_t extra = ql[i] + oout;
#pragma unroll
                for (int e = 1; e < NP; e++)
#pragma unroll
                    for (int j = e; j < NP; j++) extra += digit(h, j, k + e - j);
                serr[h] = extra != 0;
            }
        }
    }
    __syncthreads();
    if (tid < H && prod0 + tid < a.cnt) {
        const uint32_t err = serr[tid];
        if (a.ncn) a.ncn[prod0 + tid] = slen[tid] | (uint64_t)err << 63;
        if (!a.ld) { a.ctl[0] = 0; a.ctl[1] = err; }
        else if (err && a.ctl) atomicOr(a.ctl + 1, 1u);
    }
    if (a.stamps) stamp_clock(a.stamps + 3);
}

/* the points of the kernel for a transform of 2^logn points (0: too long) */
int nttm_small_log(int logn) { return logn > SMALL_LOG_MAX ? 0 : logn < SMALL_LOG_MIN ? SMALL_LOG_MIN : logn; }

/* cnt products of at most 2^logn coefficients (logn from nttm_small_log), from device descriptors, or (ld null) the one
 * product ld1, cd1, whose flags go to ctl's two words (device or pinned host memory).  stage / istage: the forward and
 * inverse stage tables of the np primes; ninv: 2^-logn modulo each */
int nttm_run_small(int np, int logn, const LoadDesc *ld, const CrtDesc *cd, const LoadDesc *ld1, const CrtDesc *cd1,
                   uint64_t cnt, uint64_t *ncn, uint32_t *ctl, const TwTables *fwd, const TwTables *inv, const double2 *ninv,
                   const CrtConst &cc, hipStream_t s, double alg_bytes, uint64_t *stamps)
{
    if (np < 3 || np > NTTM_MAX_PRIMES || logn < SMALL_LOG_MIN || logn > SMALL_LOG_MAX || !cnt || (!ld != !cd) ||
        (!ld && (!ld1 || !cd1 || cnt != 1 || !ctl)))
        return nttm_fail(NTTM_EINVAL, "internal: small products");
    SmallArgs a; memset(&a, 0, sizeof a);
    a.ld = ld; a.cd = cd; a.cnt = cnt; a.ncn = ncn; a.ctl = ctl; a.stamps = stamps; a.cc = cc;
    if (ld1) a.ld1 = *ld1;
    if (cd1) a.cd1 = *cd1;
    for (int i = 0; i < np; i++) { a.stage[i] = fwd[i].stage; a.istage[i] = inv[i].stage; a.ninv[i] = ninv[i]; }
    /* Few products: a block each and 4 or 8 points a thread, so that more waves share a product's chain of rounds; many:
     * 16 points, and at least a wave per prime (12 waves a block at 2^11 points, whose 6 of one product leave room for no
     * second block: waves of 144 registers start on the same SIMDs).  The line is 2^11 points a CU, one block at 2^11.
     * A plan's replay, us, many / few: 2^7 points 1 product 22 / 18, 4096 32 / 27, 8192 42 / 43; 2^9 256 26 / 22, 2048 44 / 44;
     * 2^10 1 24 / 21, 512 33 / 31, 1024 45 / 62; 2^11 1 38 / 26, 256 43 / 29, 512 46 / 52, 8192 572 / 668 (6 waves of
     * 16 points: 789).  One 64 x 64 limb call 35 -> 27 us, 1000 x 1000 46 -> 40. */
    const bool few = small_few(cnt, logn, nttm_ncu());
    const int tl = few ? (logn < 8 ? 8 : logn) : logn == 11 ? 12 : logn > 10 ? logn : 10, h = 1 << (tl - logn);
    const int pts = !few ? 16 : tl <= 8 ? 4 : tl <= 11 ? 8 : 16;
    const uint64_t blocks = (cnt + h - 1) / h;
    if (blocks > 0x7fffffffULL) return nttm_fail(NTTM_EINVAL, "internal: too many small products");
    const dim3 grid((unsigned)blocks), blk((unsigned)((np << tl) / pts));
    prof_begin("k_small", alg_bytes, s);
#define SMALL_LAUNCH(L, TL, P) \
    if (logn == L && tl == TL && pts == P) { \
        if (np == 3) hipLaunchKernelGGL((k_small<L, 3, TL, P>), grid, blk, 0, s, a); \
        else hipLaunchKernelGGL((k_small<L, 4, TL, P>), grid, blk, 0, s, a); \
    }
    SMALL_LAUNCH(7, 8, 4) SMALL_LAUNCH(8, 8, 4) SMALL_LAUNCH(9, 9, 8) SMALL_LAUNCH(10, 10, 8) SMALL_LAUNCH(11, 11, 8)
    SMALL_LAUNCH(12, 12, 16)
    SMALL_LAUNCH(10, 10, 16) SMALL_LAUNCH(7, 10, 16) SMALL_LAUNCH(8, 10, 16) SMALL_LAUNCH(9, 10, 16) SMALL_LAUNCH(11, 12, 16)
#undef SMALL_LAUNCH
    prof_end(s);
    return nttm_hip_check(hipGetLastError(), "k_small launch");
}

/* ---- uneven products in segments of the result ------------------------------------------------------------------------------
 * A product of a long operand by one of blen limbs, 2^12 points at a time: limbs [s, s + S) of the result need coefficients
 * s - 4 .. s + S - 1 (three digits below, and one limb more for the quotient), which are coefficients blen - 1 .. of the
 * cyclic convolution of the short operand with the long one's limbs from s - 4 - (blen - 1) on, S = 4093 - blen rounded down
 * to whole words.  A workgroup keeps the short operand's transforms in registers and walks several (the descriptor's
 * `over`) consecutive segments:
 * forward, pointwise product and inverse of every prime, digits and limbs as in k_small, so that nothing but operand and
 * result limbs crosses memory.  A segment is one block of the carry launch.  The overlapping limbs are transformed twice:
 * the rules that choose it (choose_segments, batch_segments) weigh that.
 * Bound by vector issue (64% of the issue rate) and latency at one workgroup a CU (12 waves, 115 KB of LDS): 13 us for the short operand and 26 to 31
 * for a segment of 2048 to 4032 limbs.  Through passes of 2^13 points and more, us, before / now: 500 products of
 * 8000 x 500 limbs 458 / 210, of 60000 x 1000 1743 / 1178, 8 of 60000 x 300 72 / 50; one of 1000000 x 1000 116 / 88,
 * of 20000000 x 300 2660 / 625 (in pieces 1080). */
struct SegArgs {
    const LoadDesc *ld; const CrtDesc *cd;      /* nprod products in device memory, or null: the one product below */
    LoadDesc ld1; CrtDesc cd1;
    uint64_t nprod;
    uint32_t *status, *ctl;
    uint64_t *stamps;                           /* or null: block 0's clock at its start, after B's transforms and at its end, and
                                                 * the time it spent on digits, limbs and carries */
    const double2 *stage[NTTM_MAX_PRIMES], *istage[NTTM_MAX_PRIMES];
    double2 ninv[NTTM_MAX_PRIMES];
    CrtConst cc;
};
template <int NP>
__global__ __launch_bounds__(NP * 256) void k_segments(SegArgs a)
{
    constexpr int LOGN = SMALL_LOG_MAX, N = 1 << LOGN, PTS = 16, NT = N / PTS, NTH = NP * NT, NW = NTH / 64, SW = 8, NR = 3;
    constexpr int IT = (63 + NW - 1) / NW;                           /* words of a wave */
    typedef __attribute__((address_space(1))) uint64_t *GOut;
    __shared__ double pl[NP][LDS_WORDS(N)];
    __shared__ double2 stw[NP][1 << SW];
    __shared__ uint64_t sgx[64], sgy[64];
    __shared__ uint32_t s_prod, s_err;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t pi = __builtin_amdgcn_readfirstlane((uint32_t)tid / NT);
    const int t = tid & (NT - 1);
    if (a.stamps) stamp_clock(a.stamps);
    if (blockIdx.x == 0 && tid == 0) { a.ctl[0] = 0; a.ctl[1] = 0; }
    stw[pi][t] = a.stage[pi][t];                                     /* (256 threads and entries a prime) */
    if (tid == 0) {
        uint64_t lo = 0, hi = a.cd ? a.nprod - 1 : 0;                /* the product whose workgroups hold this one */
        while (lo < hi) { const uint64_t mid = (lo + hi + 1) >> 1; if (a.cd[mid].tn <= blockIdx.x) lo = mid; else hi = mid - 1; }
        s_prod = (uint32_t)lo;
    }
    __syncthreads();
    LoadDesc l = a.ld1; CrtDesc d = a.cd1;
    if (a.ld) { const uint32_t prod = __builtin_amdgcn_readfirstlane(s_prod); l = a.ld[prod]; d = a.cd[prod]; }
    const int nb = (int)l.nb, S = (int)d.step, nw = S >> 6;
    const uint32_t per = (uint32_t)d.over, nseg = (uint32_t)((d.nc + S - 1) / S), seg0 = (blockIdx.x - (uint32_t)d.tn) * per;
    const uint32_t seg1 = seg0 + per < nseg ? seg0 + per : nseg;

    const double p = a.cc.pk[pi].p, pinv = a.cc.pk[pi].pinv;
    const SwzLds xs{pl[pi]};
    const double2 *lt = stw[pi];
    const GTab gf(a.stage[pi]), gi(a.istage[pi]);
    PassPos pp; pp.m = LOGN; pp.logw = 0; pp.lo = 0; pp.nthr = NT; pp.t = t;
    int s_lo, logR;
    double v[PTS], bv[PTS];
    uint64_t raw[PTS];
    uint32_t in = 0;                                                 /* bit sl: the slot lies inside the operand */
    auto request = [&](const uint64_t *src, uint64_t n, int64_t base) {
        in = 0;
        for_slots<4, PTS>(pp, 8, [&](int sl, uint32_t, uint32_t o, uint32_t, uint32_t) {
            const uint64_t k = (uint64_t)(base + o);                 /* (before the first limb: beyond any length) */
            const bool inside = k < n;
            raw[sl] = ((GLimb)src)[inside ? k : 0];
            in |= (uint32_t)inside << sl;
        });
    };
    auto forward = [&]() {                                           /* of raw, into v in the last round's layout */
#pragma unroll
        for (int sl = 0; sl < PTS; sl++) v[sl] = (in >> sl) & 1 ? limb_to_res(raw[sl], p, pinv) : 0.0;
#pragma unroll
        for (int i = 0; i < NR; i++) {
            round_split(LOGN, i, &s_lo, &logR, false, 4);
            if (i > 0) {
                __syncthreads();
                for_slots<4, PTS, true>(pp, s_lo, [&](int sl, uint32_t e, uint32_t, uint32_t, uint32_t) { v[sl] = xs.at(e); });
            }
            if (i == 0) round_compute<4, false, PTS>(v, pp, s_lo, gf, p, pinv);
            else round_compute<4, false, PTS, LTab>(v, pp, s_lo, lt, p, pinv);
            if (i + 1 < NR) for_slots<4, PTS, true>(pp, s_lo, [&](int sl, uint32_t e, uint32_t, uint32_t, uint32_t) { xs.at(e) = v[sl]; });
        }
    };
    auto first = [&](uint32_t seg) { return (int64_t)seg * S - 4 - (nb - 1); };   /* the coefficient of the window's element 0 */
    request(l.b, l.nb, 0);
    forward();
    const double2 ninv = a.ninv[pi];
#pragma unroll
    for (int sl = 0; sl < PTS; sl++) bv[sl] = mul_shoup(v[sl], ninv.x, ninv.y, p);
    const bool clk = a.stamps && blockIdx.x == 0;
    uint64_t crt_ticks = 0;
    if (clk) stamp_clock(a.stamps + 1);

    __syncthreads();                                                 /* B's last LDS reads before A's first writes */
    for (uint32_t seg = seg0; seg < seg1; seg++) {
        /* opaque to the compiler, which otherwise keeps every twiddle and address of the loop in registers it has not got */
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63;
        pp.t = tid & (NT - 1);
        request(l.a, l.na, first(seg));
        forward();
#pragma unroll
        for (int sl = 0; sl < PTS; sl++) v[sl] = mul_barrett(v[sl], bv[sl], p, pinv);
#pragma unroll
        for (int i = 0; i < NR; i++) {                               /* bit 0 first; round 0 has the layout in v */
            round_split(LOGN, i, &s_lo, &logR, true, 4);
            if (i > 0) {
                __syncthreads();
                for_slots<4, PTS, true>(pp, s_lo, [&](int sl, uint32_t e, uint32_t, uint32_t, uint32_t) { v[sl] = xs.at(e); });
            }
            if (i == NR - 1) round_compute<4, true, PTS>(v, pp, s_lo, gi, p, pinv, true, false);
            else round_compute_mirror<4, PTS>(v, pp, s_lo, lt, p, pinv, i > 0, true);
            for_slots<4, PTS, true>(pp, s_lo, [&](int sl, uint32_t e, uint32_t, uint32_t, uint32_t) { xs.at(e) = v[sl]; });
        }
        /* the segment's x limbs are requested, the next one's operand limbs drawn into the L2 (a word of every line; in registers
         * they would be spilled); residues become digits in place */
        const uint64_t s0 = (uint64_t)seg * S;
        uint64_t xk[IT], xp[IT];
#pragma unroll
        for (int i = 0; i < IT; i++) {
            const int w = wave + i * NW;
            const uint64_t k = s0 + (uint64_t)w * 64 + lane;
            xk[i] = xp[i] = 0;
            if (w < nw) {
                if (k < d.nx && k < d.nc) xk[i] = ((GLimb)d.x)[k];
                if (lane == 0 && k >= 1 && k - 1 < d.nx) xp[i] = ((GLimb)d.x)[k - 1];
            }
        }

        uint64_t touch = 0;
        if (pi == 0 && seg + 1 < seg1) {
            const uint64_t k = (uint64_t)(first(seg + 1) + 16 * tid);
            touch = ((GLimb)l.a)[k < l.na ? k : 0];
        }
        if (tid == 0) s_err = 0;
        __syncthreads();
        if (clk) crt_ticks -= wall_clock64();
        const int64_t c0 = first(seg);
        for (int e = tid; e < N; e += NTH) {
            if (e < nb - 1) continue;                                /* (wrapped coefficients: never read) */
            const bool live = (uint64_t)(c0 + e) < d.ncoef;
            double r[NP];
            uint64_t dg[NP];
#pragma unroll
            for (int j = 0; j < NP; j++) r[j] = live ? pl[j][e + (e >> 5)] : 0.0;
            crt_digits<NP>(a.cc, r, dg);
#pragma unroll
            for (int j = 0; j < NP; j++) pl[j][e + (e >> 5)] = __longlong_as_double((long long)dg[j]);
        }
        __syncthreads();
        /* limbs: coefficient k - j of limb k = s0 + u is element nb + 3 + u - j >= nb - 1 */
        auto digit = [&](int j, int u) -> uint64_t {
            const int e = nb + 3 + u;
            return (uint64_t)__double_as_longlong(pl[j][e + (e >> 5)]);
        };
        auto vsum = [&](int u, uint64_t x) -> uint64_t {
            uint64_t y = x;
#pragma unroll
            for (int j = 0; j < NP; j++) y += digit(j, u - j);
            return y;
        };
        auto quot = [](uint64_t y) -> uint32_t {
            uint32_t q = 0;
#pragma unroll
            for (int c = 1; c <= NP; c++) q += y >= (uint64_t)c * NTTM_B;
            return q;
        };
        uint64_t wv[IT], GX[IT], GY[IT];
        uint32_t ql[IT];
#pragma unroll
        for (int i = 0; i < IT; i++) {
            const int w = wave + i * NW, u = w * 64 + lane;
            wv[i] = GX[i] = GY[i] = 0; ql[i] = 0;
            if (w < nw) {
                const uint64_t k = s0 + u;
                const uint64_t y = k < d.nc ? vsum(u, xk[i]) : 0;
                const uint32_t q = quot(y);
                uint32_t qp = __shfl_up(q, 1, 64);
                if (lane == 0) qp = k >= 1 && k <= d.nc ? quot(vsum(u - 1, xp[i])) : 0u;
                wv[i] = y - (uint64_t)q * NTTM_B + qp;
                if (k >= d.nc) wv[i] = 0;
                ql[i] = q;
                const uint64_t g = __ballot(wv[i] >= NTTM_B), pr = __ballot(wv[i] == NTTM_B - 1);
                GX[i] = g; GY[i] = g | pr;
                if (lane == 0) { sgx[w] = g; sgy[w] = g | pr; }
            }
        }
        __syncthreads();
        /* the carry into every word for a carry of 0 (C0) and 1 (C1) into the segment; bit nw: out of it */
        uint64_t C0, C1;
        {
            uint32_t f0 = 0, f1 = 0;
            if (lane < nw) { f0 = add_cout(sgx[lane], sgy[lane], 0); f1 = add_cout(sgx[lane], sgy[lane], 1); }
            const uint64_t G = __ballot(f0 != 0), GP = __ballot(f1 != 0);
            C0 = (G + GP) ^ G ^ GP; C1 = (G + GP + 1) ^ G ^ GP;
        }
#pragma unroll
        for (int i = 0; i < IT; i++) {
            const int w = wave + i * NW, u = w * 64 + lane;
            if (w < nw) {
                const uint64_t k = s0 + u;
                const uint32_t c = (uint32_t)(C0 >> w) & 1u;
                const uint64_t CB = (GX[i] + GY[i] + c) ^ GX[i] ^ GY[i];      /* bit b: the carry into bit b */
                const uint32_t oin = (uint32_t)(CB >> lane) & 1u;
                const uint32_t oout = lane == 63 ? add_cout(GX[i], GY[i], c) : (uint32_t)(CB >> (lane + 1)) & 1u;
                if (k < d.nc) ((GOut)d.c)[k] = wv[i] + oin - (oout ? NTTM_B : 0);
                if (k + 1 == d.nc && !d.trunc) {                     /* the last limb: nothing may remain beyond it */
                    const uint32_t c1 = (uint32_t)(C1 >> w) & 1u;
                    const uint64_t CB1 = (GX[i] + GY[i] + c1) ^ GX[i] ^ GY[i];
                    const uint32_t o1 = lane == 63 ? add_cout(GX[i], GY[i], c1) : (uint32_t)(CB1 >> (lane + 1)) & 1u;
                    uint64_t extra = ql[i];
#pragma unroll
                    for (int e = 1; e < NP; e++)
#pragma unroll
                        for (int j = e; j < NP; j++) extra += digit(j, u + e - j);
                    s_err = (extra + oout ? CRT_ST_E0 : 0u) | (extra + o1 ? CRT_ST_E1 : 0u);
                }
            }
        }
        asm volatile("" :: "v"(touch));
        __syncthreads();                                             /* (the digits are read, s_err is stored) */
        if (tid == 0)
            a.status[d.first_block + seg] = ((uint32_t)(C0 >> nw) & 1u) | ((uint32_t)(C1 >> nw) & 1u) << 1 | s_err | (seg ? 0u : CRT_ST_FIRST);
        if (clk) crt_ticks += wall_clock64();
    }
    if (clk) { stamp_clock(a.stamps + 2); if (threadIdx.x == 0) a.stamps[3] = crt_ticks; }
}

/* limbs of a segment for a short operand of nb limbs (whole words; 0: too long a one) */
uint64_t nttm_seg_len(uint64_t nb) { return nb < 1 || nb > ((uint64_t)1 << SMALL_LOG_MAX) - 3 - 512 ? 0 : (((uint64_t)1 << SMALL_LOG_MAX) - 3 - nb) & ~(uint64_t)63; }
/* nprod products in segments, from device descriptors, or (ld null) the one product ld1, cd1: the longer operand as a, step =
 * nttm_seg_len(nb), over the segments of a workgroup, tn the product's first workgroup, first_block its first segment among the status
 * words.  The limbs are for a carry of 0 into every segment: nttm_crt_launch_carry(.., NTTM_CRT_SEGS) follows */
int nttm_run_segments(int np, const LoadDesc *ld, const CrtDesc *cd, const LoadDesc *ld1, const CrtDesc *cd1, uint64_t nprod,
                      uint64_t groups, const TwTables *fwd, const TwTables *inv, const double2 *ninv,
                      const CrtConst &cc, uint32_t *scratch, uint32_t *ctl, hipStream_t s, double alg_bytes, uint64_t *stamps)
{
    if (np < 3 || np > NTTM_MAX_PRIMES || !nprod || !groups || (!ld != !cd) || (!ld && (!ld1 || !cd1 || nprod != 1)) || !ctl)
        return nttm_fail(NTTM_EINVAL, "internal: products in segments");
    if (!ld && (!cd1->step || !cd1->over || cd1->step != nttm_seg_len(ld1->nb))) return nttm_fail(NTTM_EINVAL, "internal: segments of %llu limbs", (unsigned long long)cd1->step);
    if (groups > 0x7fffffffULL) return nttm_fail(NTTM_EINVAL, "internal: too many segments");
    SegArgs a; memset(&a, 0, sizeof a);
    a.ld = ld; a.cd = cd; a.nprod = nprod; a.status = scratch + CRT_CTL_WORDS; a.ctl = ctl; a.stamps = stamps; a.cc = cc;
    if (ld1) a.ld1 = *ld1;
    if (cd1) a.cd1 = *cd1;
    for (int i = 0; i < np; i++) { a.stage[i] = fwd[i].stage; a.istage[i] = inv[i].stage; a.ninv[i] = ninv[i]; }
    prof_begin("k_segments", alg_bytes, s);
    if (np == 3) hipLaunchKernelGGL(k_segments<3>, dim3((unsigned)groups), dim3(3 * 256), 0, s, a);
    else hipLaunchKernelGGL(k_segments<4>, dim3((unsigned)groups), dim3(4 * 256), 0, s, a);
    prof_end(s);
    return nttm_hip_check(hipGetLastError(), "k_segments launch");
}
