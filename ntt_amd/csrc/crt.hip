/* crt.hip - Chinese remaindering of the residue planes into base-10^18 limbs, with the carry resolved on the device.
 *
 * Coefficient k of the convolution is rebuilt from its np residues by Garner's mixed radix (modular steps in the
 * FP64 arithmetic of arith.h), and its value X = sum_i t_i p_0 ... p_{i-1} is split into np base-10^18 digits
 * d_0..d_{np-1} from the products of the t_i with the base-10^18 digits of the prime prefixes (mulmod_b), and
 *     limb_k = d_0[k] + d_1[k-1] + ... + d_{np-1}[k-np+1] + x_k + carry_k            (E/rns_mul.c:332-405)
 * The top digit is small (X < 2^(50 np) gives d_{np-1} < 2^31), so v_k = sum of the digits + x_k < np B + 2^31.  With
 * q_k = floor(v_k / B) <= np, r_k = v_k mod B and w_k = r_k + q_{k-1} (<= B + np - 1), the carry into limb k+1 is
 * q_k + o_k where
 * the overflow bit o_k = [w_k + o_{k-1} >= B] = g_k | (p_k & o_{k-1}), g_k = [w_k >= B], p_k = [w_k = B - 1]: a binary
 * carry-lookahead chain.  For 64 consecutive limbs it is resolved by one 64-bit addition of the ballot masks
 * X = G, Y = G | P (the carries into the bits of X + Y + cin are the o's, the textbook adder identity).  Words chain
 * inside a wave and waves inside a block; each block then stores its limbs for a carry in of 0 together with its
 * (cin -> cout) map of one bit.  A second launch (k_carry) finds each block's carry in from the maps before it and adds
 * 1 to the limbs of the blocks that receive one: the limbs for cin = 1 are those for cin = 0 plus one, a ripple through
 * the leading limbs equal to B - 1.  No block waits on another.
 * The reference instead ripples each 256-coefficient chunk on one thread of a wave64 ballot scan, writes a 4-limb spill
 * per stripe and merges the spills serially on the host or on one thread per product (E/rns_mul.c:452-470;
 * E/dbig.c:1007-1052).  The final carry beyond limb nc-1 must be zero; a non-zero one sets an error flag.
 */
#include <string.h>
#include "internal.h"
#include "crt_dev.h"
#include "rounds.h"

#define CRT_T 256
#define CRT_WIDE 8                       /* limbs per thread of a block (2048-limb blocks); groups of small products
                                            use 1 (256-limb blocks, less of a block idle past a product's end) */
#define CRT_RUNS 0                       /* in place of the limbs per thread: the blocks are k_inv_crt's runs, */
#define CRT_SEGS (-1)                    /* or k_segments' segments */
#define CRT_HALO 4                       /* digits of coefficients k0-4 .. k0-1: v_{k0-1} with four primes */
#define CRT_ID_MAP 0x2u                  /* one-bit carry maps: bit c = cout(cin = c); the identity is 0b10 */

struct CrtArgs {
    const CrtDesc *desc; uint64_t nprod; /* null: the one product `one` */
    CrtDesc one;
    uint32_t *status;                    /* one word per block (CRT_ST_*) */
    uint32_t block0;                     /* the launch's first block */
    uint32_t *ctl;                       /* words 0 and 1 cleared by block 0 (k_carry sets word 1 on an error) */
    uint64_t *stamp;                     /* or null: the device clock at the launch's start */
    const uint64_t *res[NTTM_MAX_PRIMES];/* the planes of a k_crt<.., U>: canonical residues, one array per prime */
    CrtConst cc;
};

/* U: the residues are canonical uint64 in a.res[prime] (the primitive's planes) instead of the product's FP64 planes.
 * ST: the product of a descriptor with a step: coefficient kk = i step + pos (pos < step, at least the block's limbs, so that
 * a block meets at most two pieces) is piece i's residue at pos plus, below `over`, piece i - 1's at step + pos. */
template <int NP, int PER, bool U = false, bool ST = false>
__global__ __launch_bounds__(CRT_T) void k_crt(CrtArgs a)
{
    constexpr int CH = CRT_T * PER;                                  /* limbs per block */
    __shared__ uint64_t D[NP][CH + CRT_HALO];
    __shared__ uint32_t s_prod, s_err;
    __shared__ uint32_t s_wave[CRT_T / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t blk = a.block0 + blockIdx.x;
    stamp_clock(a.stamp);
    if (tid == 0 && blk == 0) { a.ctl[0] = 0; a.ctl[1] = 0; }
    if (tid == 0 && !a.desc) { s_prod = 0; s_err = 0; }
    else if (tid == 0) {
        uint64_t lo = 0, hi = a.nprod - 1;                  /* the product whose block range holds blk */
        while (lo < hi) { const uint64_t mid = (lo + hi + 1) >> 1; if (a.desc[mid].first_block <= blk) lo = mid; else hi = mid - 1; }
        s_prod = (uint32_t)lo; s_err = 0;
    }
    __syncthreads();
    CrtDesc dsc = a.one;                             /* (copied as values: see input_limb_raw) */
    if (a.desc) dsc = a.desc[s_prod];
    const uint32_t first = (uint32_t)dsc.first_block, local = blk - first;
    const uint64_t k0 = (uint64_t)local * CH;

    /* digits of coefficients k0 - HALO .. k0 + CH - 1 into LDS (coalesced plane reads, all of a thread's residues
     * requested before the first is used) */
    uint64_t xk[PER];
    {
        const bool halo = tid < CRT_HALO && k0 + tid >= CRT_HALO;   /* coefficient k0 - HALO + tid exists */
        /* the planes as global-space pointers: generic (flat) loads would also count against the LDS counter, whose
         * limit of 15 outstanding operations would serialize the prefetch */
        const __attribute__((address_space(1))) double *pl = (const __attribute__((address_space(1))) double *)dsc.pl;
        const __attribute__((address_space(1))) uint64_t *xg = (const __attribute__((address_space(1))) uint64_t *)dsc.x;
        auto residue = [&](int j, uint64_t kk) -> double {
            if (U) return u64_to_res(((const __attribute__((address_space(1))) uint64_t *)a.res[j])[kk]);
            return pl[j * dsc.plane + kk];
        };
        double rr[PER + 1][NP];
        if (ST) {
            /* the piece of the block's first limb; each coefficient's own by one comparison (the halo's: the piece before) */
            const uint64_t i0 = k0 / dsc.step, s0 = i0 * dsc.step;
            double pv[PER + 1][NP];
#pragma unroll
            for (int i = 0; i <= PER; i++) {
                const uint64_t kk = i < PER ? k0 + i * CRT_T + tid : k0 + tid - CRT_HALO;
                const bool live = (i < PER || halo) && kk < dsc.ncoef;
                uint64_t pc = i0, pos = kk - s0;
                if (i == PER && pos > kk) { pc--; pos += dsc.step; }         /* (kk below s0: the difference wrapped) */
                if (i < PER && pos >= dsc.step) { pc++; pos -= dsc.step; }
                const uint64_t at = pc * dsc.tn + pos;
                const bool own = live && pc * dsc.step < dsc.alen, prev = live && pc && pos < dsc.over;
#pragma unroll
                for (int j = 0; j < NP; j++) {
                    rr[i][j] = own ? residue(j, at) : 0.0;
                    pv[i][j] = prev ? residue(j, at - dsc.tn + dsc.step) : 0.0;
                }
            }
#pragma unroll
            for (int i = 0; i <= PER; i++)
#pragma unroll
                for (int j = 0; j < NP; j++) rr[i][j] = reduce(rr[i][j] + pv[i][j], a.cc.pk[j].p, a.cc.pk[j].pinv);
        } else {
#pragma unroll
            for (int i = 0; i < PER; i++) {
                const uint64_t kk = k0 + i * CRT_T + tid;
#pragma unroll
                for (int j = 0; j < NP; j++) rr[i][j] = kk < dsc.ncoef ? residue(j, kk) : 0.0;
            }
            const uint64_t kk = k0 + tid - CRT_HALO;
#pragma unroll
            for (int j = 0; j < NP; j++) rr[PER][j] = halo && kk < dsc.ncoef ? residue(j, kk) : 0.0;
        }
#pragma unroll
        for (int i = 0; i < PER; i++) {                          /* x at the limbs of the limb phase below */
            const uint64_t k = k0 + wave * 64 * PER + i * 64 + lane;
            xk[i] = k < dsc.nx && k < dsc.nc ? xg[k] : 0;
        }
#pragma unroll
        for (int i = 0; i < PER; i++) {
            uint64_t d[NP];
            crt_digits<NP>(a.cc, rr[i], d);                          /* zero residues give zero digits */
#pragma unroll
            for (int j = 0; j < NP; j++) D[j][CRT_HALO + i * CRT_T + tid] = d[j];
        }
        if (tid < CRT_HALO) {
            uint64_t d[NP];
            crt_digits<NP>(a.cc, rr[PER], d);
#pragma unroll
            for (int j = 0; j < NP; j++) D[j][tid] = d[j];
        }
    }
    __syncthreads();

    /* limb k = k0 + wave 64 PER + i 64 + lane for i < PER: one ballot per i gives 64 consecutive limbs */
    /* v_k = sum_j d_j[k - j] + x_k < NP B + 2^31: its quotient by B is at most NP */
    auto vsum = [&](uint64_t k, int li, uint64_t xv) -> uint64_t {
        uint64_t v = 0;
        if (k < dsc.nc) {
#pragma unroll
            for (int j = 0; j < NP; j++) v += D[j][li - j];
            v += xv;
        }
        return v;
    };
    auto quot = [](uint64_t v) -> uint32_t {
        uint32_t q = 0;
#pragma unroll
        for (int c = 1; c <= NP; c++) q += v >= (uint64_t)c * NTTM_B;
        return q;
    };
    uint64_t wv[PER];
    uint64_t GX[PER], GY[PER];
    uint32_t qlast = 0, qprev = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int off = wave * 64 * PER + i * 64 + lane;          /* offset of limb k inside the block */
        const uint64_t k = k0 + off;
        const int li = CRT_HALO + off;
        const uint64_t v = vsum(k, li, xk[i]);
        const uint32_t q = quot(v);
        /* q_{k-1}: from the lane below; lane 0 from the previous word's lane 63, or (first word) computed */
        uint32_t qp = __shfl_up(q, 1, 64);
        if (i > 0) { if (lane == 0) qp = qprev; }
        else if (lane == 0) qp = k >= 1 ? quot(vsum(k - 1, li - 1, k - 1 < dsc.nx ? dsc.x[k - 1] : 0)) : 0u;
        qprev = __builtin_amdgcn_readlane(q, 63);
        const uint64_t w = v - (uint64_t)q * NTTM_B + qp;            /* <= B + NP */
        wv[i] = w;
        const uint64_t g = __ballot(w >= NTTM_B), pr = __ballot(w == NTTM_B - 1);
        GX[i] = g; GY[i] = g | pr;
        if (k + 1 == dsc.nc) qlast = q;
    }
    /* the wave's map cin -> cout over its PER words */
    uint32_t F = CRT_ID_MAP;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const uint32_t f = add_cout(GX[i], GY[i], 0) | (add_cout(GX[i], GY[i], 1) << 1);
        F = map_compose(f, F);
    }
    if (lane == 0) s_wave[wave] = F;
    __syncthreads();
    uint32_t P = CRT_ID_MAP, A = CRT_ID_MAP;
    for (int w = 0; w < CRT_T / 64; w++) {
        if (w < wave) P = map_compose(s_wave[w], P);
        A = map_compose(s_wave[w], A);
    }

    /* final limbs for a carry of 0 into the block: out_k = w_k + o_{k-1} - B o_k, stored directly (lanes hold
     * consecutive limbs).  c1 follows the carries for a carry of 1 into the block, for the check of the last limb. */
    __attribute__((address_space(1))) uint64_t *cg = (__attribute__((address_space(1))) uint64_t *)dsc.c;
    uint32_t c = map_apply(P, 0), c1 = map_apply(P, 1);              /* the carries into this wave's first word */
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const uint64_t S = GX[i] + GY[i] + c;
        const uint32_t cout = add_cout(GX[i], GY[i], c);
        const uint64_t CI = S ^ GX[i] ^ GY[i];                      /* bit b: the carry into bit b (o_{k-1}) */
        const uint32_t oin = (uint32_t)(CI >> lane) & 1u;
        const uint32_t oout = lane == 63 ? cout : (uint32_t)(CI >> (lane + 1)) & 1u;
        const int off = wave * 64 * PER + i * 64 + lane;
        const uint64_t k = k0 + off;
        if (k < dsc.nc) cg[k] = wv[i] + oin - (oout ? NTTM_B : 0);
        const uint32_t cout1 = add_cout(GX[i], GY[i], c1);
        if (k + 1 == dsc.nc && !dsc.trunc) {                       /* the last limb: nothing may remain beyond it */
            const uint64_t CI1 = (GX[i] + GY[i] + c1) ^ GX[i] ^ GY[i];
            const uint32_t oout1 = lane == 63 ? cout1 : (uint32_t)(CI1 >> (lane + 1)) & 1u;
            uint64_t extra = qlast;
            const int li = CRT_HALO + off;
#pragma unroll
            for (int e = 1; e < NP; e++)
#pragma unroll
                for (int j = e; j < NP; j++) extra += D[j][li + e - j];
            s_err = (extra + oout ? CRT_ST_E0 : 0u) | (extra + oout1 ? CRT_ST_E1 : 0u);
        }
        c = cout; c1 = cout1;
    }
    __syncthreads();
    if (tid == 0) a.status[blk] = A | s_err | (local == 0 ? CRT_ST_FIRST : 0u);
}

/* a block's map as the next block sees it: a product's first block ignores the carry before it.  Monotone: constant 0
 * (0b00), identity (0b10) or constant 1 (0b11) */
__device__ __forceinline__ uint32_t crt_step_map(uint32_t st)
{
    const uint32_t m = st & 3u;
    return (st & CRT_ST_FIRST) ? (m & 1u) * 3u : m;
}
/* The carry into every block, the limbs of the blocks that receive one, and the error flags.  A workgroup takes 64 blocks.
 * The carry into its first is the value of the nearest block before it whose map is not the identity (a map that
 * passes a carry through needs 2048 limbs equal to B - 1, so the block just before almost always decides; otherwise the
 * workgroup goes on looking, 256 words at a time).  Among its own 64 blocks the carries are one addition of the ballot
 * masks of the maps.  The limbs of a block whose carry in is 1 are its stored limbs (for carry 0) plus one, i.e. the
 * leading limbs equal to B - 1 become 0 and the first other one grows by 1: each of the 4 waves takes every 4th such block
 * and rewrites it (CH / 64 limbs per lane, all loads in flight at once).  A product's last block has its error flag taken
 * for its actual carry in; k_crt has cleared ctl.
 * (Two launches before, one workgroup scanning the maps of all blocks and the fix: 57 + 6 us at 131072 blocks, 5 + 4 at
 * few.) */
#define CRT_CARRY_W 64
/* the runs of k_inv_crt: a product of 2^m rows of 2^RUN_LO limbs has RUN_BLOCKS runs per row, RUN_LEN limbs each (the last
 * shorter), and one more for the limbs beyond the transform */
#define RUN_LO 12
#define RUN_LEN 60
#define RUN_GROUPS(m) ((m) == 4 ? 1 : 2)        /* runs per row and wave */
#define RUN_BLOCKS (((1 << RUN_LO) + RUN_LEN - 1) / RUN_LEN)
/* PER = CRT_RUNS, CRT_SEGS: the blocks are k_inv_crt's runs of limbs, or step limbs of each product, instead of PER 256 */
template <int PER>
__global__ __launch_bounds__(256) void k_carry(const CrtDesc *desc, CrtDesc one, uint64_t nprod, const uint32_t *status,
                                               uint64_t n, uint32_t *ctl, uint64_t *stamp)
{
    constexpr bool RUNS = PER == CRT_RUNS, SEGS = PER == CRT_SEGS;
    constexpr int CH = RUNS || SEGS ? 64 : CRT_T * PER;             /* limbs rewritten at a time */
    stamp_clock(stamp);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t b0 = (uint64_t)blockIdx.x * CRT_CARRY_W;
    const bool own = b0 + lane < n;
    const uint32_t st = own ? status[b0 + lane] : 0u;
    uint32_t cin = 0;                                            /* the carry into block b0 */
    for (uint64_t pos = b0; pos; pos -= pos < 256 ? pos : 256) { /* words [pos - 256, pos), nearest first */
        uint32_t w[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint64_t back = (uint64_t)u * 64 + 64 - lane;  /* word pos - back */
            w[u] = back <= pos ? crt_step_map(status[pos - back]) : 0u;   /* nothing before the first block: constant 0 */
        }
        bool found = false;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint64_t dec = __ballot(w[u] != CRT_ID_MAP), val = __ballot((w[u] & 1u) != 0);
            if (!found && dec) { cin = (uint32_t)(val >> (63 - __clzll((long long)dec))) & 1u; found = true; }
        }
        if (found) break;
    }
    const uint32_t m = own ? crt_step_map(st) : 0u;
    const uint64_t X = __ballot(m == 3u), Y = X | __ballot(m == CRT_ID_MAP), CI = (X + Y + cin) ^ X ^ Y;
    const uint32_t ci = (st & CRT_ST_FIRST) ? 0u : (uint32_t)(CI >> lane) & 1u;
    if (__ballot(own && (st & (ci ? CRT_ST_E1 : CRT_ST_E0)) != 0) && threadIdx.x == 0) ctl[1] = 1;
    uint64_t todo = __ballot(own && ci);
    for (int r = 0; todo; r++) {
        const int f = __ffsll((long long)todo) - 1;
        todo &= todo - 1;
        if ((r & 3) != wave) continue;
        const uint64_t blk = b0 + f;
        uint64_t lo = 0, hi = desc ? nprod - 1 : 0;
        while (lo < hi) { const uint64_t mid = (lo + hi + 1) >> 1; if (desc[mid].first_block <= blk) lo = mid; else hi = mid - 1; }
        CrtDesc d = one;
        if (desc) d = desc[lo];
        const uint64_t bl = blk - d.first_block;
        uint64_t k0 = bl * CH, end = k0 + CH;
        if (RUNS) {
            const uint64_t row = bl / RUN_BLOCKS, ch = bl - row * RUN_BLOCKS;
            k0 = (row << RUN_LO) + ch * RUN_LEN; end = ch + 1 < RUN_BLOCKS ? k0 + RUN_LEN : (row + 1) << RUN_LO;
        }
        if (SEGS) { k0 = bl * d.step; end = k0 + d.step; }
        end = end < d.nc ? end : d.nc;
        if (SEGS) {                                             /* word by word: nearly always the first is the last */
            for (; k0 < end; k0 += 64) {
                const uint64_t k = k0 + lane, x = k < end ? d.c[k] : 0;
                const uint64_t ne = __ballot(k < end && x != NTTM_B - 1);
                const int at = ne ? __ffsll((long long)ne) - 1 : 64;
                if (k < end && lane <= at) d.c[k] = lane < at ? 0 : x + 1;
                if (ne) break;
            }
            continue;
        }
        uint64_t v[CH / 64];
#pragma unroll
        for (int j = 0; j < CH / 64; j++) { const uint64_t k = k0 + j * 64 + lane; v[j] = k < end ? d.c[k] : 0; }
        int first_ne = CH;                                      /* offset of the first limb below B - 1 */
#pragma unroll
        for (int j = CH / 64 - 1; j >= 0; j--) {
            const uint64_t ne = __ballot(k0 + j * 64 + lane < end && v[j] != NTTM_B - 1);
            if (ne) first_ne = j * 64 + __ffsll((long long)ne) - 1;
        }
#pragma unroll
        for (int j = 0; j < CH / 64; j++) {
            const int o = j * 64 + lane;
            const uint64_t k = k0 + o;
            if (k < end && o <= first_ne) d.c[k] = o < first_ne ? 0 : v[j] + 1;
        }
    }
}

/* ---- the last inverse pass and the CRT in one kernel ------------------------------------------------------------------
 * For transforms of 2^m rows of 2^12 points, m = 1 .. 4 (one strided pass): a lane takes one column of the plane of each
 * prime, all 2^m rows of it in registers, multiplies in the boundary twiddles w^-(c brev(j)) (powers of the column's table entry),
 * runs the 2^m-point DIT and has the residues of 2^m coefficients of every prime, which it turns into digits and
 * limbs as k_crt does.  Nothing is exchanged but between neighbouring lanes: a wave covers 60 columns and, in its first
 * four lanes, the four before them (a row's first run takes the last four columns and their previous row), so
 * every limb's lower digits and the quotient before the first limb come by shuffles.  A wave's run of 60 limbs is
 * one ballot word and one block of the carry launch.  For m < 4 a wave takes two runs, every load requested at once.
 * It replaces a pass over the planes (16 B read and written per point and prime) and the CRT's reads (8 B): bound by
 * vector issue, 269 instructions per coefficient at m = 1, 283, 323 and 368 at m = 4, of which 1 in 16 is spent on the four
 * repeated columns, at 86, 86, 62 and 68% of the issue rate (2 to 5 waves per SIMD).  4096 products of 64 to 65536 limbs: 1.15 ms against 0.64 (inverse pass) + 0.65 (k_crt). */
struct InvCrtArgs {
    const CrtDesc *desc; uint64_t nprod;        /* null: the one product `one` */
    CrtDesc one;
    uint32_t *status, *ctl;
    int first;                                  /* the launch that clears ctl */
    uint64_t *stamp;
    const double2 *stage[NTTM_MAX_PRIMES];      /* inverse stage tables */
    const double2 *step[NTTM_MAX_PRIMES];       /* (w, wq) of w_(2^(12 + m))^-c, c < 2^12 */
    CrtConst cc;
};
__device__ __forceinline__ uint64_t shfl_up64(uint64_t v, int d) { return (uint64_t)__shfl_up((unsigned long long)v, d, 64); }

template <int M, int NP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_inv_crt(InvCrtArgs a)
{
    constexpr int R = 1 << M, G = RUN_GROUPS(M), COLS = 1 << RUN_LO, WPP = (RUN_BLOCKS + G - 1) / G;
    typedef const __attribute__((address_space(1))) double *GRes;
    typedef const __attribute__((address_space(1))) uint64_t *GIn;
    typedef __attribute__((address_space(1))) uint64_t *GOut;
    typedef const __attribute__((address_space(1))) char *GByte;
    typedef __attribute__((address_space(1))) char *GByteW;
    stamp_clock(a.stamp);
    if (a.first && blockIdx.x == 0 && threadIdx.x == 0) { a.ctl[0] = 0; a.ctl[1] = 0; }
    const int lane = threadIdx.x & 63;
    const uint32_t wid = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    const uint32_t prod = wid / WPP, ch0 = (wid - prod * WPP) * G;
    if (prod >= a.nprod) return;
    CrtDesc d = a.one;
    if (a.desc) d = a.desc[prod];
    /* (products of at most 2^16 + 2 limbs) */
    const int ncoef = (int)d.ncoef, nc = (int)d.nc, nx = (int)(d.nx < d.nc ? d.nx : d.nc);

    /* uniform bases and 32-bit lane offsets: a load's address costs no vector registers of its own */
    double r[NP][G][R];
    int col[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        col[g] = (int)(ch0 + g) * RUN_LEN + lane - 4;            /* a row's first run: -4 .. -1 are the previous row's end */
        const uint32_t off = 8u * (uint32_t)(col[g] < 0 ? col[g] + COLS : col[g] < COLS ? col[g] : COLS - 1);
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int j = 0; j < R; j++)
                r[p][g][j] = *(GRes)((GByte)(d.pl + p * d.plane + ((uint32_t)j << RUN_LO)) + off);
    }
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const double P = a.cc.pk[p].p, PI = a.cc.pk[p].pinv;
#pragma unroll
        for (int g = 0; g < G; g++) {
            const uint32_t c = (uint32_t)(col[g] < 0 ? col[g] + COLS : col[g] < COLS ? col[g] : COLS - 1);
            typedef double v2d __attribute__((ext_vector_type(2)));
            const v2d step = *(const __attribute__((address_space(1))) v2d *)((GByte)a.step[p] + 16u * c);
            double w = step[0];
            r[p][g][R / 2] = mul_shoup(r[p][g][R / 2], step[0], step[1], P);     /* brev(R / 2) = 1 */
#pragma unroll
            for (int i = 2; i < R; i++) {
                w = mul_shoup(w, step[0], step[1], P);
                r[p][g][brev_c<M>(i)] = mul_barrett(r[p][g][brev_c<M>(i)], w, P, PI);
            }
            dit_group<M, CTab>(r[p][g], 0, 0u, CTab(a.stage[p]), P, PI);
            __builtin_amdgcn_sched_barrier(0);                   /* one column at a time: the registers hold the residues */
        }
    }
    auto quot = [](uint64_t v) -> uint32_t {
        uint32_t q = 0;
#pragma unroll
        for (int c = 1; c <= NP; c++) q += v >= (uint64_t)c * NTTM_B;
        return q;
    };
    /* the limbs and the carry map of the run of row `row` from the lane's digits and x limb */
    auto finish = [&](int g, int row, const uint64_t *dg, uint64_t x) {
        const bool in = col[g] < COLS;
        const int k = (row << RUN_LO) + col[g];
        const bool limb = in && k >= 0 && k < nc, act = lane >= 4 && in;
        uint64_t v = dg[0] + x;
#pragma unroll
        for (int j = 1; j < NP; j++) v += shfl_up64(dg[j], j);       /* (lanes below 3: unused) */
        v = limb ? v : 0;
        const uint32_t q = quot(v), qp = __shfl_up(q, 1, 64);
        const uint64_t w = v - (uint64_t)q * NTTM_B + qp;
        const uint64_t live = __ballot(act) >> 4;
        const uint64_t X = __ballot(act && limb && w >= NTTM_B) >> 4;
        const uint64_t Y = X | (__ballot(act && limb && w == NTTM_B - 1) >> 4) | ~live;   /* past the run: passed on */
        const uint64_t CI = (X + Y) ^ X ^ Y;
        const uint32_t oin = (uint32_t)(CI >> (lane - 4)) & 1u, oout = (uint32_t)(CI >> (lane - 3)) & 1u;
        if (act && k < nc) *(GOut)((GByteW)d.c + 8u * (uint32_t)k) = w + oin - (oout ? NTTM_B : 0);
        uint32_t st = add_cout(X, Y, 0) | (add_cout(X, Y, 1) << 1);
        const uint64_t top = __ballot(act && k + 1 == nc);
        if (top && !d.trunc) {                                   /* the last limb: nothing may remain beyond it */
            uint64_t extra = q;
#pragma unroll
            for (int e = 1; e < NP; e++)
#pragma unroll
                for (int j = e; j < NP; j++) extra += j == e ? dg[j] : shfl_up64(dg[j], j - e);
            const uint64_t C1 = (X + Y + 1) ^ X ^ Y;
            const uint32_t o1 = (uint32_t)(C1 >> (lane - 3)) & 1u;
            const int l = __ffsll((long long)top) - 1;
            if ((__ballot(extra + oout != 0) >> l) & 1) st |= CRT_ST_E0;
            if ((__ballot(extra + o1 != 0) >> l) & 1) st |= CRT_ST_E1;
        }
        const uint32_t b = (uint32_t)row * RUN_BLOCKS + ch0 + g;
        if (lane == 0) a.status[d.first_block + b] = st | (b == 0 ? CRT_ST_FIRST : 0u);
    };
    /* the run's limbs in one row: the x limb requested, the residues (the previous row's in a row's first four lanes) to digits */
#define RUN_ROW(ROW) { \
        const int rw = (ROW), k = (rw << RUN_LO) + col[g]; \
        uint64_t xv = 0, dg[NP]; \
        if (nx && col[g] < COLS && k >= 0 && k < nx) xv = *(GIn)((GByte)d.x + 8u * (uint32_t)k); \
        const bool coef = col[g] < COLS && k >= 0 && k < ncoef; \
        double rz[NP]; \
        _Pragma("unroll") \
        for (int p = 0; p < NP; p++) { \
            const double here = rw < R ? r[p][g][rw < R ? rw : 0] : 0.0, prev = rw ? r[p][g][rw ? rw - 1 : 0] : 0.0; \
            rz[p] = coef ? (wrap ? prev : here) : 0.0; \
        } \
        crt_digits<NP>(a.cc, rz, dg); \
        finish(g, rw, dg, xv); \
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
        if (ch0 + g >= RUN_BLOCKS) break;
        const bool wrap = col[g] < 0;
#pragma unroll
        for (int row = 0; row < R; row++) RUN_ROW(row)
        if (ch0 + g == 0) RUN_ROW(R)                             /* the limbs from 2^logn on: the last coefficients' upper digits */
    }
#undef RUN_ROW
}

/* c[0 .. n) += *carry (0 or 1), the carry rippling through the leading limbs equal to B - 1 (one workgroup, 2048
 * limbs per step; a carry beyond limb n - 1 is dropped: the caller's bound makes it zero) */
__global__ __launch_bounds__(256) void k_add_carry(uint64_t *c, uint64_t n, const uint64_t *carry)
{
    __shared__ uint32_t s_first;
    const int tid = threadIdx.x;
    const uint64_t cin = *carry;
    if (!cin) return;
    for (uint64_t base = 0; base < n; base += 256 * 8) {
        if (tid == 0) s_first = 0xffffffffu;
        __syncthreads();
        uint64_t v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t off = (uint32_t)(i * 256 + tid);
            const uint64_t k = base + off;
            v[i] = k < n ? c[k] : 0;
            if (k < n && v[i] != NTTM_B - 1) atomicMin(&s_first, off);
        }
        __syncthreads();
        const uint32_t f = s_first;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const uint32_t off = (uint32_t)(i * 256 + tid);
            const uint64_t k = base + off;
            if (k < n && off <= f) c[k] = off < f ? 0 : v[i] + cin;
        }
        if (f != 0xffffffffu) return;
        __syncthreads();
    }
}
int nttm_run_add_carry(uint64_t *c, uint64_t n, const uint64_t *carry, hipStream_t s)
{
    if (!n) return 0;
    hipLaunchKernelGGL(k_add_carry, dim3(1), dim3(256), 0, s, c, n, carry);
    return nttm_hip_check(hipGetLastError(), "k_add_carry launch");
}

__global__ void k_norm(const CrtDesc *d, uint64_t nprod, uint64_t *ncn)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nprod) return;
    uint64_t n = d[i].nc;
    while (n && d[i].c[n - 1] == 0) n--;
    ncn[i] = n;
}

/* blocks of a product of nc limbs at per limbs per thread (CRT_WIDE, or 1) */
uint64_t nttm_crt_blocks(uint64_t nc, int per) { const uint64_t ch = (uint64_t)CRT_T * (per == 1 ? 1 : CRT_WIDE); return (nc + ch - 1) / ch; }

uint64_t nttm_crt_scratch_words(uint64_t nblocks) { return nblocks + CRT_CTL_WORDS; }

/* desc_dev: nprod descriptors in device memory whose block ranges tile [blk0, blk0 + nblk) of scratch's status words
 * (null: the one product `one`): their limbs for a carry into every block of 0, and the blocks' carry maps */
int nttm_crt_launch_limbs(const CrtDesc *desc_dev, const CrtDesc *one, uint64_t nprod, uint64_t blk0, uint64_t nblk, int np,
                          const CrtConst &cc, uint32_t *scratch, uint32_t *ctl, hipStream_t s, double alg_bytes, int per,
                          uint64_t *stamp, const uint64_t *const *res)
{
    if (per != 1 && per != CRT_WIDE) return nttm_fail(NTTM_EINVAL, "crt: %d limbs per thread", per);
    if (np < 3 || np > NTTM_MAX_PRIMES) return nttm_fail(NTTM_EINVAL, "crt: np = %d", np);
    if (!nprod || !nblk) return 0;
    if (!desc_dev && (!one || nprod != 1)) return nttm_fail(NTTM_EINVAL, "crt: no descriptors");
    if (blk0 + nblk > 0x7fffffffULL) return nttm_fail(NTTM_EINVAL, "crt: too many blocks");
    if ((uintptr_t)scratch & 15) return nttm_fail(NTTM_EINVAL, "crt: scratch not 16-byte aligned");
    CrtArgs a;
    memset(&a.one, 0, sizeof a.one);
    if (one) a.one = *one;
    a.desc = desc_dev; a.nprod = nprod; a.block0 = (uint32_t)blk0; a.stamp = stamp; a.ctl = ctl;
    a.status = scratch + CRT_CTL_WORDS; a.cc = cc;
    for (int j = 0; j < NTTM_MAX_PRIMES; j++) a.res[j] = res && j < np ? res[j] : nullptr;
    if (one && one->step && (per == 1 || res || one->step < CRT_T * CRT_WIDE || one->over > one->step || !one->tn))
        return nttm_fail(NTTM_EINVAL, "crt: pieces of %llu limbs", (unsigned long long)one->step);
    if (res && per == 1) return nttm_fail(NTTM_EINVAL, "crt: residue planes take the wide blocks");
    prof_begin("k_crt", alg_bytes, s);
    if (res) {
        if (np == 3) hipLaunchKernelGGL((k_crt<3, CRT_WIDE, true>), dim3((unsigned)nblk), dim3(CRT_T), 0, s, a);
        else hipLaunchKernelGGL((k_crt<4, CRT_WIDE, true>), dim3((unsigned)nblk), dim3(CRT_T), 0, s, a);
    } else if (one && one->step) {
        if (np == 3) hipLaunchKernelGGL((k_crt<3, CRT_WIDE, false, true>), dim3((unsigned)nblk), dim3(CRT_T), 0, s, a);
        else hipLaunchKernelGGL((k_crt<4, CRT_WIDE, false, true>), dim3((unsigned)nblk), dim3(CRT_T), 0, s, a);
    } else if (per == 1) {
        if (np == 3) hipLaunchKernelGGL((k_crt<3, 1>), dim3((unsigned)nblk), dim3(CRT_T), 0, s, a);
        else hipLaunchKernelGGL((k_crt<4, 1>), dim3((unsigned)nblk), dim3(CRT_T), 0, s, a);
    } else {
        if (np == 3) hipLaunchKernelGGL((k_crt<3, CRT_WIDE>), dim3((unsigned)nblk), dim3(CRT_T), 0, s, a);
        else hipLaunchKernelGGL((k_crt<4, CRT_WIDE>), dim3((unsigned)nblk), dim3(CRT_T), 0, s, a);
    }
    prof_end(s);
    return nttm_hip_check(hipGetLastError(), "k_crt launch");
}
/* every block's carry in, and the limbs of the blocks that receive one; word 1 of ctl (scratch, or pinned host memory)
 * receives the error flag */
int nttm_crt_launch_carry(const CrtDesc *desc_dev, const CrtDesc *one, uint64_t nprod, uint64_t nblocks, uint32_t *scratch,
                          uint32_t *ctl, hipStream_t s, int per, uint64_t *stamp)
{
    if (!nprod || !nblocks) return 0;
    const uint32_t *status = scratch + CRT_CTL_WORDS;
    CrtDesc d1; memset(&d1, 0, sizeof d1);
    if (one) d1 = *one;
    prof_begin("k_carry", 4.0 * (double)nblocks, s);
    const dim3 grid((unsigned)((nblocks + CRT_CARRY_W - 1) / CRT_CARRY_W));
    if (per == CRT_RUNS) hipLaunchKernelGGL((k_carry<CRT_RUNS>), grid, dim3(256), 0, s, desc_dev, d1, nprod, status, nblocks, ctl, stamp);
    else if (per == CRT_SEGS) hipLaunchKernelGGL((k_carry<CRT_SEGS>), grid, dim3(256), 0, s, desc_dev, d1, nprod, status, nblocks, ctl, stamp);
    else if (per == 1) hipLaunchKernelGGL((k_carry<1>), grid, dim3(256), 0, s, desc_dev, d1, nprod, status, nblocks, ctl, stamp);
    else hipLaunchKernelGGL((k_carry<CRT_WIDE>), grid, dim3(256), 0, s, desc_dev, d1, nprod, status, nblocks, ctl, stamp);
    prof_end(s);
    return nttm_hip_check(hipGetLastError(), "k_carry launch");
}
/* whether the last inverse pass of a 2^logn-point transform (bits [lo, lo + m) of the index) runs fused with the CRT */
int nttm_inv_crt_ok(int logn, int lo, int m) { return lo == RUN_LO && m >= 1 && m <= 4 && lo + m == logn; }
/* a product's blocks there (runs) */
uint64_t nttm_inv_crt_blocks(int m) { return ((uint64_t)RUN_BLOCKS << m) + 1; }
/* the last inverse pass and the CRT of nprod products of 2^(12 + m) points, from device descriptors (null: `one`), with
 * nttm_inv_crt_blocks(m) blocks each from its descriptor's first_block on; first: the launch that clears ctl */
int nttm_run_inv_crt(int np, int m, const CrtDesc *desc_dev, const CrtDesc *one, uint64_t nprod, const TwTables *inv,
                     const CrtConst &cc, uint32_t *scratch, uint32_t *ctl, int first, hipStream_t s, double alg_bytes,
                     uint64_t *stamp)
{
    if (np < 3 || np > NTTM_MAX_PRIMES || m < 1 || m > 4 || !nprod || (!desc_dev && (!one || nprod != 1)))
        return nttm_fail(NTTM_EINVAL, "internal: inverse pass with the CRT");
    InvCrtArgs a; memset(&a, 0, sizeof a);
    a.desc = desc_dev; a.nprod = nprod; a.status = scratch + CRT_CTL_WORDS; a.ctl = ctl; a.first = first; a.stamp = stamp; a.cc = cc;
    if (one) a.one = *one;
    for (int i = 0; i < np; i++) { a.stage[i] = inv[i].stage; a.step[i] = m <= 2 ? inv[i].stage + ((size_t)1 << (RUN_LO - 1 + m)) : inv[i].col + ((size_t)(m - 3) << RUN_LO); }
    const uint64_t g = RUN_GROUPS(m), waves = nprod * ((RUN_BLOCKS + g - 1) / g), blocks = (waves + 3) / 4;
    if (blocks > 0x3fffffffULL || nprod * nttm_inv_crt_blocks(m) > 0x7fffffffULL) return nttm_fail(NTTM_EINVAL, "internal: too many products");
    const dim3 grid((unsigned)blocks);
    prof_begin("k_inv_crt", alg_bytes, s);
#define INV_CRT_LAUNCH(L) \
    if (np == 3) hipLaunchKernelGGL((k_inv_crt<L, 3>), grid, dim3(256), 0, s, a); \
    else hipLaunchKernelGGL((k_inv_crt<L, 4>), grid, dim3(256), 0, s, a);
    switch (m) {
    case 1: INV_CRT_LAUNCH(1) break;
    case 2: INV_CRT_LAUNCH(2) break;
    case 3: INV_CRT_LAUNCH(3) break;
    default: INV_CRT_LAUNCH(4) break;
    }
#undef INV_CRT_LAUNCH
    prof_end(s);
    return nttm_hip_check(hipGetLastError(), "k_inv_crt launch");
}
/* one product, its descriptor passed with the launches: scratch 16-byte aligned, nttm_crt_scratch_words(nblocks) words.
 * stamps (or null): the device clock at the start of both launches.  res (or null): the np planes as
 * arrays of canonical residues, in place of d's */
int nttm_crt_launch_one(const CrtDesc &d, uint64_t nblocks, int np, const CrtConst &cc, uint32_t *scratch, uint32_t *ctl,
                        hipStream_t s, double alg_bytes, uint64_t *stamps, const uint64_t *const *res)
{
    RCK(nttm_crt_launch_limbs(nullptr, &d, 1, 0, nblocks, np, cc, scratch, ctl, s, alg_bytes, CRT_WIDE, stamps, res));
    return nttm_crt_launch_carry(nullptr, &d, 1, nblocks, scratch, ctl, s, CRT_WIDE, stamps ? stamps + 1 : nullptr);
}

/* ---- addition and subtraction of limb arrays, with the carry resolved like the CRT's -------------------------------
 * r[0 .. nout) = a B^sa + b B^sb, or a B^sa - b B^sb computed as a B^sa + (B^nout - 1 - b B^sb) + 1 (b's limbs
 * complemented, 1 added at limb 0): its carry out of limb nout - 1 is 1 exactly when the difference is >= 0.
 * b may instead be B^bpow (bpow >= 0).  Each 2048-limb block writes its limbs for a carry in of 0 and its one-bit
 * carry map, with the same status words as k_crt; k_carry then adds every block's carry (and, from the last block's error
 * bits, gives the final carry out).  Limbs past nout count as B - 1 so that
 * the last block's map is the carry out of limb nout - 1. */
struct AddArgs {
    const uint64_t *a; uint64_t na, sa;
    const uint64_t *b; uint64_t nb, sb;
    int64_t apow, bpow;
    uint64_t *r; uint64_t nout, nblocks;
    int sub;
    uint32_t *status, *ctl;
};
__device__ __forceinline__ uint64_t add_limb(const uint64_t *p, uint64_t n, uint64_t s, uint64_t k)
{
    return (k >= s && k - s < n) ? p[k - s] : 0;
}
__global__ __launch_bounds__(CRT_T) void k_addsub(AddArgs a)
{
    constexpr int PER = CRT_WIDE, CH = CRT_T * PER;
    __shared__ uint32_t s_wave[CRT_T / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t blk = blockIdx.x, k0 = blk * CH;
    if (tid == 0 && blk == 0) { a.ctl[0] = 0; a.ctl[1] = 0; }
    uint64_t wv[PER], GX[PER], GY[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const uint64_t k = k0 + wave * 64 * PER + i * 64 + lane;
        uint64_t w = NTTM_B - 1;
        if (k < a.nout) {
            const uint64_t x = a.apow >= 0 ? (k == (uint64_t)a.apow ? 1u : 0u) : add_limb(a.a, a.na, a.sa, k);
            const uint64_t y = a.bpow >= 0 ? (k == (uint64_t)a.bpow ? 1u : 0u) : add_limb(a.b, a.nb, a.sb, k);
            w = x + (a.sub ? NTTM_B - 1 - y : y) + (a.sub && k == 0 ? 1u : 0u);          /* <= 2B - 1 */
        }
        wv[i] = w;
        const uint64_t g = __ballot(w >= NTTM_B), pr = __ballot(w == NTTM_B - 1);
        GX[i] = g; GY[i] = g | pr;
    }
    uint32_t F = CRT_ID_MAP;
#pragma unroll
    for (int i = 0; i < PER; i++) F = map_compose(add_cout(GX[i], GY[i], 0) | (add_cout(GX[i], GY[i], 1) << 1), F);
    if (lane == 0) s_wave[wave] = F;
    __syncthreads();
    uint32_t P = CRT_ID_MAP, A = CRT_ID_MAP;
    for (int w = 0; w < CRT_T / 64; w++) {
        if (w < wave) P = map_compose(s_wave[w], P);
        A = map_compose(s_wave[w], A);
    }
    uint32_t c = map_apply(P, 0);
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const uint64_t S = GX[i] + GY[i] + c;
        const uint32_t cout = add_cout(GX[i], GY[i], c);
        const uint64_t CI = S ^ GX[i] ^ GY[i];
        const uint32_t oin = (uint32_t)(CI >> lane) & 1u;
        const uint32_t oout = lane == 63 ? cout : (uint32_t)(CI >> (lane + 1)) & 1u;
        const uint64_t k = k0 + wave * 64 * PER + i * 64 + lane;
        if (k < a.nout) a.r[k] = wv[i] + oin - (oout ? NTTM_B : 0);
        c = cout;
    }
    if (tid == 0) {
        uint32_t st = A | (blk == 0 ? CRT_ST_FIRST : 0u);
        if (blk + 1 == a.nblocks) st |= ((A & 1u) ? CRT_ST_E0 : 0u) | ((A & 2u) ? CRT_ST_E1 : 0u);
        a.status[blk] = st;
    }
}
int nttm_run_addsub(uint64_t *r, uint64_t nout, const uint64_t *a, uint64_t na, uint64_t sa, int64_t apow, const uint64_t *b,
                    uint64_t nb, uint64_t sb, int64_t bpow, int sub, uint32_t *scratch, hipStream_t s)
{
    if (!nout) return 0;
    const uint64_t nblocks = nttm_crt_blocks(nout, CRT_WIDE);
    if (nblocks > 0x7fffffffULL) return nttm_fail(NTTM_EINVAL, "addsub: too many blocks");
    if ((uintptr_t)scratch & 15) return nttm_fail(NTTM_EINVAL, "addsub: scratch not 16-byte aligned");
    AddArgs A;
    A.a = a; A.na = a ? na : 0; A.sa = sa; A.apow = apow; A.b = b; A.nb = b ? nb : 0; A.sb = sb; A.bpow = bpow;
    A.r = r; A.nout = nout; A.nblocks = nblocks; A.sub = sub; A.status = scratch + CRT_CTL_WORDS;
    A.ctl = scratch;
    hipLaunchKernelGGL(k_addsub, dim3((unsigned)nblocks), dim3(CRT_T), 0, s, A);
    int rc = nttm_hip_check(hipGetLastError(), "k_addsub launch");
    if (rc) return rc;
    CrtDesc d; memset(&d, 0, sizeof d);
    d.c = r; d.nc = nout;
    return nttm_crt_launch_carry(nullptr, &d, 1, nblocks, scratch, scratch, s, CRT_WIDE, nullptr);
}

/* the normalized length of x[0 .. n): one more than the index of the highest nonzero limb */
/* one more than the index of the top non-zero limb of x[0 .. n) (0 if none), by atomicMax into *out (cleared first).
 * Chunk c covers [n - (c + 1) C, n - c C): the chunks are taken from the top down, block b taking b, b + G, b + 2G, ...
 * (G blocks, at most one per CU), and a block stops as soon as *out reaches the top of its next chunk (nothing below
 * can raise the maximum).  A number with a few leading zero limbs costs one chunk per block; one with many streams
 * its zero top at full bandwidth until the first non-zero chunk. */
#define TOPNZ_PER 16
#define TOPNZ_CHUNK (256 * TOPNZ_PER)
#define TOPNZ_GRID 256
__global__ __launch_bounds__(256) void k_top_nonzero(const uint64_t *x, uint64_t n, unsigned long long *out)
{
    const uint64_t nchunk = (n + TOPNZ_CHUNK - 1) / TOPNZ_CHUNK;
    for (uint64_t c = blockIdx.x; c < nchunk; c += gridDim.x) {
        const uint64_t hi = n - c * TOPNZ_CHUNK, lo = hi > TOPNZ_CHUNK ? hi - TOPNZ_CHUNK : 0;
        if (__hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= hi) return;
        unsigned long long best = 0;
#pragma unroll
        for (int j = 0; j < TOPNZ_PER; j++) {
            const uint64_t k = lo + (uint64_t)j * 256 + threadIdx.x;
            if (k < hi && x[k]) best = k + 1;
        }
        for (int d = 32; d; d >>= 1) {
            const unsigned long long o = __shfl_down(best, d, 64);
            best = o > best ? o : best;
        }
        if ((threadIdx.x & 63) == 0 && best) atomicMax(out, best);
    }
}
int nttm_run_top_nonzero(const uint64_t *x, uint64_t n, uint64_t *out_dev, hipStream_t s)
{
    int rc = nttm_hip_check(hipMemsetAsync(out_dev, 0, 8, s), "clear length");
    if (rc || !n) return rc;
    const uint64_t chunks = (n + TOPNZ_CHUNK - 1) / TOPNZ_CHUNK;
    const unsigned blocks = (unsigned)(chunks < TOPNZ_GRID ? chunks : TOPNZ_GRID);
    hipLaunchKernelGGL(k_top_nonzero, dim3(blocks), dim3(256), 0, s, x, n, (unsigned long long *)out_dev);
    return nttm_hip_check(hipGetLastError(), "k_top_nonzero launch");
}
/* the normalized length of x[0 .. n) into *len_dev (device pointers), for tests */
extern "C" int nttm_debug_top_nonzero(const uint64_t *x, size_t n, uint64_t *len_dev, void *stream)
{
    if (!len_dev || (n && !x)) return nttm_fail(NTTM_EINVAL, "nttm_debug_top_nonzero arguments");
    return nttm_run_top_nonzero(x, n, len_dev, (hipStream_t)stream);
}

/* products with an empty operand: c[0 .. nc) = x zero-extended (a kernel, not a memset, so a captured graph holds it) */
__global__ __launch_bounds__(256) void k_fill_x(const CrtDesc *d, uint64_t nprod)
{
    const CrtDesc q = d[blockIdx.x];
    for (uint64_t k = threadIdx.x; k < q.nc; k += 256) q.c[k] = k < q.nx ? q.x[k] : 0;
}
int nttm_run_fill_x(const void *desc_dev, uint64_t nprod, hipStream_t s)
{
    if (!nprod) return 0;
    if (nprod > 0x7fffffffULL) return nttm_fail(NTTM_EINVAL, "fill: too many products");
    hipLaunchKernelGGL(k_fill_x, dim3((unsigned)nprod), dim3(256), 0, s, (const CrtDesc *)desc_dev, nprod);
    return nttm_hip_check(hipGetLastError(), "k_fill_x launch");
}

int nttm_run_norm(const void *desc_dev, uint64_t nprod, uint64_t *ncn_dev, hipStream_t s)
{
    if (!nprod) return 0;
    hipLaunchKernelGGL(k_norm, dim3((unsigned)((nprod + 255) / 256)), dim3(256), 0, s, (const CrtDesc *)desc_dev, nprod, ncn_dev);
    return nttm_hip_check(hipGetLastError(), "k_norm launch");
}
