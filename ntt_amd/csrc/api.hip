/* api.hip - the C ABI of libnttm.so: context and tables, the product schedule (one large product, batches of leaf
 * products) and the transform primitives.  See include/nttm.h for the contract and the reference entry points each
 * function replaces. */
#include <stdarg.h>
#include <stdio.h>
#include <string.h>
#include <stdlib.h>
#include <vector>
#include <map>
#include <array>
#include <algorithm>
#include <chrono>
#include <thread>
#include <atomic>
#include "internal.h"
#include "plan.h"
#include "segrule.h"

int nttm_run_pass(bool inv, const PassArgs &a, const PassGeom &g, hipStream_t s, const JobSet *jobs = nullptr);
int nttm_run_fused2(const PassArgs &a, const FusedB &fb, const PassGeom &g, hipStream_t s, const FusedSet &js);
bool nttm_fwd_pass_streams(const PassArgs &a, const PassGeom &g);
void nttm_set_pts(int pts);
int nttm_get_pts(void);
void nttm_set_fixed_shapes(int on);
void nttm_set_stream(int on, int ncu);
int nttm_ncu(void);
#define NTTM_CRT_RUNS 0            /* the carry launch's blocks are k_inv_crt's runs, */
#define NTTM_CRT_SEGS (-1)         /* or k_segments' segments */
#define NTTM_FUSED_LOG 12          /* tile of the fused forward + pointwise + inverse pass (k_fused2) */
#define NTTM_TILE_LOG_DEFAULT 13   /* tile of the strided passes: 2^13 points (64 KiB of LDS), runs of 32 columns */
#define NTTM_PRODUCT_LOGN_MIN 4    /* products use at least 2^4 points, so every fused tile has >= 16 */
#define NTTM_STAGE_CHUNK ((size_t)1 << 30)   /* staged bytes per sub-batch of a batch with host operands (default) */
struct LoadArgs;
int nttm_run_cvt_u64_f64(double *dst, const uint64_t *src, uint64_t count, hipStream_t s);
int nttm_run_f64_to_canon(double *x, uint64_t count, const PrimeK &pk, hipStream_t s);
int nttm_run_pw_u64(uint64_t *x, const uint64_t *y, uint64_t count, const PrimeK &pk, hipStream_t s);
int nttm_run_load_planes(double *dst, uint64_t plane, const uint64_t *src, uint64_t nlimbs, uint64_t npoints, int np,
                         const PrimeK *pk, const double2 *scale, int out_u64, hipStream_t s);
/* the CRT of products whose blocks are [blk0, blk0 + nblk) of the launch's block numbering (limbs for a carry in of 0),
 * then every block's carry; nttm_crt_launch_one: both for one product */
int nttm_crt_launch_limbs(const CrtDesc *desc_dev, const CrtDesc *one, uint64_t nprod, uint64_t blk0, uint64_t nblk, int np,
                          const CrtConst &cc, uint32_t *scratch, uint32_t *ctl, hipStream_t s, double alg_bytes, int per,
                          uint64_t *stamp = nullptr, const uint64_t *const *res = nullptr);
int nttm_crt_launch_carry(const CrtDesc *desc_dev, const CrtDesc *one, uint64_t nprod, uint64_t nblocks, uint32_t *scratch,
                          uint32_t *ctl, hipStream_t s, int per, uint64_t *stamp = nullptr);
int nttm_crt_launch_one(const CrtDesc &d, uint64_t nblocks, int np, const CrtConst &cc, uint32_t *scratch, uint32_t *ctl,
                        hipStream_t s, double alg_bytes, uint64_t *stamps = nullptr, const uint64_t *const *res = nullptr);
uint64_t nttm_crt_blocks(uint64_t nc, int per = 8);      /* per: CRT limbs per thread, 8 (2048-limb blocks) or 1 (256) */
uint64_t nttm_crt_scratch_words(uint64_t nblocks);
int nttm_inv_crt_ok(int logn, int lo, int m);
uint64_t nttm_inv_crt_blocks(int m);
int nttm_run_inv_crt(int np, int m, const CrtDesc *desc_dev, const CrtDesc *one, uint64_t nprod, const TwTables *inv,
                     const CrtConst &cc, uint32_t *scratch, uint32_t *ctl, int first, hipStream_t s, double alg_bytes,
                     uint64_t *stamp);
int nttm_small_log(int logn);
int nttm_run_small(int np, int logn, const LoadDesc *ld, const CrtDesc *cd, const LoadDesc *ld1, const CrtDesc *cd1,
                   uint64_t cnt, uint64_t *ncn, uint32_t *ctl, const TwTables *fwd, const TwTables *inv, const double2 *ninv,
                   const CrtConst &cc, hipStream_t s, double alg_bytes, uint64_t *stamps);
uint64_t nttm_seg_len(uint64_t nb);
int nttm_run_segments(int np, const LoadDesc *ld, const CrtDesc *cd, const LoadDesc *ld1, const CrtDesc *cd1, uint64_t nprod,
                      uint64_t groups, const TwTables *fwd, const TwTables *inv, const double2 *ninv,
                      const CrtConst &cc, uint32_t *scratch, uint32_t *ctl, hipStream_t s, double alg_bytes, uint64_t *stamps);
int nttm_run_norm(const void *desc_dev, uint64_t nprod, uint64_t *ncn_dev, hipStream_t s);
int nttm_run_fill_x(const void *desc_dev, uint64_t nprod, hipStream_t s);
int nttm_run_dft16_mfma(const uint64_t *x, double *y, int logn, uint64_t batch, const void *etab, const double *tlo,
                        const double *thi, const double *consts, double p, hipStream_t s);
int nttm_run_add_carry(uint64_t *c, uint64_t n, const uint64_t *carry, hipStream_t s);
int nttm_run_r3(bool inv, int logk, const JobSet &js, hipStream_t s, uint64_t *stamp = nullptr, bool u64 = false);

/* ---- errors ----------------------------------------------------------------------------------------------------- */
/* per host thread: the library's own helper threads (the e pipeline's download preparation) may fail too */
static thread_local char g_err[512] = "";
int nttm_fail(int code, const char *fmt, ...)
{
    va_list ap; va_start(ap, fmt); vsnprintf(g_err, sizeof g_err, fmt, ap); va_end(ap);
    return code;
}
int nttm_hip_check(hipError_t e, const char *what)
{
    if (e == hipSuccess) return 0;
    return nttm_fail(NTTM_EHIP, "%s: %s", what, hipGetErrorString(e));
}
extern "C" const char *nttm_last_error(void) { return g_err; }

/* ---- host modular arithmetic (exact, __int128) -------------------------------------------------------------------- */
typedef unsigned __int128 u128;
static uint64_t h_mulmod(uint64_t a, uint64_t b, uint64_t p) { return (uint64_t)((u128)a * b % p); }
static uint64_t h_powmod(uint64_t a, uint64_t e, uint64_t p)
{
    uint64_t r = 1 % p; a %= p;
    while (e) { if (e & 1) r = h_mulmod(r, a, p); a = h_mulmod(a, a, p); e >>= 1; }
    return r;
}
static uint64_t h_inv(uint64_t a, uint64_t p) { return h_powmod(a, p - 2, p); }
static uint64_t h_generator(uint64_t p)
{
    uint64_t f[64]; int nf = 0, t2 = 0; uint64_t t = p - 1;
    while (!(t & 1)) { t >>= 1; t2 = 1; }
    if (t2) f[nf++] = 2;
    for (uint64_t q = 3; q * q <= t; q += 2) if (t % q == 0) { f[nf++] = q; while (t % q == 0) t /= q; }
    if (t > 1) f[nf++] = t;
    for (uint64_t g = 2; g < p; g++) {
        int ok = 1;
        for (int i = 0; i < nf && ok; i++) if (h_powmod(g, (p - 1) / f[i], p) == 1) ok = 0;
        if (ok) return g;
    }
    return 0;
}
static double h_bal(uint64_t v, uint64_t p) { return v > p / 2 ? -(double)(p - v) : (double)v; }
static double2 h_shoup(uint64_t v, uint64_t p) { double w = h_bal(v, p); return make_double2(w, w / (double)p); }

/* ---- the context ------------------------------------------------------------------------------------------------------ */
struct Ctx {
    int init, dev;
    nttm_config cfg;
    PrimeK pk[NTTM_MAX_PRIMES];
    uint64_t root32[NTTM_MAX_PRIMES];        /* root of order 2^32 */
    uint64_t root3x32[NTTM_MAX_PRIMES];      /* root of order 3 2^32 */
    TwTables twf[NTTM_MAX_PRIMES], twi[NTTM_MAX_PRIMES];
    double2 *tables;
    CrtConst cc;
    char *ws; size_t ws_bytes;               /* device workspace */
    uint64_t *tmp; size_t tmp_limbs;         /* a piece product of a grid (above one transform) */
    uint64_t *bsp[2]; size_t bsp_limbs[2];   /* the inner levels of a binary-splitting tree (even / odd levels) */
    char *tdesc; size_t tdesc_bytes;         /* the descriptors of a batch's groups, or of every group of a planned tree */
    char *tpin; size_t tpin_bytes;           /* their pinned host image, and the groups' flags */
    hipStream_t tcs;                         /* descriptor copies (ahead of the launches on the caller's stream) */
    void *dfree[8]; int ndfree;              /* buffers the planned tree outgrew, freed after its final synchronization */
    void *hfree[4]; int nhfree;
    hipEvent_t tev[8];                       /* the last copies on tcs, in turn */
    uint64_t *hpin; size_t hpin_bytes;       /* pinned host staging (descriptors, flags) */
    char *stage; size_t stage_bytes;         /* device copies of host-resident operands and results */
    size_t stage_chunk;                      /* staged bytes per sub-batch of a batch */
    char *chk; size_t chk_bytes;             /* device scratch of the residue post-condition */
    uint64_t *xc; size_t xc_limbs;           /* copies of the x operands that lie under their results */
    char *bounce; size_t bounce_half;        /* pinned bounce buffer of the host copies: two halves */
    char *dl; size_t dl_half; hipEvent_t dlev[2];   /* pinned halves of the large downloads (nttm_copy_to_host) */
    hipEvent_t bev[2]; int bev_live[2];      /* the last copy through each half */
    uint64_t gen;                            /* which nttm_init this context is (plans record it) */
    hipEvent_t ev[4];
    hipEvent_t pev[2 * NTTM_MAX_PRIMES];      /* around B's transform of each prime (phase times of nttm_mul) */
    double last_ms[3];
    uint64_t *stamps; int last_stamped;      /* pinned: the device clock at the last short product's phase boundaries */
    double last_b;                           /* B's share of its joint forward launches (0: a product in segments) */
};
static Ctx g;
static uint64_t g_init_count;
static int g_prof_on;                        /* live kernel timing on (nttm_profile) */
static int g_no_defer;                       /* NTTM_NO_DEFER=1: every pass applies its own boundary twiddles */
static int g_no_small;                       /* NTTM_GENERIC_PASSES=1: no whole product in one kernel either */
static int g_tree_levelwise;                 /* NTTM_TREE_LEVELWISE=1: the tree level by level (for comparison) */
static int g_fused_bits_env;                 /* NTTM_FUSED_BITS=10|11|12: that last-pass width for every product
                                              * transform above it (for comparison measurements) */

/* Products of at most g_par_points points per prime run each pass as ONE launch for all primes and both operands, each
 * prime with a B plane of its own (2 np planes); longer ones run prime after prime through np + 1 planes.  A launch
 * costs about 6 us beside its work (the gap, the blocks' tables, the last tiles), and one prime's pass of 2^21 points has one
 * tile per CU: nothing to fetch ahead.  Measured per call, prime after prime against one launch for all: 32 K-limb
 * operands 163 -> 86 us, 2^20 276 -> 202, 2^22 840 -> 724, 2^23 (2^24 points) 1529 -> 1405; at 2^25 points the two are
 * equal (2.77 and 2.75 ms) and the planes twice as large.  NTTM_PAR_POINTS overrides it, 0 turns it off. */
static uint64_t g_par_points = (uint64_t)1 << 24;
/* points of one prime per chunk of a batch group: a group's products run chunk after chunk through the same planes, so
 * that the planes stay below 2 np 128 MiB.  Smaller chunks, whose planes would fit the last-level cache, are slower:
 * the 4096 leaves' replay takes 5.83 ms at 2^24 points, 5.91 at 2^22, 6.71 at 2^21, 8.41 at 2^20 (four more launches
 * per chunk).  NTTM_CHUNK_POINTS overrides it. */
static uint64_t g_chunk_points = (uint64_t)1 << 24;
static int64_t g_pieces_points = -1;         /* NTTM_PIECES: 0 never in pieces, else pieces of that many points */
static uint64_t g_inv_crt_points = (uint64_t)1 << 22;   /* the last inverse pass with the CRT (inv_crt_bits): 2^14 points a CU */

/* the workspace of nttm_mul_noalloc: a file-scope device array, one copy per GPU, held until the process ends.  Host
 * code never uses its name as an address (on the host it is a stand-in, not the device address): nttm_init looks up
 * the address on its device with hipGetSymbolAddress and keeps it in g_scratch_dev[device]. */
#define NTTM_NOALLOC_BYTES ((size_t)40 << 20)
#define NTTM_NOALLOC_MAX_DEV 64
static __device__ __align__(256) char scratch[NTTM_NOALLOC_BYTES];
static char *g_scratch_dev[NTTM_NOALLOC_MAX_DEV];                /* nttm_init calls so far: a plan made under an earlier one is stale */

static uint64_t max_terms_np(int np)
{
    /* floor((prod p - 1) / (B - 1)^2) by long division of the product (< 2^200) */
    uint64_t M[4] = {1, 0, 0, 0};
    for (int i = 0; i < np; i++) {
        uint64_t carry = 0;
        for (int w = 0; w < 4; w++) { u128 s = (u128)M[w] * NTTM_PRIMES[i] + carry; M[w] = (uint64_t)s; carry = (uint64_t)(s >> 64); }
    }
    for (int w = 0; w < 4; w++) { if (M[w]--) break; }
    const u128 D = (u128)(NTTM_B - 1) * (NTTM_B - 1);
    u128 rem = 0; uint64_t q[4] = {0, 0, 0, 0};
    for (int bit = 255; bit >= 0; bit--) {
        int top = (int)(rem >> 127);
        rem = (rem << 1) | ((M[bit / 64] >> (bit % 64)) & 1);
        if (top || rem >= D) { rem -= D; q[bit / 64] |= 1ULL << (bit % 64); }
    }
    if (q[1] || q[2] || q[3]) return UINT64_MAX;
    return q[0];
}

extern "C" uint64_t nttm_prime(int i) { return (i >= 0 && i < NTTM_MAX_PRIMES) ? NTTM_PRIMES[i] : 0; }
extern "C" uint64_t nttm_max_terms(int np) { return (np >= 1 && np <= NTTM_MAX_PRIMES) ? max_terms_np(np) : 0; }
extern "C" uint64_t nttm_root(int i, int logn)
{
    if (i < 0 || i >= NTTM_MAX_PRIMES || logn < 0 || logn > NTTM_LOGN_MAX) return 0;
    const uint64_t p = NTTM_PRIMES[i];
    return h_powmod(h_generator(p), (p - 1) >> logn, p);
}
extern "C" uint64_t nttm_root3(int i, int logk)
{
    if (i < 0 || i >= NTTM_MAX_PRIMES || logk < 0 || logk > NTTM_LOGN_MAX) return 0;
    const uint64_t p = NTTM_PRIMES[i];
    return h_powmod(h_generator(p), ((p - 1) >> logk) / 3, p);
}

static void build_crt_const(CrtConst &cc)
{
    memset(&cc, 0, sizeof cc);
    for (int i = 0; i < NTTM_MAX_PRIMES; i++) {
        const uint64_t p = NTTM_PRIMES[i];
        cc.pk[i].p = (double)p; cc.pk[i].pinv = 1.0 / (double)p; cc.pk[i].pu = p;
        /* prefix product p_0 ... p_{i-1} in words, and its residue mod p_i */
        uint64_t M[NTTM_MAX_PRIMES] = {1, 0, 0, 0};
        for (int j = 0; j < i; j++) {
            uint64_t carry = 0;
            for (int w = 0; w < NTTM_MAX_PRIMES; w++) { u128 s = (u128)M[w] * NTTM_PRIMES[j] + carry; M[w] = (uint64_t)s; carry = (uint64_t)(s >> 64); }
        }
        for (int w = 0; w < NTTM_MAX_PRIMES; w++) cc.mprod[i][w] = M[w];
        {   /* the same in base 10^18 (digits j < i; the product is below 2^(50 i) < 10^(18 i)) */
            uint64_t W[NTTM_MAX_PRIMES];
            for (int w = 0; w < NTTM_MAX_PRIMES; w++) W[w] = M[w];
            for (int j = 0; j < NTTM_MAX_PRIMES; j++) {
                u128 rem = 0;
                for (int w = NTTM_MAX_PRIMES - 1; w >= 0; w--) {
                    const u128 cur = (rem << 64) | W[w];
                    W[w] = (uint64_t)(cur / NTTM_B); rem = cur % NTTM_B;
                }
                cc.mb[i][j] = (uint64_t)rem;
                cc.mbp[i][j] = (uint64_t)(((u128)rem << 64) / NTTM_B);
            }
        }
        for (int j = 1; j <= i; j++) {
            uint64_t m = 1;
            for (int k = 0; k < j; k++) m = h_mulmod(m, NTTM_PRIMES[k] % p, p);
            if (j < i) cc.mmod[i][j] = h_bal(m, p);
            if (j == i) cc.cinv[i] = h_bal(h_inv(m, p), p);
        }
    }
}

static int build_tables(void)
{
    const size_t nst = (size_t)1 << NTTM_STAGE_LOG;
    const size_t nbq = (size_t)4 << NTTM_BQ_LOG, nb3 = nbq + 1, ncol = (size_t)2 << 12;
    const size_t per_dir = nst + nbq + nb3, per_prime = 2 * per_dir + ncol, total = (size_t)NTTM_MAX_PRIMES * per_prime;
    std::vector<double2> h(total);
    for (int i = 0; i < NTTM_MAX_PRIMES; i++) {
        const uint64_t p = NTTM_PRIMES[i];
        const uint64_t gen = h_generator(p);
        g.root32[i] = h_powmod(gen, (p - 1) >> 32, p);
        g.root3x32[i] = h_powmod(gen, ((p - 1) >> 32) / 3, p);
        for (int dir = 0; dir < 2; dir++) {
            const uint64_t w32 = dir ? h_inv(g.root32[i], p) : g.root32[i];
            double2 *st = &h[i * per_prime + dir * per_dir], *bq = st + nst;
            double2 *b3 = bq + nbq;
            const uint64_t W3 = dir ? h_inv(g.root3x32[i], p) : g.root3x32[i];
            for (int k = 0; k < 4; k++) {                                /* b3[k 2^8 + x] = W3^(x 2^(8k)) */
                const uint64_t wk = h_powmod(W3, (uint64_t)1 << (NTTM_BQ_LOG * k), p);
                uint64_t v = 1;
                for (size_t x = 0; x < ((size_t)1 << NTTM_BQ_LOG); x++) {
                    b3[((size_t)k << NTTM_BQ_LOG) + x] = h_shoup(v, p); v = h_mulmod(v, wk, p);
                }
            }
            b3[nbq] = h_shoup(h_powmod(g.root3x32[i], (uint64_t)1 << 32, p), p);   /* the forward cube root */
            double2 *co = b3 + nb3;
            for (int m = 3; dir && m <= 4; m++) {                        /* (the inverse direction's only) */
                const uint64_t wm = h_powmod(w32, (uint64_t)1 << (32 - 12 - m), p);
                uint64_t v = 1;
                for (size_t c = 0; c < ((size_t)1 << 12); c++) { co[((size_t)(m - 3) << 12) + c] = h_shoup(v, p); v = h_mulmod(v, wm, p); }
            }
            st[0] = h_shoup(1, p);
            for (int s = 0; s + 1 < NTTM_STAGE_LOG + 1 && ((size_t)1 << s) < nst; s++) {
                const uint64_t ws = h_powmod(w32, (uint64_t)1 << (32 - (s + 1)), p);   /* order 2^(s+1) */
                uint64_t v = 1;
                for (size_t j = 0; j < ((size_t)1 << s); j++) { st[((size_t)1 << s) + j] = h_shoup(v, p); v = h_mulmod(v, ws, p); }
            }
            for (int k = 0; k < 4; k++) {                                /* bq[k 2^8 + x] = w32^(x 2^(8k)) */
                const uint64_t wk = h_powmod(w32, (uint64_t)1 << (NTTM_BQ_LOG * k), p);
                uint64_t v = 1;
                for (size_t x = 0; x < ((size_t)1 << NTTM_BQ_LOG); x++) {
                    bq[((size_t)k << NTTM_BQ_LOG) + x] = h_shoup(v, p); v = h_mulmod(v, wk, p);
                }
            }
        }
    }
    HIPCK(hipMalloc(&g.tables, total * sizeof(double2)));
    HIPCK(hipMemcpy(g.tables, h.data(), total * sizeof(double2), hipMemcpyHostToDevice));
    for (int i = 0; i < NTTM_MAX_PRIMES; i++)
        for (int dir = 0; dir < 2; dir++) {
            const double2 *st = g.tables + i * per_prime + dir * per_dir;
            TwTables t; t.stage = st; t.bq = st + nst;
            t.b3 = t.bq + nbq; t.col = dir ? t.b3 + nb3 : nullptr;
            if (dir) g.twi[i] = t; else g.twf[i] = t;
        }
    return 0;
}

/* an outgrown buffer: freed at once after a device synchronization, or (defer: work queued before it may still read
 * it, the caller synchronizes later) listed for free_deferred, so that growing it does not wait for that work */
static int drop_dev(void *p, bool defer)
{
    if (!p) return 0;
    if (defer && g.ndfree < 8) { g.dfree[g.ndfree++] = p; return 0; }
    HIPCK(hipDeviceSynchronize());
    HIPCK(hipFree(p));
    return 0;
}
static int drop_host(void *p, bool defer)
{
    if (!p) return 0;
    if (defer && g.nhfree < 4) { g.hfree[g.nhfree++] = p; return 0; }
    HIPCK(hipDeviceSynchronize());
    HIPCK(hipHostFree(p));
    return 0;
}
/* after the synchronization that ends every use of the listed buffers */
static void free_deferred(void)
{
    for (int i = 0; i < g.ndfree; i++) (void)hipFree(g.dfree[i]);
    for (int i = 0; i < g.nhfree; i++) (void)hipHostFree(g.hfree[i]);
    g.ndfree = g.nhfree = 0;
}
static int ws_need(size_t bytes, bool defer = false)
{
    if (g.cfg.workspace_bytes && bytes > g.cfg.workspace_bytes)
        return nttm_fail(NTTM_ENOMEM, "workspace of %zu bytes exceeds the configured cap %zu", bytes, g.cfg.workspace_bytes);
    if (bytes <= g.ws_bytes) return 0;
    if (g.ws) { RCK(drop_dev(g.ws, defer)); g.ws = nullptr; g.ws_bytes = 0; }
    if (hipMalloc(&g.ws, bytes) != hipSuccess) { (void)hipGetLastError(); return nttm_fail(NTTM_ENOMEM, "hipMalloc of %zu bytes failed", bytes); }
    g.ws_bytes = bytes;
    return 0;
}
static int hpin_need(size_t bytes)
{
    if (bytes <= g.hpin_bytes) return 0;
    if (g.hpin) { HIPCK(hipDeviceSynchronize()); HIPCK(hipHostFree(g.hpin)); g.hpin = nullptr; g.hpin_bytes = 0; }
    HIPCK(hipHostMalloc((void **)&g.hpin, bytes, hipHostMallocDefault));
    g.hpin_bytes = bytes;
    return 0;
}

/* ---- where an operand lives -------------------------------------------------------------------------------------------
 * Kernels read and write HBM only (XNACK is off: a kernel touching host memory faults the GPU).  Every pointer an entry
 * point takes is classed before any launch: device memory of this device is used in place; host memory -- pageable,
 * pinned (hipHostMalloc) or managed -- is copied through library-owned HBM by the entry points that stage (the
 * products, as the reference's batch stages products outside registered memory, E/rns_mul.h:42-47,
 * E/rns_mul.c:807-817) and refused with NTTM_EINVAL by the others.  One MemMap lives for one call: it remembers the
 * device allocations it has seen, so the operands of a large batch carved from a few allocations cost one runtime
 * query per allocation. */
enum { MEM_DEV = 0, MEM_HOST = 1, MEM_PINNED = 2, MEM_BAD = 3 };
struct MemMap {
    std::map<uintptr_t, uintptr_t> dev;                          /* base -> end of the device allocations seen */
    uintptr_t last_b = 0, last_e = 0;                            /* the last one hit */
    const char *why = "";
    int kind(const void *p, size_t bytes)
    {
        if (!p || !bytes) return MEM_DEV;                        /* nothing is read or written */
        const uintptr_t a = (uintptr_t)p, e = a + bytes;
        if (e < a) { why = "wraps the address space"; return MEM_BAD; }
        if (a >= last_b && a < last_e) return e <= last_e ? MEM_DEV : (why = "runs past the end of its device allocation", MEM_BAD);
        auto it = dev.upper_bound(a);
        if (it != dev.begin()) {
            --it;
            if (a < it->second) {
                last_b = it->first; last_e = it->second;
                return e <= it->second ? MEM_DEV : (why = "runs past the end of its device allocation", MEM_BAD);
            }
        }
        hipPointerAttribute_t at;
        memset(&at, 0, sizeof at);
        if (hipPointerGetAttributes(&at, p) != hipSuccess) { (void)hipGetLastError(); return MEM_HOST; }   /* pageable */
        if (at.type == hipMemoryTypeDevice) {
            if (at.device != g.dev) { why = "is device memory of another device"; return MEM_BAD; }
            hipDeviceptr_t base = nullptr; size_t sz = 0;
            if (hipMemGetAddressRange(&base, &sz, (hipDeviceptr_t)p) == hipSuccess && base && sz) {
                const uintptr_t b = (uintptr_t)base;
                dev[b] = b + sz; last_b = b; last_e = b + sz;
                if (e > b + sz) { why = "runs past the end of its device allocation"; return MEM_BAD; }
            } else (void)hipGetLastError();
            return MEM_DEV;
        }
        if (at.type == hipMemoryTypeHost) return MEM_PINNED;
        return MEM_HOST;                                         /* managed, unified or unregistered */
    }
};
/* NTTM_EINVAL unless [p, p + bytes) is device memory of the library's device (entry points that do not stage) */
int nttm_require_device(const void *p, size_t bytes, const char *what)
{
    MemMap mm;
    const int k = mm.kind(p, bytes);
    if (k == MEM_DEV) return 0;
    return nttm_fail(NTTM_EINVAL, "%s %s", what, k == MEM_BAD ? mm.why : "is host memory (this entry point takes device memory)");
}
#define DEVCK(p, bytes, what) RCK(nttm_require_device((p), (bytes), (what)))
/* NTTM_EINVAL unless [p, p + bytes) is host memory (pageable, pinned or managed): entry points whose output the host
 * writes or first-touches */
int nttm_require_host(const void *p, size_t bytes, const char *what)
{
    MemMap mm;
    const int k = mm.kind(p, bytes);
    if (k == MEM_HOST || k == MEM_PINNED) return 0;
    return nttm_fail(NTTM_EINVAL, "%s %s", what, k == MEM_BAD ? mm.why : "is device memory (this entry point takes host memory)");
}

extern "C" int nttm_init(int device, const nttm_config *cfg)
{
    if (g.init) return nttm_fail(NTTM_ESTATE, "nttm_init: already initialised");
    memset(&g, 0, sizeof g);
    if (cfg) g.cfg = *cfg;
    if (g.cfg.nprimes && g.cfg.nprimes != 3 && g.cfg.nprimes != 4)
        return nttm_fail(NTTM_EINVAL, "nttm_init: nprimes must be 0, 3 or 4");
    if (!g.cfg.tile_log) g.cfg.tile_log = NTTM_TILE_LOG_DEFAULT;
    if (g.cfg.tile_log != 12 && g.cfg.tile_log != 13) return nttm_fail(NTTM_EINVAL, "nttm_init: tile_log must be 12 or 13");
    if (g.cfg.pts && g.cfg.pts != 8 && g.cfg.pts != 16) return nttm_fail(NTTM_EINVAL, "nttm_init: pts must be 0, 8 or 16");
    if (g.cfg.radix3 < NTTM_R3_AUTO || g.cfg.radix3 > NTTM_R3_FIT)
        return nttm_fail(NTTM_EINVAL, "nttm_init: radix3 must be 0, 1 or 2");
    if (g.cfg.check != 0 && g.cfg.check != 1) return nttm_fail(NTTM_EINVAL, "nttm_init: check must be 0 or 1");
    nttm_set_pts(g.cfg.pts ? g.cfg.pts : 16);
    {   /* NTTM_GENERIC_PASSES=1: runtime-geometry pass kernels only (for comparison) */
        const char *e = getenv("NTTM_GENERIC_PASSES");
        nttm_set_fixed_shapes(!(e && e[0] == '1'));
        g_no_small = e && e[0] == '1';
    }
    int nd = 0;
    HIPCK(hipGetDeviceCount(&nd));
    if (device < 0 || device >= nd) return nttm_fail(NTTM_EINVAL, "nttm_init: device %d of %d", device, nd);
    HIPCK(hipSetDevice(device));
    g.dev = device;
    if (device < NTTM_NOALLOC_MAX_DEV && !g_scratch_dev[device]) {   /* once per device, with it current */
        void *ptr = nullptr;
        HIPCK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (!ptr) return nttm_fail(NTTM_EHIP, "nttm_init: no device address for the no-allocation workspace");
        g_scratch_dev[device] = (char *)ptr;
    }
    {   /* NTTM_STREAM=0: strided passes without the LDS-streaming kernel (for comparison); one streaming block per CU */
        const char *st = getenv("NTTM_STREAM");
        int ncu = 0;
        HIPCK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device));
        nttm_set_stream(!(st && st[0] == '0'), ncu);
    }
    for (int i = 0; i < NTTM_MAX_PRIMES; i++) { g.pk[i].p = (double)NTTM_PRIMES[i]; g.pk[i].pinv = 1.0 / (double)NTTM_PRIMES[i]; g.pk[i].pu = NTTM_PRIMES[i]; }
    build_crt_const(g.cc);
    RCK(build_tables());
    for (int i = 0; i < 4; i++) HIPCK(hipEventCreate(&g.ev[i]));
    for (int i = 0; i < 2 * NTTM_MAX_PRIMES; i++) HIPCK(hipEventCreate(&g.pev[i]));
    RCK(hpin_need(1 << 16));
    HIPCK(hipHostMalloc((void **)&g.stamps, 64, hipHostMallocDefault));
    {
        const char *e = getenv("NTTM_NO_DEFER");
        g_no_defer = e && e[0] == '1';
    }
    {
        const char *e = getenv("NTTM_PAR_POINTS"), *c = getenv("NTTM_CHUNK_POINTS"), *v = getenv("NTTM_INV_CRT_POINTS");
        g_par_points = e ? strtoull(e, nullptr, 0) : (uint64_t)1 << 24;
        g_chunk_points = c && strtoull(c, nullptr, 0) ? strtoull(c, nullptr, 0) : (uint64_t)1 << 24;
        const char *pp = getenv("NTTM_PIECES");
        g_pieces_points = pp ? (int64_t)strtoull(pp, nullptr, 0) : -1;
        g_inv_crt_points = v && strtoull(v, nullptr, 0) ? strtoull(v, nullptr, 0) : (uint64_t)nttm_ncu() << 14;
    }
    {
        const char *e = getenv("NTTM_TREE_LEVELWISE");
        g_tree_levelwise = e && e[0] == '1';
    }
    {
        const char *e = getenv("NTTM_FUSED_BITS");
        g_fused_bits_env = e ? atoi(e) : 0;
    }
    {   /* NTTM_STAGE_CHUNK=<bytes>: staged bytes per sub-batch (default 1 GiB; smaller values exercise the split) */
        const char *e = getenv("NTTM_STAGE_CHUNK");
        g.stage_chunk = e && atoll(e) > 0 ? (size_t)atoll(e) : NTTM_STAGE_CHUNK;
    }
    g.gen = ++g_init_count;
    g.init = 1;
    return 0;
}

static void prof_release(void);
extern "C" void nttm_shutdown(void)
{
    if (!g.init) return;
    (void)hipDeviceSynchronize();
    prof_release();
    if (g.ws) (void)hipFree(g.ws);
    if (g.tmp) (void)hipFree(g.tmp);
    for (int k = 0; k < 2; k++) if (g.bsp[k]) (void)hipFree(g.bsp[k]);
    if (g.tdesc) (void)hipFree(g.tdesc);
    if (g.tpin) (void)hipHostFree(g.tpin);
    if (g.tables) (void)hipFree(g.tables);
    if (g.hpin) (void)hipHostFree(g.hpin);
    if (g.stamps) (void)hipHostFree(g.stamps);
    if (g.stage) (void)hipFree(g.stage);
    if (g.chk) (void)hipFree(g.chk);
    if (g.xc) (void)hipFree(g.xc);
    if (g.bounce) (void)hipHostFree(g.bounce);
    if (g.dl) (void)hipHostFree(g.dl);
    for (int k = 0; k < 2; k++) if (g.dlev[k]) (void)hipEventDestroy(g.dlev[k]);
    for (int k = 0; k < 2; k++) if (g.bev[k]) (void)hipEventDestroy(g.bev[k]);
    for (int k = 0; k < 8; k++) if (g.tev[k]) (void)hipEventDestroy(g.tev[k]);
    if (g.tcs) (void)hipStreamDestroy(g.tcs);
    free_deferred();
    for (int i = 0; i < 4; i++) (void)hipEventDestroy(g.ev[i]);
    for (int i = 0; i < 2 * NTTM_MAX_PRIMES; i++) if (g.pev[i]) (void)hipEventDestroy(g.pev[i]);
    memset(&g, 0, sizeof g);
}

/* ---- transforms on FP64 planes ------------------------------------------------------------------------------------------ */
static int ceil_log2(uint64_t n) { int l = 0; while (((uint64_t)1 << l) < n) l++; return l; }

static PassArgs base_args(int prime, double *x, int logn, uint64_t batch, bool inv)
{
    PassArgs a; memset(&a, 0, sizeof a);
    a.x = x; a.y = nullptr; a.logn = logn; a.batch = batch; a.ymode = NTTM_Y_FULL;
    a.pk = g.pk[prime]; a.tw = inv ? g.twi[prime] : g.twf[prime]; a.twi = g.twi[prime];
    return a;
}
/* in_u64 / out_u64: the plane holds canonical uint64 residues before / after the transform (converted in its first and
 * last pass) */
static int fwd_planes(int prime, double *x, int logn, uint64_t batch, hipStream_t s, int in_u64 = 0, int out_u64 = 0)
{
    Plan pl; plan_make(&pl, logn, batch, g.cfg.tile_log);
    for (int i = 0; i < pl.npass; i++) {
        PassArgs a = base_args(prime, x, logn, batch, false);
        a.in_u64 = in_u64 && i == 0; a.out_u64 = out_u64 && i == pl.npass - 1;
        RCK(nttm_run_pass(false, a, pl.p[i], s));
    }
    return 0;
}
/* inverse with the pointwise product by y (ymode layout) fused into the first pass; scale by n^-1 in the last pass.
 * r3y: the batch is the thirds of transforms of 3 2^logn points, y holds whole such transforms */
static int inv_planes(int prime, double *x, const double *y, int ymode, int logn, uint64_t batch, int scale, hipStream_t s,
                      int r3y = 0, int in_u64 = 0, int y_u64 = 0, int out_u64 = 0)
{
    Plan pl; plan_make(&pl, logn, batch, g.cfg.tile_log);
    PassArgs a = base_args(prime, x, logn, batch, true);
    for (int i = pl.npass - 1; i >= 0; i--) {
        PassArgs b = a;
        if (i == pl.npass - 1) { b.y = y; b.ymode = ymode; b.r3y = r3y; b.in_u64 = in_u64; b.y_u64 = y && y_u64; }
        if (i == 0) b.out_u64 = out_u64;
        if (i == 0 && scale) {
            const uint64_t p = NTTM_PRIMES[prime];
            b.scale = h_shoup(h_inv(((uint64_t)1 << logn) % p, p), p); b.do_scale = 1;
        }
        RCK(nttm_run_pass(true, b, pl.p[i], s));
    }
    return 0;
}

/* ---- the product ------------------------------------------------------------------------------------------------------- */
static int choose_np(size_t mn, int *np)
{
    int want = g.cfg.nprimes;
    if (!want) want = (uint64_t)mn <= max_terms_np(3) ? 3 : 4;
    if ((uint64_t)mn > max_terms_np(want))
        return nttm_fail(NTTM_EBOUND, "a product of %zu terms exceeds the %d-prime bound of %llu terms", mn, want,
                         (unsigned long long)max_terms_np(want));
    *np = want;
    return 0;
}

static size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

/* the transforms of one length group of products (cnt transforms of 2^logn points per prime):
 *   B: forward, the first pass reading b's limbs (times n^-1, folded here once);
 *   A: forward up to its last pass, the first pass reading a's limbs;
 *   A: the fused last forward pass + pointwise product with B + first inverse pass (k_fused2);
 *   A: the remaining inverse passes.
 * Operand limbs come from (a, na, b, nb) when cnt == 1 and ldesc is null, else from the device descriptors ldesc.
 * Result: plane i of A holds the cyclic convolution mod p_i. */
/* the strided-pass tile for a 2^logn product transform: the configured one, or 2^13 where that saves a pass */
static int product_tile_log(int logn, int tl = 0)
{
    if (!tl) tl = g.cfg.tile_log;
    const int R = logn > NTTM_FUSED_LOG ? logn - NTTM_FUSED_LOG : 0;
    const int k_cfg = (R + tl - 5) / (tl - 4), k_13 = (R + 8) / 9;
    return k_13 < k_cfg ? 13 : tl;
}

/* bits of the double-fused last pass of a 2^logn product transform (its tiles stay 2^12 points): 12, or 10 and 11 for
 * 2^26 and 2^27 points, so that their two strided passes take 8 bits each (8+8+10, 8+8+11, 8+8+12 up to 2^28) and run
 * as the 8 x 32 streamed shape -- a level moved out of the fused pass (instruction-bound: both forward transforms and
 * the inverse run there) costs less in an HBM-bound strided pass.  Measured per pass at 2^28 points on one MI355X:
 * 8-bit streamed passes 0.78-0.85 ms, 9-bit (16-column rows) 0.96-1.14 ms, the fused pass 2.08 ms at 12 bits and 1.68
 * at 10, so 9+9+10 loses to 8+8+12 there, and 2^29 / 2^30 points keep 9+8+12 / 9+9+12. */
static int fused_bits(int logn, int tile_log)
{
    if (tile_log == 13 && g_fused_bits_env >= 10 && g_fused_bits_env <= 12 && logn > g_fused_bits_env &&
        logn - g_fused_bits_env <= 18)
        return g_fused_bits_env;
    if (tile_log != 13 || logn < 26 || logn > 30) return NTTM_FUSED_LOG;
    return logn <= 28 ? logn - 16 : NTTM_FUSED_LOG;
}
static void product_plan(Plan *pl, int logn, uint64_t batch, int tile_log)
{
    plan_make3(pl, logn, batch, tile_log, fused_bits(logn, tile_log), NTTM_FUSED_LOG);
}
/* the bits of a product transform's last inverse pass where it runs fused with the CRT (k_inv_crt: transforms of 2^13 to
 * 2^16 points, whose one strided pass has at most 16 rows), else 0.  With 2 and 4 rows always: a batch of equal products
 * against the two kernels, us, 2^13: 1 of them 53 / 59, 16 55 / 62, 256 138 / 162; 2^14: 52 / 55, 63 / 68, 215 / 250.
 * With 8 and 16 a wave is long (120 to 250 registers) and few of them are slower than the two kernels that spread the same
 * work wider: from 2^22 points.  2^15: 1 60 / 55, 64 152 / 153, 128 237 / 243, 256 441 / 464; 2^16: 1 63 / 57, 32 154 / 151,
 * 64 242 / 244, 128 445 / 461, 256 839 / 894.  NTTM_INV_CRT_POINTS overrides that line. */
static int inv_crt_bits(int logn, int r3, uint64_t cnt)
{
    if (r3 || g_no_small || g_fused_bits_env || logn <= NTTM_FUSED_LOG || logn > NTTM_FUSED_LOG + 4) return 0;
    return logn <= NTTM_FUSED_LOG + 2 || (cnt << logn) >= g_inv_crt_points ? logn - NTTM_FUSED_LOG : 0;
}
/* the most blocks of the CRT of a product of nc limbs from a 2^logn (3 2^logn) point transform of n points */
static uint64_t prod_crt_blocks(int logn, int r3, uint64_t n, uint64_t nc)
{
    const int m = inv_crt_bits(logn, r3, (uint64_t)1 << 32);
    return std::max(m ? nttm_inv_crt_blocks(m) : 0, nttm_crt_blocks(nc, n <= 1024 ? 1 : 8));
}

/* the transforms of cnt products of one length: 2^logn points (r3 = 0), or 3 2^logn points (r3 = 1: a radix-3 layer,
 * reading the limbs, and the 2^logn engine on the 3 cnt thirds).  Plane i of A holds the cnt transforms of prime i back
 * to back.  After it, A holds the cyclic convolutions mod each prime, natural order.
 * Shared B operands (bmap non-null): B's plane holds the cnt_b distinct operands of ldesc_b; A's engine transform t
 * pairs with B's engine transform bmap[t] in the double-fused pass.
 * pev (or null): 2 np events recorded around B's transform of each prime.  stamps (or null): the device clock at the
 * start of the first forward launch and of the double-fused pass.  inv_crt: A's last inverse pass is left to k_inv_crt. */
/* the first forward pass (from limbs) leaves its boundary twiddles to the second when both are streamed strided
 * passes (a transform of three or more passes): the limb pass has no VALU to spare, the second pass, bound by HBM, has.
 * q: the first pass's arguments (limbs set, in_scale as the caller wants it applied) */
static bool defer_ok(const PassArgs &q, const Plan &pl, int last)
{
    if (last < 2 || g_no_defer || !(q.limbs || q.ldesc)) return false;
    PassArgs nx = q; nx.limbs = nullptr; nx.ldesc = nullptr; nx.do_in_scale = 0;
    return nttm_fwd_pass_streams(q, pl.p[0]) && nttm_fwd_pass_streams(nx, pl.p[1]) && pl.p[1].m >= 4;
}
/* the deferral's flags for pass j of the plan (a job's dfr_scale goes with the pass that has dfr_in) */
static void defer_set(PassArgs &q, const Plan &pl, int j, bool on)
{
    q.dfr_out = on && j == 0;
    q.dfr_in = on && j == 1;
    if (q.dfr_in) { q.dfr_lom = pl.p[0].lo + pl.p[0].m; q.dfr_gm = pl.p[0].m; }
}
/* a job of prime i on plane x, in one direction */
static PassJob prime_job(int i, double *x, uint64_t batch, bool inv)
{
    PassJob j; memset(&j, 0, sizeof j);
    j.x = x; j.batch = batch; j.p = g.pk[i].p; j.pinv = g.pk[i].pinv; j.tw = inv ? g.twi[i] : g.twf[i];
    return j;
}
/* bstride = 0: one prime after another, sharing the one B plane at Bp; bstride > 0: one launch per pass for every prime
 * and both operands, prime i's B plane at Bp + i bstride */
static int product_transforms(int np, int logn, int r3, uint64_t cnt, double *A, double *Bp, uint64_t bstride,
                              const uint64_t *a, uint64_t na, const uint64_t *b, uint64_t nb, const LoadDesc *ldesc,
                              hipStream_t s, hipEvent_t *pev, uint64_t cnt_b = 0, const LoadDesc *ldesc_b = nullptr,
                              const uint32_t *bmap = nullptr, uint64_t *stamps = nullptr, bool inv_crt = false)
{
    if (!bmap) { cnt_b = cnt; ldesc_b = ldesc; }
    const uint64_t tb = r3 ? 3 * cnt : cnt, tbb = r3 ? 3 * cnt_b : cnt_b;   /* engine transforms of 2^logn points */
    Plan pl; product_plan(&pl, logn, tb, product_tile_log(logn));
    Plan plb; product_plan(&plb, logn, tbb, product_tile_log(logn));
    const uint64_t n = (uint64_t)1 << logn, plane = tb * n, ntot = r3 ? 3 * n : n;
    const int last = pl.npass - 1;
    if (bmap && (plb.npass != pl.npass || pl.p[last].m + pl.p[last].logh > logn || (last == 0 && !r3)))
        return nttm_fail(NTTM_EINVAL, "internal: shared B operands on this length");
    if (inv_crt && (last != 1 || !nttm_inv_crt_ok(logn, pl.p[0].lo, pl.p[0].m)))
        return nttm_fail(NTTM_EINVAL, "internal: no CRT with the inverse pass at this length");
    /* both operands' strided passes in one launch where every prime is too, and where their geometry is the same (it
     * differs only in the blocks a tile spans, by the powers of two in the two batch counts) */
    bool pair = bstride > 0;
    for (int j = 0; j < last; j++) if (memcmp(&pl.p[j], &plb.p[j], sizeof(PassGeom))) pair = false;
    const int step = bstride ? np : 1;
    for (int i0 = 0; i0 < np; i0 += step) {
        JobSet jb, ja, ji;                                         /* B, A, A's inverse */
        FusedSet jf;                                               /* the double-fused pass */
        memset(&jb, 0, sizeof jb); memset(&ja, 0, sizeof ja); memset(&jf, 0, sizeof jf); memset(&ji, 0, sizeof ji);
        jb.n = ja.n = jf.n = ji.n = step;
        for (int k = 0; k < step; k++) {
            const int i = i0 + k;
            const uint64_t p = NTTM_PRIMES[i];
            double *Ai = A + (size_t)i * plane, *Bi = Bp + (size_t)i * bstride;
            const double2 ninv = h_shoup(h_inv(ntot % p, p), p);     /* the inverse's 1/length, folded into B */
            jb.j[k] = prime_job(i, Bi, tbb, false);
            jb.j[k].limbs = ldesc_b ? nullptr : b; jb.j[k].nlimbs = nb; jb.j[k].ldesc = ldesc_b; jb.j[k].which = 1;
            jb.j[k].in_scale = ninv; jb.j[k].do_in_scale = 1;
            ja.j[k] = prime_job(i, Ai, tb, false);
            ja.j[k].limbs = ldesc ? nullptr : a; ja.j[k].nlimbs = na; ja.j[k].ldesc = ldesc; ja.j[k].which = 0;
            jf.j[k] = FusedJob{Ai, Bi, g.pk[i].p, g.pk[i].pinv, g.twf[i].stage, g.twi[i].stage, ninv};
            ji.j[k] = prime_job(i, Ai, tb, true);
        }
        /* the forward passes but the last, of the given jobs; the first reads the operand limbs (a radix-3 layer does
         * where there is one).  j0: the jobs as the caller set them up */
        auto forward = [&](JobSet js, const Plan &q, uint64_t *stamp) -> int {
            auto limbs_done = [&]() { for (int k = 0; k < js.n; k++) { PassJob &j = js.j[k]; j.limbs = nullptr; j.ldesc = nullptr; j.do_in_scale = 0; } };
            if (r3) {
                JobSet r = js;
                for (int k = 0; k < r.n; k++) r.j[k].batch /= 3;
                RCK(nttm_run_r3(false, logn, r, s, stamp));
                stamp = nullptr;
                limbs_done();
            }
            PassArgs f = base_args(i0, js.j[0].x, logn, js.j[0].batch, false);
            f.limbs = js.j[0].limbs; f.nlimbs = js.j[0].nlimbs; f.ldesc = js.j[0].ldesc;
            const bool dfr = !r3 && defer_ok(f, q, last);
            for (int j = 0; j < last; j++) {
                defer_set(f, q, j, dfr);
                f.stamp = j == 0 ? stamp : nullptr;
                if (dfr && j == 0) for (int k = 0; k < js.n; k++) js.j[k].dfr_do_scale = js.j[k].do_in_scale;
                RCK(nttm_run_pass(false, f, q.p[j], s, &js));
                f.limbs = nullptr; f.ldesc = nullptr;
                limbs_done();
            }
            return 0;
        };
        if (pair && (last > 0 || r3)) {
            JobSet all = jb;
            for (int k = 0; k < step; k++) all.j[all.n++] = ja.j[k];
            if (pev) HIPCK(hipEventRecord(pev[2 * i0], s));
            RCK(forward(all, pl, stamps));
            if (pev) HIPCK(hipEventRecord(pev[2 * i0 + 1], s));
        } else {
            if (pev) HIPCK(hipEventRecord(pev[2 * i0], s));
            if (last > 0 || r3) RCK(forward(jb, plb, stamps));
            if (pev) HIPCK(hipEventRecord(pev[2 * i0 + 1], s));
            if (last > 0 || r3) RCK(forward(ja, pl, nullptr));
        }
        /* B's last forward pass, A's last forward pass, the pointwise product and A's first inverse pass */
        PassArgs fa = base_args(i0, jf.j[0].x, logn, tb, false);
        FusedB fb{nullptr, 0, nullptr, bmap};
        fa.stamp = stamps ? stamps + 1 : nullptr;
        if (last == 0 && !r3) {                                  /* a single-pass transform reads both operands here */
            fa.limbs = ldesc ? nullptr : a; fa.nlimbs = na; fa.ldesc = ldesc; fa.which = 0;
            fb.limbs = ldesc ? nullptr : b; fb.nlimbs = nb; fb.ldesc = ldesc;
        }
        RCK(nttm_run_fused2(fa, fb, pl.p[last], s, jf));
        PassArgs ia = base_args(i0, ji.j[0].x, logn, tb, true);
        for (int j = last - 1; j >= (inv_crt ? 1 : 0); j--) RCK(nttm_run_pass(true, ia, pl.p[j], s, &ji));
        if (r3) {
            for (int k = 0; k < step; k++) ji.j[k].batch = cnt;
            RCK(nttm_run_r3(true, logn, ji, s));
        }
    }
    return 0;
}

/* HBM bytes per point of a 2^logn transform of one prime in the product schedule (both operands' forward
 * transforms, the double-fused pass, the inverse; limb reads and the CRT excluded: equal for both lengths) */
static double sched_bytes(int logn, int r3, int tile_log)
{
    static double memo[NTTM_LOGN_MAX + 1][2][2];                 /* per length, radix, tile 12 / 13 (0: not yet) */
    const bool cacheable = logn >= 0 && logn <= NTTM_LOGN_MAX && (tile_log == 12 || tile_log == 13);
    double *m = cacheable ? &memo[logn][r3 ? 1 : 0][tile_log - 12] : nullptr;
    if (m && *m > 0) return *m;
    Plan pl; product_plan(&pl, logn, 1, product_tile_log(logn, tile_log));
    const int P = pl.npass;
    const double v = r3 ? 3.0 * (2 * (8 + 16 * (P - 1)) + 24 + 16 * (P - 1) + 16)
                        : (P >= 2 ? 2 * (8 + 16 * (P - 2)) + 24 + 16 * (P - 1) : 8);
    if (m) *m = v;
    return v;
}
/* the transform length of a product with ncoef coefficients: 2^logn, or 3 2^(logn - 2) when it fits and the rule
 * (NTTM_R3_*) takes it (the reference takes it whenever it fits, E/rns_mul.c:270-277) */
static void choose_len(uint64_t ncoef, int mode, int tile_log, int *logn_out, int *r3_out)
{
    int logn = ceil_log2(ncoef); if (logn < NTTM_PRODUCT_LOGN_MIN) logn = NTTM_PRODUCT_LOGN_MIN;
    int r3 = 0;
    if (mode != NTTM_R3_NEVER && logn - 2 >= NTTM_PRODUCT_LOGN_MIN && ncoef <= ((uint64_t)3 << (logn - 2)))
        r3 = mode == NTTM_R3_FIT ||
             sched_bytes(logn - 2, 1, tile_log) * ldexp(1.0, logn - 2) < sched_bytes(logn, 0, tile_log) * ldexp(1.0, logn);
    *logn_out = r3 ? logn - 2 : logn; *r3_out = r3;
}
static void choose_len(uint64_t ncoef, int *logn_out, int *r3_out)
{
    choose_len(ncoef, g.cfg.radix3, g.cfg.tile_log, logn_out, r3_out);
}

/* c = a b (+ x), device pointers; synchronous (returns after the stream has drained) */
/* the one-transform schedule of an na x nb product writing nc limbs: primes, length and workspace bytes; nonzero when
 * no transform holds it (the prime set's bound, or more than 2^32 points) */
struct OnePlan { int np, logn, r3; uint64_t n; size_t planes_bytes, crt_words, ws_bytes; };
static int one_plan(size_t na, size_t nb, size_t nc, OnePlan *o)
{
    const int want = g.cfg.nprimes;
    const size_t mn = na < nb ? na : nb;
    o->np = want ? want : (uint64_t)mn <= max_terms_np(3) ? 3 : 4;
    if ((uint64_t)mn > max_terms_np(o->np)) return 1;
    choose_len(na + nb - 1, &o->logn, &o->r3);
    if (o->logn > NTTM_LOGN_MAX) return 1;
    o->n = (uint64_t)(o->r3 ? 3 : 1) << o->logn;
    o->planes_bytes = (size_t)(o->np + 1) * o->n * 8;
    o->crt_words = nttm_crt_scratch_words(std::max(nttm_crt_blocks(nc), prod_crt_blocks(o->logn, o->r3, o->n, nc)));
    o->ws_bytes = align_up(o->planes_bytes, 256) + 256 + o->crt_words * 4 + 256;
    return 0;
}
static bool fits_one(size_t na, size_t nb, size_t nc)
{
    OnePlan o;
    return !one_plan(na, nb, nc, &o) && (!g.cfg.workspace_bytes || o.ws_bytes <= g.cfg.workspace_bytes);
}

/* ---- uneven products -----------------------------------------------------------------------------------------------------
 * A product of a long operand (alen limbs) by a shorter one (blen) need not take one transform that holds both: the long one is
 * cut into cnt pieces of `step` limbs, each piece times the short operand fits a transform of n >= 2 blen points, all
 * pieces run as one batch that shares the short operand's transform, and the CRT adds the overlap of neighbouring pieces
 * (the first blen - 1 coefficients of a piece to the last ones of the piece before: sums of residues of one convolution,
 * so the bound of its coefficients is the whole product's).  It saves the short operand's forward transform at full
 * length, a pass where the pieces take two and the whole product three, and padding.  Per call, us, whole / in pieces:
 * 300000 x 300 limbs 87 / 70, 1000000 x 100000 176 / 147, 5000003 x 300007 568 / 374, 5000003 x 2000 545 / 305,
 * 20000000 x 1000000 2650 / 1950, 100000000 x 300 10500 / 5200; the rest of the plane lies where the model below sees less
 * than its error: 30011 x 2100 56 / 57, 5000003 x 1500000 681 / 700. */
struct Pieces { int logn, r3; uint64_t n, cnt, step; double us; };   /* cnt = 0: the product whole; us: the time to beat */
/* a product's time by its passes, us: 12 for the call, 7 per launch (its own and its first and last tiles') and, per point and prime, 2.4 ps for the limb pass and 1.6 more where it
 * reads limbs, 3.6 a forward and 3.3 an inverse strided pass (9-bit rows 1.0 and 0.8 more), 3.8 (and the limbs) and 3.0 the radix-3 layers, 7.6
 * the double-fused pass; the CRT 2.5 per coefficient, 3.3 from pieces (kernel times of products of 2^20 to 2^28 points).  A
 * partition of the device has its share of the CUs and of the memory */
static double passes_us(int np, int logn, int r3, uint64_t cnt, uint64_t alen, uint64_t blen)
{
    Plan pl; product_plan(&pl, logn, 1, product_tile_log(logn));
    const int st = pl.npass - 1;
    const double n = (double)(r3 ? 3 : 1) * ldexp(1.0, logn), ca = (double)cnt * n;
    double fwd = r3 ? 3.8 + 3.6 * st : st ? 2.4 + 3.6 * (st - 1) : 0.0, inv = 3.3 * st + (r3 ? 3.0 : 0.0);
    for (int j = 0; j < st; j++) if (pl.p[j].m == 9) { fwd += 1.0; inv += 0.8; }
    return 12.0 + 7.0 * (2 * st + (r3 ? 2 : 0) + 3) + (cnt > 1 ? 4.0 : 0.0) +
           1e-6 * NTTM_CUS / nttm_ncu() * np * (ca * (fwd + 7.6 + inv) + n * fwd + 1.6 * (double)(alen + blen) + (cnt > 1 ? 3.3 : 2.5) * (double)(alen + blen));
}
static Pieces choose_pieces(int np, size_t alen, size_t blen, int logn, int r3)
{
    Pieces best{0, 0, 0, 0, 0, 0.0};
    const uint64_t whole = (uint64_t)(r3 ? 3 : 1) << logn;
    /* in pieces where the model saves 8 us and a tenth: its error is up to 8 % either way, the descriptors take 4 us */
    double most = passes_us(np, logn, r3, 1, alen, blen);
    best.us = most = std::min(0.9 * most, most - 8.0);
    if (alen < 2 * blen || g_pieces_points == 0) return best;    /* (two pieces of at least blen limbs) */
    for (int l = 12; l <= 26; l++)
        for (int t = l == 12; t < 2; t++) {                      /* 2^l points from 2^13, 3 2^l from 3 2^12 */
            const uint64_t n = (uint64_t)(t ? 3 : 1) << l;
            if (n >= whole || n < 2 * (uint64_t)blen || (t && g.cfg.radix3 == NTTM_R3_NEVER)) continue;
            const uint64_t step = (n - blen + 1) & ~(uint64_t)31;        /* (aligned as the operand is) */
            if (step < 2048 || step < blen) continue;
            const uint64_t cnt = (alen + step - 1) / step;
            if (cnt < 2 || cnt > 0x100000) continue;
            const double us = passes_us(np, l, t, cnt, alen, blen);
            if (g_pieces_points < 0 ? us < most : n == (uint64_t)g_pieces_points) { most = us; best = Pieces{l, t, n, cnt, step, us}; }
        }
    return best;
}
/* whether products of this transform length run as one kernel each (small.hip): 2^k points up to 2^12 */
static bool small_len(int logn, int r3) { return !r3 && !g_no_small && nttm_small_log(logn) != 0; }
/* ---- products in segments of the result (k_segments): short operands of up to some 2000 limbs -------------------------------- */
static bool seg_forced(void) { return g_pieces_points == 1 << 12; }
static bool seg_allowed(uint64_t S) { return S && !g_no_small && (g_pieces_points < 0 || seg_forced()); }
/* the result shares memory with a or b: segments, which write limbs while others still read theirs, are not for it (the
 * passes read every limb of both before the first result limb is written; an x under the result is read from a copy,
 * x_apart) */
static bool shares(const uint64_t *c, size_t nc, const uint64_t *p, size_t n)
{
    return p && n && (uintptr_t)p < (uintptr_t)(c + nc) && (uintptr_t)c < (uintptr_t)(p + n);
}
static bool result_over_operands(const uint64_t *c, size_t nc, const uint64_t *a, size_t na, const uint64_t *b, size_t nb)
{
    return shares(c, nc, a, na) || shares(c, nc, b, nb);
}
/* one product: the segments of a workgroup that give it the least time, if that is below `most`; else 0 */
static uint32_t choose_segments(size_t nc, size_t blen, double most)
{
    const uint64_t S = nttm_seg_len(blen);
    if (!seg_allowed(S)) return 0;
    const uint64_t segs = (nc + S - 1) / S;
    if (segs > 0x7fffffffULL) return 0;
    return seg_choose(segs, S, most, nttm_ncu(), seg_forced());
}
/* a product of a batch, whose launches fill the device either way: segments against the passes and the CRT of its own length
 * at 17 ps a point and prime from 2^16 points, 1.5 more for each bit below (measured 17.3 there, 19 at 2^15, 21 at 2^14).  Both
 * sides in time of the whole device: a partition takes longer for either alike */
static bool batch_segments(const nttm_prod &q, int logn, int r3)
{
    const size_t na = q.na, nb = q.nb;
    const size_t alen = std::max(na, nb), blen = std::min(na, nb);
    const uint64_t S = nttm_seg_len(blen);
    if (!seg_allowed(S) || (uint64_t)na + nb > 0xffffffffULL) return false;
    if (result_over_operands(q.c, na + nb + (q.x ? 1 : 0), q.a, na, q.b, nb)) return false;
    if (seg_forced()) return true;
    if (small_len(logn, r3) || alen < 2 * blen) return false;
    const double segs = ceil((double)(na + nb) / (double)S);
    const double ps = 17.0 + 1.5 * std::max(0, 16 - logn - (r3 ? 1 : 0));
    return (segs * seg_us(S) + SEG_B_US * ceil(segs / 6)) / NTTM_CUS < 0.95 * ps * 3e-6 * (double)((uint64_t)(r3 ? 3 : 1) << logn);
}
/* the descriptors of the pieces and the map to their one B operand: written by a kernel, since nothing on the host would
 * live until a copy of them has run in a call that does not wait */
__global__ __launch_bounds__(256) void k_pieces(LoadDesc *ld, uint32_t *bmap, const uint64_t *a, uint64_t alen, uint64_t step,
                                                uint32_t cnt, const uint64_t *b, uint64_t blen, int r3)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= cnt) return;
    const uint64_t o = i * step;
    LoadDesc d; d.a = a + o; d.na = alen - o < step ? alen - o : step; d.b = b; d.nb = blen;
    ld[i] = d;
    if (!i) ld[cnt] = d;
    if (r3) { for (int j = 0; j < 3; j++) bmap[3 * i + j] = (uint32_t)j; }
    else bmap[i] = 0;
}

/* the workspace of a one-transform product: the planes, its CRT descriptor (the pieces' descriptors) and the CRT's scratch
 * (bytes from ws).  n: points of the transforms, plane: of one prime's plane of A */
struct CoreLayout { int np, logn, r3, par; uint32_t seg_per; uint64_t n, plane, ncoef, cnt, step; size_t nc, nc_full, off_desc, off_bmap, off_crt, bytes; };
/* allow_par: one launch per pass for all primes, each with its own B plane (in the library's workspace), or the product in
 * pieces or (allow_segs: no result over its operands) in segments */
static int core_layout(size_t na, size_t nb, bool has_x, size_t wcut, CoreLayout *L, bool allow_par = false, bool allow_segs = true)
{
    L->nc_full = na + nb + (has_x ? 1 : 0); L->nc = L->nc_full < wcut ? L->nc_full : wcut;
    RCK(choose_np(na < nb ? na : nb, &L->np));
    const uint64_t ncoef_full = na + nb - 1;
    L->ncoef = ncoef_full < L->nc ? ncoef_full : L->nc;           /* coefficients read */
    choose_len(ncoef_full, &L->logn, &L->r3);
    if (L->logn > NTTM_LOGN_MAX) return nttm_fail(NTTM_EBOUND, "transform length 2^%d above 2^%d", L->logn, NTTM_LOGN_MAX);
    L->n = L->plane = (uint64_t)(L->r3 ? 3 : 1) << L->logn;       /* points per plane */
    L->cnt = L->step = 0; L->off_bmap = 0; L->seg_per = 0;
    if (allow_par) {                                             /* (the library's own workspace) */
        const size_t alen = std::max(na, nb), blen = std::min(na, nb);
        const Pieces q = choose_pieces(L->np, alen, blen, L->logn, L->r3);
        if (allow_segs && !small_len(L->logn, L->r3) && (L->seg_per = choose_segments(L->nc, blen, q.us))) {
            L->step = nttm_seg_len(blen); L->cnt = (L->nc + L->step - 1) / L->step; L->par = 1;
            L->off_desc = L->off_crt = 0;
            L->bytes = nttm_crt_scratch_words(L->cnt) * 4 + 256;
            return 0;
        }
        if (q.cnt) {
            const uint64_t plane = q.cnt * q.n;
            const int par = L->np > 1 && plane <= g_par_points;
            const size_t off_desc = align_up((size_t)(L->np * plane + (par ? L->np : 1) * q.n) * 8, 256);
            const size_t off_bmap = off_desc + align_up((q.cnt + 1) * sizeof(LoadDesc), 256);
            const size_t off_crt = off_bmap + align_up((q.r3 ? 3 : 1) * q.cnt * 4, 256);
            const size_t bytes = off_crt + nttm_crt_scratch_words(nttm_crt_blocks(L->nc)) * 4 + 256;
            if (!g.cfg.workspace_bytes || bytes <= g.cfg.workspace_bytes) {
                L->logn = q.logn; L->r3 = q.r3; L->n = q.n; L->plane = plane; L->cnt = q.cnt; L->step = q.step; L->par = par;
                L->off_desc = off_desc; L->off_bmap = off_bmap; L->off_crt = off_crt; L->bytes = bytes;
                return 0;
            }
        }
    }
    /* np planes of A and one of B: B's transform of each prime is made just before A's of that prime; primes in one
     * launch take a B plane each */
    const size_t crt_words = nttm_crt_scratch_words(std::max(nttm_crt_blocks(L->nc), prod_crt_blocks(L->logn, L->r3, L->n, L->nc)));
    for (int par = allow_par && L->np > 1 && L->n <= g_par_points; par >= 0; par--) {
        const size_t planes_bytes = (size_t)(par ? 2 * L->np : L->np + 1) * L->n * 8;
        L->par = par;
        L->off_desc = align_up(planes_bytes, 256); L->off_crt = L->off_desc + 256;
        L->bytes = L->off_crt + crt_words * 4 + 256;
        if (!g.cfg.workspace_bytes || L->bytes <= g.cfg.workspace_bytes) break;   /* together only within the cap */
    }
    return 0;
}

static int run_small(int np, int logn, const LoadDesc *ld, const CrtDesc *cd, const LoadDesc *ld1, const CrtDesc *cd1,
                     uint64_t cnt, uint64_t *ncn, uint32_t *ctl, hipStream_t s, double bytes, uint64_t *stamps = nullptr)
{
    const int sl = nttm_small_log(logn);
    double2 ninv[NTTM_MAX_PRIMES];
    for (int i = 0; i < np; i++) { const uint64_t p = NTTM_PRIMES[i]; ninv[i] = h_shoup(h_inv((uint64_t)1 << sl, p), p); }
    return nttm_run_small(np, sl, ld, cd, ld1, cd1, cnt, ncn, ctl, g.twf, g.twi, ninv, g.cc, s, bytes, stamps);
}

static int run_segments(int np, const LoadDesc *ld, const CrtDesc *cd, const LoadDesc *ld1, const CrtDesc *cd1, uint64_t nprod,
                        uint64_t groups, uint32_t *scratch, uint32_t *ctl, hipStream_t s, double bytes, uint64_t *stamps = nullptr)
{
    double2 ninv[NTTM_MAX_PRIMES];
    for (int i = 0; i < np; i++) { const uint64_t p = NTTM_PRIMES[i]; ninv[i] = h_shoup(h_inv((uint64_t)1 << 12, p), p); }
    return nttm_run_segments(np, ld, cd, ld1, cd1, nprod, groups, g.twf, g.twi, ninv, g.cc, scratch, ctl, s, bytes, stamps);
}
/* c = a b (+ x), device pointers.  wcut: write only the low wcut limbs of the result (the value mod B^wcut; no check of
 * what lies above).  ws: the workspace (null: the library's, grown to fit; else ws_cap bytes of the caller's).
 * sync = 1: returns after the stream has drained and the CRT's flags are checked; sync = 0: returns after the launches,
 * the flags in pinned slot `slot` (g.hpin + 128 slot + 96, read by the caller after a synchronization).
 * Nothing is copied in either direction: the CRT's descriptor goes with its launches, and the carry scan writes the flags
 * straight to the pinned slot.  The phase times of a product whose primes run together come from the device clock
 * (stamps in pinned memory): an event costs 2.2 us of the call, a copy 3 us. */
static int mul_core(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, const uint64_t *x, size_t nx,
                    hipStream_t s, size_t wcut = SIZE_MAX, char *ws = nullptr, size_t ws_cap = 0, int sync = 1,
                    size_t slot = 0)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    const size_t nc_full = na + nb + (x ? 1 : 0), nc = nc_full < wcut ? nc_full : wcut;
    if (x && nx > na + nb) return nttm_fail(NTTM_EINVAL, "nx = %zu exceeds na + nb = %zu", nx, na + nb);
    if (!c && nc) return nttm_fail(NTTM_EINVAL, "null result pointer");
    if ((na && !a) || (nb && !b) || (nx && !x)) return nttm_fail(NTTM_EINVAL, "null operand pointer");
    if (!na || !nb) {
        if (nc) HIPCK(hipMemsetAsync(c, 0, nc * 8, s));
        if (x && nx && nc) HIPCK(hipMemcpyAsync(c, x, (nx < nc ? nx : nc) * 8, hipMemcpyDeviceToDevice, s));
        if (sync) HIPCK(hipStreamSynchronize(s));
        else ((uint32_t *)((char *)g.hpin + 128 * slot + 96))[1] = 0;
        return 0;
    }
    if (!nc) return 0;
    CoreLayout L; RCK(core_layout(na, nb, x != nullptr, wcut, &L, !ws, !result_over_operands(c, nc, a, na, b, nb)));
    uint32_t *ctl = (uint32_t *)((char *)g.hpin + 128 * slot + 96);
    CrtDesc hd; memset(&hd, 0, sizeof hd);
    hd.plane = L.plane; hd.ncoef = L.ncoef; hd.x = x; hd.nx = x ? nx : 0; hd.c = c; hd.nc = nc; hd.first_block = 0;
    hd.trunc = nc < nc_full;
    if (!L.cnt && small_len(L.logn, L.r3)) {
        const LoadDesc ld{a, na, b, nb};
        RCK(run_small(L.np, L.logn, nullptr, nullptr, &ld, &hd, 1, nullptr, ctl, s, 8.0 * (double)(na + nb + nc + hd.nx),
                      sync ? g.stamps : nullptr));
        if (!sync) return 0;
        HIPCK(hipStreamSynchronize(s));
        g.last_stamped = 1; g.last_b = 0.5;
        return ctl[1] & 1 ? nttm_fail(NTTM_ECHECK, "crt: non-zero carry beyond the top limb (wrong residues)") : 0;
    }
    if (ws) {
        if (L.bytes > ws_cap) return nttm_fail(NTTM_EINVAL, "the product needs %zu bytes of workspace, above the %zu given", L.bytes, ws_cap);
    } else {
        int rc = ws_need(L.bytes);
        if (rc == NTTM_ENOMEM && L.par + L.cnt) {                 /* the device is nearly full: whole, prime after prime */
            RCK(core_layout(na, nb, x != nullptr, wcut, &L));
            rc = ws_need(L.bytes);
        }
        RCK(rc);
        ws = g.ws;
        hd.plane = L.plane;
    }
    if (L.seg_per) {
        const bool sw = na < nb;
        const LoadDesc ld{sw ? b : a, sw ? nb : na, sw ? a : b, sw ? na : nb};
        hd.step = L.step; hd.over = L.seg_per;
        uint64_t *st = sync ? g.stamps : nullptr;
        RCK(run_segments(L.np, nullptr, nullptr, &ld, &hd, 1, (L.cnt + L.seg_per - 1) / L.seg_per, (uint32_t *)ws, ctl, s,
                         8.0 * (double)(na + nb + nc + hd.nx), st));
        RCK(nttm_crt_launch_carry(nullptr, &hd, 1, L.cnt, (uint32_t *)ws, ctl, s, NTTM_CRT_SEGS, st ? st + 4 : nullptr));
        if (!sync) return 0;
        HIPCK(hipStreamSynchronize(s));
        g.last_stamped = 1; g.last_b = 0.0;
        return ctl[1] & 1 ? nttm_fail(NTTM_ECHECK, "crt: non-zero carry beyond the top limb (wrong residues)") : 0;
    }
    double *A = (double *)ws, *Bp = A + (size_t)L.np * L.plane;
    uint32_t *crt_scr = (uint32_t *)(ws + L.off_crt);
    const bool events = sync && !L.par;
    uint64_t *stamps = sync && L.par ? g.stamps : nullptr;
    if (stamps) stamps[0] = ~(uint64_t)0;                        /* (a transform of one pass has no forward launch) */

    if (events) HIPCK(hipEventRecord(g.ev[0], s));
    const int im = L.cnt ? 0 : inv_crt_bits(L.logn, L.r3, 1);
    if (L.cnt) {
        const bool sw = na < nb;
        const uint64_t alen = sw ? nb : na, blen = sw ? na : nb;
        LoadDesc *ld = (LoadDesc *)(ws + L.off_desc);
        uint32_t *bmap = (uint32_t *)(ws + L.off_bmap);
        hipLaunchKernelGGL(k_pieces, dim3((unsigned)((L.cnt + 255) / 256)), dim3(256), 0, s, ld, bmap, sw ? b : a, alen, L.step,
                           (uint32_t)L.cnt, sw ? a : b, blen, L.r3);
        RCK(nttm_hip_check(hipGetLastError(), "k_pieces launch"));
        RCK(product_transforms(L.np, L.logn, L.r3, L.cnt, A, Bp, L.par ? L.n : 0, nullptr, 0, nullptr, 0, ld, s,
                               events ? g.pev : nullptr, 1, ld + L.cnt, bmap, stamps));
        hd.step = L.step; hd.tn = L.n; hd.over = blen - 1; hd.alen = alen;
    } else
        RCK(product_transforms(L.np, L.logn, L.r3, 1, A, Bp, L.par ? L.n : 0, a, na, b, nb, nullptr, s, events ? g.pev : nullptr, 0,
                               nullptr, nullptr, stamps, im != 0));
    if (events) HIPCK(hipEventRecord(g.ev[2], s));
    hd.pl = A;
    const double crt_bytes = 8.0 * L.np * (double)L.ncoef + 8.0 * (double)nc + 8.0 * (double)(x ? (nx < nc ? nx : nc) : 0);
    if (im) {
        RCK(nttm_run_inv_crt(L.np, im, nullptr, &hd, 1, g.twi, g.cc, crt_scr, ctl, 1, s, crt_bytes, stamps ? stamps + 2 : nullptr));
        RCK(nttm_crt_launch_carry(nullptr, &hd, 1, nttm_inv_crt_blocks(im), crt_scr, ctl, s, NTTM_CRT_RUNS, stamps ? stamps + 3 : nullptr));
    } else
        RCK(nttm_crt_launch_one(hd, nttm_crt_blocks(nc), L.np, g.cc, crt_scr, ctl, s, crt_bytes, stamps ? stamps + 2 : nullptr));
    if (events) HIPCK(hipEventRecord(g.ev[3], s));
    if (!sync) return 0;
    HIPCK(hipStreamSynchronize(s));
    g.last_stamped = stamps != nullptr;
    g.last_b = L.cnt ? 1.0 / (double)(1 + L.cnt) : 0.5;          /* (the pieces share one transform of B) */
    if (events) {
        float ms, tb = 0, t;
        for (int i = 0; i < L.np; i++) { HIPCK(hipEventElapsedTime(&t, g.pev[2 * i], g.pev[2 * i + 1])); tb += t; }
        HIPCK(hipEventElapsedTime(&ms, g.ev[0], g.ev[2]));
        g.last_ms[0] = tb; g.last_ms[1] = ms - tb;
        HIPCK(hipEventElapsedTime(&ms, g.ev[2], g.ev[3])); g.last_ms[2] = ms;
    }
    const uint32_t flags = ctl[1];
    if (flags & 1) return nttm_fail(NTTM_ECHECK, "crt: non-zero carry beyond the top limb (wrong residues)");
    return 0;
}

/* ---- the residue post-condition ------------------------------------------------------------------------------------
 * c = a b + x modulo the prime NTTM_CHECK_Q = 4611686018427388039 (the first prime above 2^62).  The reference's
 * "detect and retry" checks the same identity on residues it tracks through the run (level 2, E/dr.h:1-8,
 * ALGORITHM.md:441-458, modulo the same prime DR_Q); here the residues are computed from the arrays themselves on the
 * device after the product, every array of a call in 64Ki-limb chunks by one kernel (k_res_chunks), the chunks of an
 * array weighted by powers of B^65536 on the host.  Costs one read of a, b, x and c. */
#define NTTM_CHECK_Q 4611686018427388039ULL
struct ResChunkH { const uint64_t *x; uint64_t n; };          /* must match digits.hip's ResChunk */
/* the cyclic product of length L = 2^logn or 3 2^logn (at least 16 points): v[0 .. L + 3) = sum_k c_k B^k over the
 * cyclic convolution c_k = sum_(i + j = k mod L) a_i b_j, i.e. a b mod (x^L - 1) at x = B before its carries wrap (the
 * caller folds v modulo B^L - 1).  The transforms are DFTs of length L, so the pointwise product gives the cyclic
 * convolution directly; each c_k has at most min(na, nb) terms, the bound of an ordinary product.  na, nb <= L, device
 * pointers.  flag null: synchronous; else the launches only, *flag the pinned word that the carry launch writes (bit 0
 * set: a carry beyond the top limb), read by the caller after it synchronizes the stream.  The Newton reciprocal's
 * wrapped product (GMP's mpn_mulmod_bnm1 plays this part there). */
int nttm_mul_cyclic(uint64_t *v, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, size_t L, hipStream_t s,
                    const uint32_t **flag)
{
    if (flag) *flag = nullptr;
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    int logn = -1, r3 = 0;
    if (L >= 16 && !(L & (L - 1))) logn = __builtin_ctzll(L);
    else if (L % 3 == 0 && L / 3 >= 16 && !((L / 3) & (L / 3 - 1))) { logn = __builtin_ctzll(L / 3); r3 = 1; }
    if (logn < NTTM_PRODUCT_LOGN_MIN || logn > NTTM_LOGN_MAX)
        return nttm_fail(NTTM_EINVAL, "cyclic product: length %zu is not 2^k or 3 2^k (k in [%d, %d])", L,
                         NTTM_PRODUCT_LOGN_MIN, NTTM_LOGN_MAX);
    if (na > L || nb > L) return nttm_fail(NTTM_EINVAL, "cyclic product: operands of %zu and %zu limbs above %zu", na, nb, L);
    if (!v || (na && !a) || (nb && !b)) return nttm_fail(NTTM_EINVAL, "cyclic product: null pointer");
    const size_t nc = L + 3;
    if (!na || !nb) { HIPCK(hipMemsetAsync(v, 0, nc * 8, s)); return flag ? 0 : nttm_hip_check(hipStreamSynchronize(s), "cyclic product"); }
    int np; RCK(choose_np(na < nb ? na : nb, &np));
    bool par = L <= g_par_points;
    size_t planes_bytes = (size_t)(par ? 2 * np : np + 1) * L * 8;
    const size_t crt_bytes = nttm_crt_scratch_words(nttm_crt_blocks(nc)) * 4 + 256;
    int rc = ws_need(align_up(planes_bytes, 256) + 256 + crt_bytes);
    if (rc == NTTM_ENOMEM && par) {                               /* above the cap, or the device is nearly full */
        par = false; planes_bytes = (size_t)(np + 1) * L * 8;
        rc = ws_need(align_up(planes_bytes, 256) + 256 + crt_bytes);
    }
    RCK(rc);
    const size_t off_desc = align_up(planes_bytes, 256), off_crt = off_desc + 256;
    double *A = (double *)g.ws, *Bp = A + (size_t)np * L;
    RCK(product_transforms(np, logn, r3, 1, A, Bp, par ? L : 0, a, na, b, nb, nullptr, s, nullptr));
    CrtDesc hd; memset(&hd, 0, sizeof hd);
    hd.pl = A; hd.plane = L; hd.ncoef = L; hd.c = v; hd.nc = nc;
    uint32_t *ctl = (uint32_t *)((char *)g.hpin + 96);            /* the flags, written by the carry scan */
    RCK(nttm_crt_launch_one(hd, nttm_crt_blocks(nc), np, g.cc, (uint32_t *)(g.ws + off_crt), ctl, s, 8.0 * np * L + 8.0 * nc));
    if (flag) { *flag = ctl + 1; return 0; }
    HIPCK(hipStreamSynchronize(s));
    if (ctl[1] & 1) return nttm_fail(NTTM_ECHECK, "cyclic product: crt: non-zero carry beyond the top limb");
    return 0;
}

extern "C" int nttm_debug_mul_cyclic(uint64_t *v, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, size_t L,
                                     void *stream)
{
    if ((na && nttm_require_device(a, na * 8, "a")) || (nb && nttm_require_device(b, nb * 8, "b")) ||
        nttm_require_device(v, (L + 3) * 8, "v"))
        return nttm_fail(NTTM_EINVAL, "nttm_debug_mul_cyclic: device pointers only");
    return nttm_mul_cyclic(v, a, na, b, nb, L, (hipStream_t)stream, nullptr);
}
/* the transform length (points) the product rule gives `need` coefficients: a supported length of the cyclic product */
size_t nttm_wrap_len(size_t need)
{
    int logn, r3;
    choose_len(need ? need : 1, &logn, &r3);
    return (size_t)(r3 ? 3 : 1) << logn;
}

int nttm_run_res_chunks(const void *chunks_dev, uint64_t nchunks, uint64_t q, uint64_t *out_dev, hipStream_t s);
uint64_t nttm_res_chunk_limbs(void);
static int chk_need(size_t bytes)
{
    if (bytes <= g.chk_bytes) return 0;
    if (g.chk) { HIPCK(hipDeviceSynchronize()); HIPCK(hipFree(g.chk)); g.chk = nullptr; g.chk_bytes = 0; }
    if (hipMalloc(&g.chk, bytes) != hipSuccess) { (void)hipGetLastError(); return nttm_fail(NTTM_ENOMEM, "residue check: %zu bytes", bytes); }
    g.chk_bytes = bytes;
    return 0;
}
/* res[i] = (sum_k arr[i][k] B^k) mod NTTM_CHECK_Q for device arrays; synchronizes */
static int residues_q(uint64_t *res, const uint64_t *const *arr, const size_t *len, size_t count, hipStream_t s)
{
    const uint64_t CH = nttm_res_chunk_limbs(), q = NTTM_CHECK_Q;
    std::vector<ResChunkH> ch;
    std::vector<size_t> owner;
    for (size_t i = 0; i < count; i++) {
        res[i] = 0;
        for (size_t off = 0; off < len[i]; off += CH) {
            ch.push_back({arr[i] + off, std::min<uint64_t>(CH, len[i] - off)});
            owner.push_back(i);
        }
    }
    if (ch.empty()) return 0;
    const size_t off_out = align_up(ch.size() * sizeof(ResChunkH), 256);
    RCK(chk_need(off_out + ch.size() * 8));
    std::vector<uint64_t> out(ch.size());
    HIPCK(hipMemcpyAsync(g.chk, ch.data(), ch.size() * sizeof(ResChunkH), hipMemcpyHostToDevice, s));
    RCK(nttm_run_res_chunks(g.chk, ch.size(), q, (uint64_t *)(g.chk + off_out), s));
    HIPCK(hipMemcpyAsync(out.data(), g.chk + off_out, ch.size() * 8, hipMemcpyDeviceToHost, s));
    HIPCK(hipStreamSynchronize(s));
    const uint64_t bch = h_powmod(NTTM_B % q, CH, q);
    uint64_t w = 1;
    for (size_t k = 0; k < ch.size(); k++) {
        if (k == 0 || owner[k] != owner[k - 1]) w = 1;
        res[owner[k]] = (uint64_t)(((u128)out[k] * w + res[owner[k]]) % q);
        w = h_mulmod(w, bch, q);
    }
    return 0;
}
/* the post-condition over N products on device memory: NTTM_ECHECK naming the first that fails */
static int check_products(const nttm_prod *P, size_t N, hipStream_t s)
{
    std::vector<const uint64_t *> arr(4 * N);
    std::vector<size_t> len(4 * N);
    for (size_t i = 0; i < N; i++) {
        const nttm_prod &q = P[i];
        arr[4 * i] = q.a; len[4 * i] = q.na;
        arr[4 * i + 1] = q.b; len[4 * i + 1] = q.nb;
        arr[4 * i + 2] = q.x; len[4 * i + 2] = q.x ? q.nx : 0;
        arr[4 * i + 3] = q.c; len[4 * i + 3] = q.na + q.nb + (q.x ? 1 : 0);
    }
    std::vector<uint64_t> r(4 * N);
    RCK(residues_q(r.data(), arr.data(), len.data(), 4 * N, s));
    for (size_t i = 0; i < N; i++) {
        const uint64_t want = (uint64_t)(((u128)r[4 * i] * r[4 * i + 1] + r[4 * i + 2]) % NTTM_CHECK_Q);
        if (want != r[4 * i + 3])
            return nttm_fail(NTTM_ECHECK, "product %zu: c differs from a b + x modulo %llu (the residue post-condition)", i,
                             (unsigned long long)NTTM_CHECK_Q);
    }
    return 0;
}

/* ---- products above one transform: the grid (E/rns_dist.c:610-700, our own form) ---------------------------------------
 * A product that no single transform holds (more than 2^32 points, the prime set's term bound, or the configured
 * workspace cap) is formed from ka x kb piece products a_i b_j (pieces of ceil(na/ka) and ceil(nb/kb) limbs).  The grid
 * takes the fewest plane points in total, then the fewest pieces (i, j <= 64).  Each piece is added into c at limb
 * o = oa + ob by one product with the window c[o .. o + la + lb) as its x (c = a_i b_j + window, written back), and its
 * top limb (0 or 1) carried into c above the window on the device.  The cuts skip whole pieces: a piece at or above
 * limb w only adds a multiple of B^w, and one ending at or below lowcut is left out (the caller reads the limbs above
 * lowcut and tolerates what those pieces would have carried into them, E/rns_dist.c:678-679). */
static int grid_shape(size_t na, size_t nb, int *ka, int *kb)
{
    double best = 0; *ka = *kb = 0;
    for (int i = 1; i <= 64; i++)
        for (int j = 1; j <= 64; j++) {
            const size_t pa = (na + i - 1) / i, pb = (nb + j - 1) / j;
            if (!fits_one(pa, pb, pa + pb + 1)) continue;
            OnePlan o; one_plan(pa, pb, pa + pb + 1, &o);
            const double cost = (double)i * j * (double)o.n;
            if (!*ka || cost < best || (cost == best && i * j < *ka * *kb)) { best = cost; *ka = i; *kb = j; }
        }
    if (!*ka) return nttm_fail(NTTM_EBOUND, "no grid of at most 64 x 64 pieces forms a %zu x %zu-limb product", na, nb);
    return 0;
}
static int tmp_need(size_t limbs)
{
    if (limbs <= g.tmp_limbs) return 0;
    if (g.tmp) { HIPCK(hipDeviceSynchronize()); HIPCK(hipFree(g.tmp)); g.tmp = nullptr; g.tmp_limbs = 0; }
    if (hipMalloc(&g.tmp, limbs * 8) != hipSuccess) { (void)hipGetLastError(); return nttm_fail(NTTM_ENOMEM, "hipMalloc of %zu limbs failed", limbs); }
    g.tmp_limbs = limbs;
    return 0;
}
static int mul_grid(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, const uint64_t *x,
                    size_t nx, hipStream_t s, size_t lowcut, size_t w)
{
    const size_t nc_full = na + nb + (x ? 1 : 0), nout = nc_full < w ? nc_full : w;
    int ka, kb; RCK(grid_shape(na, nb, &ka, &kb));
    const size_t pa = (na + ka - 1) / ka, pb = (nb + kb - 1) / kb;
    RCK(tmp_need(pa + pb + 1));
    HIPCK(hipMemsetAsync(c, 0, nout * 8, s));
    if (x && nx) HIPCK(hipMemcpyAsync(c, x, (nx < nout ? nx : nout) * 8, hipMemcpyDeviceToDevice, s));
    for (int j = 0; j < kb; j++)
        for (int i = 0; i < ka; i++) {
            const size_t oa = (size_t)i * pa, ob = (size_t)j * pb;
            if (oa >= na || ob >= nb) continue;
            const size_t la = na - oa < pa ? na - oa : pa, lb = nb - ob < pb ? nb - ob : pb, o = oa + ob, len = la + lb;
            if (o >= nout || o + len <= lowcut) continue;             /* at or above w; below the low cut */
            const size_t wp = nout - o;                               /* limbs of c from o on */
            if (wp <= len) {                                          /* the piece reaches the top: mod B^wp */
                RCK(mul_core(g.tmp, a + oa, la, b + ob, lb, c + o, wp, s, wp));
                HIPCK(hipMemcpyAsync(c + o, g.tmp, wp * 8, hipMemcpyDeviceToDevice, s));
            } else {
                RCK(mul_core(g.tmp, a + oa, la, b + ob, lb, c + o, len, s));
                HIPCK(hipMemcpyAsync(c + o, g.tmp, len * 8, hipMemcpyDeviceToDevice, s));
                RCK(nttm_run_add_carry(c + o + len, wp - len, g.tmp + len, s));
            }
        }
    HIPCK(hipStreamSynchronize(s));
    return 0;
}
/* ---- a result over its own x -------------------------------------------------------------------------------------------
 * The CRT's kernels read x while they write c, and a run's or block's first lanes need the limbs of x just before their
 * own, which another run may have overwritten where the two share memory (the quotient of such a limb differs at every
 * second edge).  Such an x is copied ahead into memory of the library's and read from there; an empty operand's c = x and the
 * residue post-condition, which reads x again, take the copy too. */
#define XCOPY_MAX 32
struct XCopy { const uint64_t *src[XCOPY_MAX]; uint64_t *dst[XCOPY_MAX]; uint64_t n[XCOPY_MAX]; };
__global__ __launch_bounds__(256) void k_copy_x(XCopy a)
{
    const uint64_t *src = a.src[blockIdx.y], n = a.n[blockIdx.y];
    uint64_t *dst = a.dst[blockIdx.y];
    for (uint64_t k = (uint64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (uint64_t)gridDim.x * 256) dst[k] = src[k];
}
static int xc_need(size_t limbs)
{
    if (limbs <= g.xc_limbs) return 0;
    if (g.xc) { HIPCK(hipDeviceSynchronize()); HIPCK(hipFree(g.xc)); g.xc = nullptr; g.xc_limbs = 0; }
    if (hipMalloc(&g.xc, limbs * 8) != hipSuccess) { (void)hipGetLastError(); return nttm_fail(NTTM_ENOMEM, "copy of x: %zu limbs", limbs); }
    g.xc_limbs = limbs;
    return 0;
}
/* whether a product's x is to be copied.  The one-kernel products read all of x before they write (every: copied too, for a
 * caller that may give them another length) */
static bool x_to_copy(const nttm_prod &q, bool every)
{
    const size_t nc = q.na + q.nb + (q.x ? 1 : 0);
    if (!shares(q.c, nc, q.x, q.nx)) return false;
    if (every || g.cfg.check || !q.na || !q.nb) return true;
    int logn, r3;
    choose_len(q.na + q.nb - 1, &logn, &r3);
    return !small_len(logn, r3) || !fits_one(q.na, q.nb, nc);
}
/* limbs of the copies of N products; their launches, the copies back to back from dst, and the products with their x there */
static size_t x_limbs(const nttm_prod *P, size_t N, bool every)
{
    size_t n = 0;
    for (size_t i = 0; i < N; i++) if (x_to_copy(P[i], every)) n += P[i].nx;
    return n;
}
static int copy_x(nttm_prod *Q, size_t N, bool every, uint64_t *dst, hipStream_t s)
{
    XCopy a;
    int k = 0;
    uint64_t most = 0;
    auto flush = [&]() -> int {
        if (!k) return 0;
        const uint64_t blocks = std::min<uint64_t>((most + 2047) / 2048, 1024);   /* (8 limbs a thread) */
        hipLaunchKernelGGL(k_copy_x, dim3((unsigned)blocks, (unsigned)k), dim3(256), 0, s, a);
        k = 0; most = 0;
        return nttm_hip_check(hipGetLastError(), "k_copy_x launch");
    };
    for (size_t i = 0; i < N; i++) {
        if (!x_to_copy(Q[i], every)) continue;
        a.src[k] = Q[i].x; a.dst[k] = dst; a.n[k] = Q[i].nx; k++;
        most = std::max<uint64_t>(most, Q[i].nx);
        Q[i].x = dst; dst += Q[i].nx;
        if (k == XCOPY_MAX) RCK(flush());
    }
    return flush();
}
/* Q: left empty, or (an x under its result) P with those x operands copied */
static int x_apart(const nttm_prod *P, size_t N, std::vector<nttm_prod> &Q, hipStream_t s)
{
    const size_t n = x_limbs(P, N, false);
    if (!n) return 0;
    RCK(xc_need(n));
    Q.assign(P, P + N);
    return copy_x(Q.data(), N, false, g.xc, s);
}

/* one transform when it holds the product, else the grid */
static int mul_any(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, const uint64_t *x, size_t nx,
                   hipStream_t s, size_t lowcut = 0, size_t w = SIZE_MAX)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    const size_t nc_full = na + nb + (x ? 1 : 0), nout = nc_full < w ? nc_full : w;
    if (!na || !nb || !nout || fits_one(na, nb, nout)) return mul_core(c, a, na, b, nb, x, nx, s, w);
    if (x && nx > na + nb) return nttm_fail(NTTM_EINVAL, "nx = %zu exceeds na + nb = %zu", nx, na + nb);
    if (!c || !a || !b || (nx && !x)) return nttm_fail(NTTM_EINVAL, "null pointer");
    return mul_grid(c, a, na, b, nb, x, nx, s, lowcut, w);
}
/* mul_any and, with nttm_config.check, the residue post-condition on a whole product (w = SIZE_MAX) */
static int mul_full(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, const uint64_t *x, size_t nx,
                    hipStream_t s, size_t lowcut = 0, size_t w = SIZE_MAX)
{
    nttm_prod q; memset(&q, 0, sizeof q);
    q.a = a; q.na = na; q.b = b; q.nb = nb; q.c = c; q.x = x; q.nx = x ? nx : 0;
    std::vector<nttm_prod> Q;
    RCK(x_apart(&q, 1, Q, s));
    if (!Q.empty()) { q = Q[0]; x = q.x; }
    RCK(mul_any(c, a, na, b, nb, x, nx, s, lowcut, w));
    if (!g.cfg.check || w != SIZE_MAX) return 0;
    return check_products(&q, 1, s);
}

/* c = a b on device memory without a synchronization where it fits one transform (no residue check configured): the
 * launches only, *flag the pinned word that the product's last launch writes (bit 0 set: a carry beyond the top limb), which
 * the caller reads after synchronizing the stream; *flag = null when the product ran synchronously (a grid) */
int nttm_mul_launch(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, hipStream_t s,
                    const uint32_t **flag)
{
    *flag = nullptr;
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (!na || !nb || g.cfg.check || !fits_one(na, nb, na + nb)) return mul_full(c, a, na, b, nb, nullptr, 0, s);
    RCK(mul_core(c, a, na, b, nb, nullptr, 0, s, SIZE_MAX, nullptr, 0, 0, 0));
    *flag = (const uint32_t *)((char *)g.hpin + 96) + 1;
    return 0;
}

extern "C" int nttm_last_phase_ms(double *f, double *i, double *c)
{
    if (g.last_stamped) {                                        /* a product whose primes ran together */
        int khz = 0;
        if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, g.dev) != hipSuccess || khz <= 0) { (void)hipGetLastError(); khz = 100000; }
        const uint64_t *t = g.stamps;
        auto ms = [&](uint64_t a, uint64_t b) { return b > a ? (double)(b - a) / khz : 0.0; };
        if (g.last_b > 0) {
            const double fwd = ms(t[0], t[1]);                   /* both operands' forward passes, one launch each */
            g.last_ms[0] = g.last_b * fwd; g.last_ms[1] = (1.0 - g.last_b) * fwd + ms(t[1], t[2]); g.last_ms[2] = ms(t[2], t[3]);
        } else {                                                 /* segments: the launch shared out as its first workgroup's time was */
            const double all = ms(t[0], t[4]), own = ms(t[0], t[2]), unit = own > 0 ? all / own : 0.0;
            g.last_ms[0] = unit * ms(t[0], t[1]); g.last_ms[2] = unit * ms(0, t[3]); g.last_ms[1] = all - g.last_ms[0] - g.last_ms[2];
        }
    }
    if (f) *f = g.last_ms[0];
    if (i) *i = g.last_ms[1];
    if (c) *c = g.last_ms[2];
    return 0;
}

/* ---- batches ---------------------------------------------------------------------------------------------------------- */
/* one length group of a batch: its products' descriptors and their layout in device memory (offsets from the group's
 * descriptor base), for a given schedule (length, strided-pass tile, points per thread) */
struct GroupBuild {
    int r3 = 0, logn = 0, tile = 0, pts = 0;
    int crt_per = 8;                                             /* CRT limbs per thread: 1 when every product is small */
    int inv_m = 0;                                               /* the last inverse pass's bits where the CRT runs it */
    uint64_t n = 0, cnt = 0, cnt_b = 0, nblk = 0;
    bool share = false, merged = false, small = false;
    uint32_t seg_per = 0;                                        /* r3 = 2: products in segments, this many a workgroup */
    uint64_t seg_groups = 0;
    struct Chunk { uint64_t c0, cn, b0, cnb, blk0, nblk; double crt_bytes; };   /* products, distinct B operands, CRT blocks */
    std::vector<Chunk> chunk;
    std::vector<CrtDesc> cd;
    std::vector<LoadDesc> ld, ldb;
    std::vector<uint32_t> bmap;
    size_t planes_bytes = 0;                                     /* (np cnt + cnt_b) n doubles */
    size_t off_cd = 0, off_ld = 0, off_ldb = 0, off_bmap = 0, off_ctl = 0, off_ncn = 0, off_crt = 0, desc_bytes = 0;
};
/* how a group of cnt products of n points runs: the products that run together (a chunk; the next one reuses their planes), and
 * whether all primes of a chunk share a launch per pass, each with a B plane of its own.  Under a cap on the planes' bytes
 * (0: none) fewer products a chunk, and where not even one has room for 2 np planes, prime after prime through np + 1 */
struct GroupShape {
    uint64_t cn;
    bool merged;
    size_t bytes(int np, uint64_t n) const { return (size_t)(merged ? 2 * np : np + 1) * cn * n * 8; }
};
static GroupShape group_shape(int np, uint64_t n, uint64_t cnt, size_t cap)
{
    GroupShape h;
    h.cn = std::min(cnt, std::max<uint64_t>(1, g_chunk_points / n));
    h.merged = n * h.cn <= std::max(g_chunk_points, g_par_points);
    if (!cap || h.bytes(np, n) <= cap) return h;
    const uint64_t room = cap / (n * 8);                         /* planes of one product */
    h.merged = h.merged && room >= 2 * (uint64_t)np;
    h.cn = std::max<uint64_t>(1, std::min(h.cn, room / (h.merged ? 2 * np : np + 1)));
    return h;
}
/* the workspace of the groups' planes under a cap (planes(cap) bytes); on a device nearly full, where that cannot be had, of the
 * least planes the groups run with, *cap set so that they are built for it */
template <typename F> static int ws_need_least(size_t *cap, F planes, bool defer = false)
{
    const int rc = ws_need(planes(*cap), defer);
    if (rc != NTTM_ENOMEM) return rc;
    *cap = 1;
    return ws_need(planes(*cap), defer);
}
#define SEG_CLASS (2 * (NTTM_LOGN_MAX + 1) + 12)   /* the group class of products in segments of 2^12 points (r3 = 2) */
static uint64_t seg_blocks(const nttm_prod &q)
{
    const uint64_t S = nttm_seg_len(std::min(q.na, q.nb)), nc = q.na + q.nb + (q.x ? 1 : 0);
    return (nc + S - 1) / S;
}
static void seg_sort(std::vector<size_t> &G, const nttm_prod *P)
{
    std::stable_sort(G.begin(), G.end(), [&](size_t u, size_t v) { return seg_blocks(P[u]) > seg_blocks(P[v]); });
}
static void group_offsets(GroupBuild &gb)
{
    gb.off_cd = 0;
    gb.off_ld = align_up(gb.off_cd + gb.cnt * sizeof(CrtDesc), 256);
    gb.off_ldb = align_up(gb.off_ld + gb.cnt * sizeof(LoadDesc), 256);
    gb.off_bmap = align_up(gb.off_ldb + gb.ldb.size() * sizeof(LoadDesc), 256);
    gb.off_ctl = align_up(gb.off_bmap + gb.bmap.size() * 4, 256);   /* a small group's flags, zeroed by the upload */
    gb.off_ncn = gb.off_ctl + 256;
    gb.off_crt = align_up(gb.off_ncn + gb.cnt * 8, 256);
    gb.desc_bytes = align_up(gb.off_crt + nttm_crt_scratch_words(gb.nblk) * 4, 256);
}
static void group_build_segments(GroupBuild &gb, const nttm_prod *P, const std::vector<size_t> &G)
{
    const uint64_t cnt = G.size();
    gb.n = (uint64_t)1 << gb.logn; gb.cnt = gb.cnt_b = cnt; gb.nblk = 0; gb.planes_bytes = 0; gb.inv_m = 0;
    gb.crt_per = NTTM_CRT_SEGS; gb.small = gb.share = false; gb.merged = true;
    gb.cd.assign(cnt, CrtDesc()); gb.ld.assign(cnt, LoadDesc()); gb.ldb.clear(); gb.bmap.clear();
    gb.chunk.assign(1, GroupBuild::Chunk{0, cnt, 0, cnt, 0, 0, 0.0});
    std::vector<uint64_t> blocks(cnt), lens(cnt);
    for (uint64_t j = 0; j < cnt; j++) { blocks[j] = seg_blocks(P[G[j]]); lens[j] = nttm_seg_len(std::min(P[G[j]].na, P[G[j]].nb)); }
    gb.seg_per = seg_batch_per(blocks.data(), lens.data(), cnt, nttm_ncu());
    gb.seg_groups = 0;
    for (uint64_t j = 0; j < cnt; j++) {
        const nttm_prod &q = P[G[j]];
        const bool sw = q.na < q.nb;
        gb.ld[j] = LoadDesc{sw ? q.b : q.a, sw ? q.nb : q.na, sw ? q.a : q.b, sw ? q.na : q.nb};
        CrtDesc &c = gb.cd[j];
        c.ncoef = q.na + q.nb - 1; c.x = q.x; c.nx = q.x ? q.nx : 0; c.c = q.c; c.nc = q.na + q.nb + (q.x ? 1 : 0);
        c.first_block = gb.nblk; c.step = nttm_seg_len(gb.ld[j].nb); c.tn = gb.seg_groups;
        const uint64_t sb = seg_blocks(q);
        const uint64_t groups = (sb + gb.seg_per - 1) / gb.seg_per;
        c.over = (sb + groups - 1) / groups;                     /* (evenly) */
        gb.nblk += sb; gb.seg_groups += groups;
        gb.chunk[0].crt_bytes += 8.0 * (double)(q.na + q.nb + c.nc + c.nx);
    }
    gb.chunk[0].nblk = gb.nblk;
    group_offsets(gb);
}
static void group_build(GroupBuild &gb, const nttm_prod *P, const std::vector<size_t> &G, int np, int r3, int logn,
                        int tile, int pts, size_t cap = 0)
{
    gb.r3 = r3; gb.logn = logn; gb.tile = tile; gb.pts = pts;
    if (r3 == 2) { group_build_segments(gb, P, G); return; }
    const uint64_t n = (uint64_t)(r3 ? 3 : 1) << logn, cnt = G.size();          /* points per product plane */
    gb.n = n; gb.cnt = cnt; gb.nblk = 0; gb.cnt_b = 0; gb.planes_bytes = 0;
    gb.inv_m = inv_crt_bits(logn, r3, cnt);
    gb.crt_per = gb.inv_m ? NTTM_CRT_RUNS : n <= 1024 ? 1 : 8;    /* (products of at most n + 1 limbs: 256-limb blocks) */
    gb.cd.assign(cnt, CrtDesc()); gb.ld.assign(cnt, LoadDesc()); gb.ldb.clear(); gb.bmap.clear(); gb.chunk.clear();
    gb.small = small_len(logn, r3);                              /* one kernel, no planes and no CRT blocks */
    const GroupShape shape = group_shape(np, n, cnt, cap);
    const uint64_t cmax = gb.small ? cnt : shape.cn;
    gb.merged = shape.merged;
    for (uint64_t c0 = 0; c0 < cnt; c0 += cmax) gb.chunk.push_back({c0, std::min(cmax, cnt - c0), 0, 0, 0, 0, 0.0});
    for (GroupBuild::Chunk &ch : gb.chunk) {
        ch.blk0 = gb.nblk;
        for (uint64_t j = ch.c0; j < ch.c0 + ch.cn; j++) {
            const nttm_prod &q = P[G[j]];
            LoadDesc &l = gb.ld[j];
            CrtDesc &c = gb.cd[j];
            l.a = q.a; l.na = q.na; l.b = q.b; l.nb = q.nb;
            c.pl = nullptr; c.plane = ch.cn * n; c.ncoef = q.na + q.nb - 1; c.x = q.x; c.nx = q.x ? q.nx : 0;
            c.c = q.c; c.nc = q.na + q.nb + (q.x ? 1 : 0); c.first_block = gb.nblk; c.trunc = 0;
            if (!gb.small) gb.nblk += gb.inv_m ? nttm_inv_crt_blocks(gb.inv_m) : nttm_crt_blocks(c.nc, gb.crt_per);
            ch.crt_bytes += gb.small ? 8.0 * (q.na + q.nb) + 8.0 * c.nc + 8.0 * c.nx : 8.0 * np * c.ncoef + 8.0 * c.nc + 8.0 * c.nx;
        }
        ch.nblk = gb.nblk - ch.blk0;
    }
    /* products that share their B operand (the same b and nb: the binary-splitting tree's P1 Q2 + P2 and Q1 Q2,
     * E/rns_mul.c:476-495) transform it once per chunk, where B has planes (a transform of more than one pass, or a
     * radix-3 length) and the double-fused tiles lie inside one transform */
    std::vector<uint32_t> slot(cnt);
    Plan pq; product_plan(&pq, logn, r3 ? 3 * cnt : cnt, product_tile_log(logn, tile));
    const bool can = !gb.small && logn >= NTTM_FUSED_LOG && (pq.npass > 1 || r3);
    if (can) gb.ldb.reserve(cnt);
    std::vector<uint32_t> tab;                                   /* open addressing: 1 + the chunk's B operand, 0 empty */
    for (GroupBuild::Chunk &ch : gb.chunk) {
        ch.b0 = gb.ldb.size();
        size_t cap = 16;
        while (can && cap < 2 * ch.cn) cap *= 2;
        if (can) tab.assign(cap, 0);
        for (uint64_t j = ch.c0; j < ch.c0 + ch.cn && can; j++) {
            const LoadDesc &l = gb.ld[j];
            size_t h = ((uintptr_t)l.b * 0x9E3779B97F4A7C15ULL ^ l.nb * 0xBF58476D1CE4E5B9ULL) >> 20;
            for (h &= cap - 1; tab[h]; h = (h + 1) & (cap - 1)) {
                const LoadDesc &o = gb.ldb[ch.b0 + tab[h] - 1];
                if (o.b == l.b && o.nb == l.nb) break;
            }
            if (!tab[h]) { gb.ldb.push_back(l); tab[h] = (uint32_t)(gb.ldb.size() - ch.b0); }
            slot[j] = tab[h] - 1;
        }
        ch.cnb = can ? gb.ldb.size() - ch.b0 : ch.cn;            /* no sharing: one B per product */
        gb.cnt_b += ch.cnb;
        if (!gb.small) gb.planes_bytes = std::max(gb.planes_bytes, ((size_t)np * ch.cn + (size_t)(gb.merged ? np : 1) * ch.cnb) * n * 8);
    }
    gb.share = gb.cnt_b < cnt;
    if (!gb.share) gb.ldb.clear();
    const uint64_t tb = r3 ? 3 * cnt : cnt;
    if (gb.share) {
        gb.bmap.resize(tb);
        for (uint64_t t = 0; t < tb; t++) gb.bmap[t] = r3 ? 3 * slot[t / 3] + (uint32_t)(t % 3) : slot[t];
    }
    group_offsets(gb);
}
/* points per thread of a batch group's passes: the configured value, else 8 up to 2^14 points and 16 above (what the
 * batch plans' autotuner chose for every such group of the 4096-leaf workload) */
static int batch_pts(int logn) { return g.cfg.pts ? g.cfg.pts : logn <= 14 ? 8 : 16; }
/* the group's descriptors as one host image (planes at A), to copy to the group's descriptor base */
static void group_image(GroupBuild &gb, double *A, char *img)
{
    for (const GroupBuild::Chunk &ch : gb.chunk)                     /* (the alignment gaps stay unread) */
        for (uint64_t j = 0; j < ch.cn; j++) gb.cd[ch.c0 + j].pl = A + j * gb.n;
    memcpy(img + gb.off_cd, gb.cd.data(), gb.cnt * sizeof(CrtDesc));
    memcpy(img + gb.off_ld, gb.ld.data(), gb.cnt * sizeof(LoadDesc));
    memset(img + gb.off_ctl, 0, 16);
    if (gb.share) {
        memcpy(img + gb.off_ldb, gb.ldb.data(), gb.ldb.size() * sizeof(LoadDesc));
        memcpy(img + gb.off_bmap, gb.bmap.data(), gb.bmap.size() * 4);
    }
}
/* the group's launches: transforms, CRT with the carries, normalized lengths; under the group's tile and points per thread
 * (the library's settings are restored afterwards).  ncn (or null: no lengths): cnt words, ctl: two words of flags, each in
 * device or pinned host memory */
static int group_launch(const GroupBuild &gb, int np, double *A, char *dbase, hipStream_t s, uint64_t *ncn, uint32_t *ctl)
{
    if (gb.small)
        return run_small(np, gb.logn, (const LoadDesc *)(dbase + gb.off_ld), (const CrtDesc *)(dbase + gb.off_cd), nullptr, nullptr,
                         gb.cnt, ncn, ncn ? nullptr : ctl, s, gb.chunk[0].crt_bytes);
    if (gb.seg_per) {
        uint32_t *scr = (uint32_t *)(dbase + gb.off_crt);
        const CrtDesc *cd = (const CrtDesc *)(dbase + gb.off_cd);
        RCK(run_segments(np, (const LoadDesc *)(dbase + gb.off_ld), cd, nullptr, nullptr, gb.cnt, gb.seg_groups, scr, ctl, s,
                         gb.chunk[0].crt_bytes));
        RCK(nttm_crt_launch_carry(cd, nullptr, gb.cnt, gb.nblk, scr, ctl, s, NTTM_CRT_SEGS));
        return ncn ? nttm_run_norm(cd, gb.cnt, ncn, s) : 0;
    }
    const int tile0 = g.cfg.tile_log, pts0 = nttm_get_pts();
    g.cfg.tile_log = gb.tile; nttm_set_pts(gb.pts);
    int rc = 0;
    for (const GroupBuild::Chunk &ch : gb.chunk) {               /* chunk after chunk through the same planes */
        double *Bp = A + (size_t)np * ch.cn * gb.n;
        const LoadDesc *ld = (const LoadDesc *)(dbase + gb.off_ld) + ch.c0;
        rc = product_transforms(np, gb.logn, gb.r3, ch.cn, A, Bp, gb.merged ? ch.cnb * gb.n : 0, nullptr, 0, nullptr, 0, ld, s,
                                nullptr, ch.cnb, gb.share ? (const LoadDesc *)(dbase + gb.off_ldb) + ch.b0 : nullptr,
                                gb.share ? (const uint32_t *)(dbase + gb.off_bmap) + (gb.r3 ? 3 : 1) * ch.c0 : nullptr, nullptr,
                                gb.inv_m != 0);
        if (!rc && gb.inv_m)
            rc = nttm_run_inv_crt(np, gb.inv_m, (const CrtDesc *)(dbase + gb.off_cd) + ch.c0, nullptr, ch.cn, g.twi, g.cc,
                                  (uint32_t *)(dbase + gb.off_crt), ctl, ch.c0 == 0, s, ch.crt_bytes, nullptr);
        else if (!rc) rc = nttm_crt_launch_limbs((const CrtDesc *)(dbase + gb.off_cd) + ch.c0, nullptr, ch.cn, ch.blk0, ch.nblk, np,
                                            g.cc, (uint32_t *)(dbase + gb.off_crt), ctl, s, ch.crt_bytes, gb.crt_per);
        if (rc) break;
    }
    uint32_t *scr = (uint32_t *)(dbase + gb.off_crt);
    if (!rc) rc = nttm_crt_launch_carry((const CrtDesc *)(dbase + gb.off_cd), nullptr, gb.cnt, gb.nblk, scr, ctl, s, gb.crt_per);
    if (!rc && ncn) rc = nttm_run_norm(dbase + gb.off_cd, gb.cnt, ncn, s);
    g.cfg.tile_log = tile0; nttm_set_pts(pts0);
    return rc;
}

/* device memory of the descriptors of a call's groups */
static int tdesc_need(size_t bytes, bool defer = false)
{
    if (bytes <= g.tdesc_bytes) return 0;
    if (g.tdesc) { RCK(drop_dev(g.tdesc, defer)); g.tdesc = nullptr; g.tdesc_bytes = 0; }
    if (hipMalloc(&g.tdesc, bytes) != hipSuccess) { (void)hipGetLastError(); return nttm_fail(NTTM_ENOMEM, "tree descriptors: %zu bytes", bytes); }
    g.tdesc_bytes = bytes;
    return 0;
}
/* the stream of the descriptor copies (the tree's and the batches') and its events */
static int side_stream(void)
{
    if (g.tcs) return 0;
    HIPCK(hipStreamCreateWithFlags(&g.tcs, hipStreamNonBlocking));
    for (int j = 0; j < 8; j++) HIPCK(hipEventCreateWithFlags(&g.tev[j], hipEventDisableTiming));
    return 0;
}

/* a group's lengths (as its launches wrote them) to put(j, n); true when a CRT's carry ran beyond a top limb.  A small group's
 * lengths carry their product's flag in bit 63; the others' flags are ctl's */
template <typename F> static bool group_lengths(const GroupBuild &gb, const uint64_t *ncn, const uint32_t *ctl, F put)
{
    bool bad = !gb.small && (ctl[1] & 1);
    for (uint64_t j = 0; j < gb.cnt; j++) {
        if (gb.small && ncn[j] >> 63) bad = true;
        put(j, ncn[j] & ~((uint64_t)1 << 63));
    }
    return bad;
}

/* the batch on device memory (every pointer of P classed MEM_DEV), no x to be copied */
static int mul_batch_apart(nttm_prod *P, size_t N, hipStream_t s)
{
    /* validate; zero-operand products are written directly */
    size_t mn_max = 0;
    /* groups by transform length: 2^logn at [logn], 3 2^logn at [NTTM_LOGN_MAX + 1 + logn] */
    std::vector<std::vector<size_t>> groups(SEG_CLASS + 1);      /* and the products in segments at SEG_CLASS */
    for (size_t i = 0; i < N; i++) {
        const nttm_prod &q = P[i];
        if (q.x && q.nx > q.na + q.nb) return nttm_fail(NTTM_EINVAL, "product %zu: nx exceeds na + nb", i);
        if (!q.c || (q.na && !q.a) || (q.nb && !q.b)) return nttm_fail(NTTM_EINVAL, "product %zu: null pointer", i);
        if (!q.na || !q.nb) continue;
        size_t mn = q.na < q.nb ? q.na : q.nb; if (mn > mn_max) mn_max = mn;
        int logn, r3;
        choose_len(q.na + q.nb - 1, &logn, &r3);
        if (logn > NTTM_LOGN_MAX) return nttm_fail(NTTM_EBOUND, "product %zu: transform above 2^%d", i, NTTM_LOGN_MAX);
        groups[batch_segments(q, logn, r3) ? SEG_CLASS : r3 * (NTTM_LOGN_MAX + 1) + logn].push_back(i);
    }
    int np; RCK(choose_np(mn_max ? mn_max : 1, &np));
    seg_sort(groups[SEG_CLASS], P);
    for (size_t i = 0; i < N; i++) {
        const nttm_prod &q = P[i];
        if (q.na && q.nb) continue;
        const size_t nc = q.na + q.nb + (q.x ? 1 : 0);
        if (nc) HIPCK(hipMemsetAsync(q.c, 0, nc * 8, s));
        if (q.x && q.nx) HIPCK(hipMemcpyAsync(q.c, q.x, q.nx * 8, hipMemcpyDeviceToDevice, s));
    }
    /* one group per transform length, the largest first: every group is enqueued without waiting for the one before, its
     * descriptors built on the host meanwhile and copied on a stream of their own (the first group's, which nothing
     * precedes, on the caller's), and the lengths and flags are written straight to pinned memory.  One
     * synchronization at the end.  (Waiting per group left the device idle for 0.9 of the 4096 leaves' 6.6 ms.) */
    std::vector<size_t> order;
    size_t cap = g.cfg.workspace_bytes, desc = 0, img = 0, words = 0;
    auto radix = [](size_t gi) { return (int)(gi / (NTTM_LOGN_MAX + 1)); };
    auto pts = [&](size_t gi) { return (uint64_t)(radix(gi) == 1 ? 3 : radix(gi) ? 8 : 1) << (gi % (NTTM_LOGN_MAX + 1)); };   /* (about 8 segments) */
    for (size_t gi = 0; gi < groups.size(); gi++) {
        const std::vector<size_t> &G = groups[gi];
        if (G.empty()) continue;
        order.push_back(gi);
        const int r3 = radix(gi), logn = (int)(gi % (NTTM_LOGN_MAX + 1));
        const uint64_t n = pts(gi), cnt = G.size();
        uint64_t blk = 0;
        for (size_t i : G) blk += r3 == 2 ? seg_blocks(P[i]) : prod_crt_blocks(logn, r3, n, P[i].na + P[i].nb + (P[i].x ? 1 : 0));
        const size_t im = align_up(cnt * sizeof(CrtDesc), 256) + 2 * align_up(cnt * sizeof(LoadDesc), 256) +
                          align_up((r3 ? 3 : 1) * cnt * 4, 256) + 512;
        img += im;
        desc += im + align_up(cnt * 8, 256) + align_up(nttm_crt_scratch_words(blk) * 4, 256) + 256;
        words += cnt + 2;
    }
    std::sort(order.begin(), order.end(), [&](size_t u, size_t v) { return pts(u) * groups[u].size() > pts(v) * groups[v].size(); });
    auto planes = [&](size_t c) {
        size_t most = 256;
        for (size_t gi : order) {
            const int logn = (int)(gi % (NTTM_LOGN_MAX + 1));
            if (radix(gi) != 2 && !small_len(logn, radix(gi))) most = std::max(most, group_shape(np, pts(gi), groups[gi].size(), c).bytes(np, pts(gi)));
        }
        return most;
    };
    RCK(ws_need_least(&cap, planes));
    RCK(tdesc_need(desc + 256));
    const size_t img0 = align_up(words * 8 + 256, 256);          /* the lengths and flags, then the descriptor images */
    RCK(hpin_need(img0 + img));
    if (order.size() > 1) {
        RCK(side_stream());
        HIPCK(hipStreamSynchronize(g.tcs));                      /* (a failed call's copies) */
    }
    uint64_t *hw = g.hpin;
    char *hi = (char *)g.hpin + img0;
    size_t dpos = 0, ipos = 0;
    std::vector<GroupBuild> gbs(order.size());
    auto enqueue = [&]() -> int {
        uint64_t *w = hw;
        for (size_t k = 0; k < order.size(); k++) {
            const std::vector<size_t> &G = groups[order[k]];
            GroupBuild &gb = gbs[k];
            const int logn = (int)(order[k] % (NTTM_LOGN_MAX + 1));
            group_build(gb, P, G, np, radix(order[k]), logn, g.cfg.tile_log, batch_pts(logn), cap);
            if (dpos + gb.desc_bytes > g.tdesc_bytes || ipos + gb.off_ncn > img || gb.planes_bytes > g.ws_bytes)
                return nttm_fail(NTTM_EINVAL, "internal: a batch group exceeds its sizing");
            char *dbase = g.tdesc + dpos;
            group_image(gb, (double *)g.ws, hi + ipos);
            const hipStream_t cs = k ? g.tcs : s;
            HIPCK(hipMemcpyAsync(dbase, hi + ipos, gb.off_ncn, hipMemcpyHostToDevice, cs));
            if (k) {
                hipEvent_t ev = g.tev[k % 8];
                HIPCK(hipEventRecord(ev, cs));
                HIPCK(hipStreamWaitEvent(s, ev, 0));
            }
            RCK(group_launch(gb, np, (double *)g.ws, dbase, s, w, (uint32_t *)(w + gb.cnt)));
            w += gb.cnt + 2;
            dpos = align_up(dpos + gb.desc_bytes, 256);
            ipos = align_up(ipos + gb.off_ncn, 256);
        }
        return 0;
    };
    const int rce = enqueue();
    if (rce) { (void)hipStreamSynchronize(s); return rce; }      /* nothing may still read the descriptors */
    HIPCK(hipStreamSynchronize(s));
    for (size_t k = 0; k < order.size(); k++) {
        const std::vector<size_t> &G = groups[order[k]];
        if (group_lengths(gbs[k], hw, (const uint32_t *)(hw + gbs[k].cnt), [&](uint64_t j, uint64_t n) { P[G[j]].ncn = n; }))
            return nttm_fail(NTTM_ECHECK, "crt: non-zero carry beyond a top limb (wrong residues)");
        hw += gbs[k].cnt + 2;
    }
    /* zero-operand products: normalized length of x */
    for (size_t i = 0; i < N; i++) {
        nttm_prod &q = P[i];
        if (q.na && q.nb) continue;
        size_t n = q.x ? q.nx : 0;
        HIPCK(hipStreamSynchronize(s));
        while (n) { uint64_t v; HIPCK(hipMemcpy(&v, q.x + n - 1, 8, hipMemcpyDeviceToHost)); if (v) break; n--; }
        q.ncn = n;
    }
    return g.cfg.check ? check_products(P, N, s) : 0;
}

static int mul_batch_dev(nttm_prod *P, size_t N, hipStream_t s)
{
    if (!N) return 0;
    std::vector<nttm_prod> Q;
    RCK(x_apart(P, N, Q, s));
    if (Q.empty()) return mul_batch_apart(P, N, s);
    const int rc = mul_batch_apart(Q.data(), N, s);
    for (size_t i = 0; i < N; i++) P[i].ncn = Q[i].ncn;
    return rc;
}

/* ---- host-resident operands: staging through HBM -----------------------------------------------------------------------
 * The products accept operands and results in host memory, as the reference's batch does: it reads registered host
 * memory in place and stages anything else through device buffers (E/rns_mul.h:42-47, E/rns_mul.c:807-817).  Kernels
 * here read HBM only, so every host input is copied into a library-owned device region (g.stage) before the products
 * and every host result copied back after them.  Copies go through a pinned bounce buffer of two halves, so that the
 * host copy into one half overlaps the DMA out of the other; pinned inputs and results of at least a half move by
 * DMA directly.  A host operand named by several products of one call (the shared B of a binary-splitting pair) is
 * copied once, so those products still share its transform.  A batch whose staged bytes exceed g.stage_chunk (1 GiB)
 * runs as consecutive sub-batches (a product larger than that is staged alone). */
/* host copies split over a few threads that live for one call (one thread copies about 10 GB/s, the link moves 50): run()
 * copies all pieces, cut into equal byte ranges, and returns when every thread has done its own */
struct CopyPiece { char *dst; const char *src; size_t n; };
class CopyTeam {
    std::vector<std::thread> th;
    const std::vector<CopyPiece> *job = nullptr;
    size_t total = 0;
    unsigned parts = 1;
    std::atomic<unsigned> gen{0}, left{0};
    std::atomic<bool> stop{false};
    void part(unsigned i)
    {
        const size_t lo = total / parts * i, hi = i + 1 == parts ? total : total / parts * (i + 1);
        size_t at = 0;
        for (const CopyPiece &p : *job) {
            const size_t a = std::max(lo, at), b = std::min(hi, at + p.n);
            if (a < b) memcpy(p.dst + (a - at), p.src + (a - at), b - a);
            at += p.n;
            if (at >= hi) break;
        }
    }
    void work(unsigned i)
    {
        for (unsigned seen = 0;;) {
            unsigned gnow;
            for (int spin = 0; (gnow = gen.load(std::memory_order_acquire)) == seen; spin++) {
                if (stop.load(std::memory_order_acquire)) return;
                if (spin > 200) std::this_thread::yield();
            }
            seen = gnow;
            part(i);
            left.fetch_sub(1, std::memory_order_release);
        }
    }
public:
    /* bytes: what the whole call will copy; short calls take no threads */
    explicit CopyTeam(size_t bytes, unsigned most)
    {
        const unsigned hw = std::thread::hardware_concurrency();
        const size_t want = std::min<size_t>({(size_t)most, (size_t)(hw ? hw : 1), bytes >> 20});
        try { for (size_t i = 1; i < want; i++) { th.emplace_back([this, i]() { work((unsigned)i); }); parts++; } }
        catch (...) { }                                          /* fewer threads then */
    }
    ~CopyTeam() { stop.store(true, std::memory_order_release); for (std::thread &t : th) t.join(); }
    CopyTeam(const CopyTeam &) = delete;
    void run(const std::vector<CopyPiece> &pieces)
    {
        job = &pieces; total = 0;
        for (const CopyPiece &p : pieces) total += p.n;
        left.store((unsigned)th.size(), std::memory_order_relaxed);
        gen.fetch_add(1, std::memory_order_release);
        part(0);
        while (left.load(std::memory_order_acquire)) std::this_thread::yield();
    }
};
#define NTTM_COPY_THREADS 4

#define NTTM_BOUNCE_HALF ((size_t)4 << 20)       /* bytes per half of the pinned bounce buffer */
#define NTTM_STAGE_ALIGN 256                     /* every staged array starts on a 256-byte boundary */

static int stage_need(size_t bytes)
{
    if (bytes <= g.stage_bytes) return 0;
    if (g.stage) { HIPCK(hipDeviceSynchronize()); HIPCK(hipFree(g.stage)); g.stage = nullptr; g.stage_bytes = 0; }
    if (hipMalloc(&g.stage, bytes) != hipSuccess) { (void)hipGetLastError(); return nttm_fail(NTTM_ENOMEM, "staging: hipMalloc of %zu bytes failed", bytes); }
    g.stage_bytes = bytes;
    return 0;
}
static int bounce_need(void)
{
    if (g.bounce) return 0;
    HIPCK(hipHostMalloc((void **)&g.bounce, 2 * NTTM_BOUNCE_HALF, hipHostMallocDefault));
    g.bounce_half = NTTM_BOUNCE_HALF;
    for (int k = 0; k < 2; k++) { HIPCK(hipEventCreateWithFlags(&g.bev[k], hipEventDisableTiming)); g.bev_live[k] = 0; }
    return 0;
}
static int bounce_wait(int h)                    /* the last copy through half h has completed */
{
    if (g.bev_live[h]) { HIPCK(hipEventSynchronize(g.bev[h])); g.bev_live[h] = 0; }
    return 0;
}

/* the host arrays of one staged call and their offsets in g.stage: the inputs first, then the results */
struct StageSet {
    struct Item { const void *p; size_t bytes; int kind; size_t off; };
    std::vector<Item> in, out;
    std::map<std::pair<const void *, size_t>, size_t> seen;
    size_t bytes = 0;
    size_t add_in(const void *p, size_t n, int kind)
    {
        const auto key = std::make_pair(p, n);
        const auto it = seen.find(key);
        if (it != seen.end()) return it->second;
        in.push_back({p, n, kind, 0});
        seen.emplace(key, in.size() - 1);
        return in.size() - 1;
    }
    size_t add_out(void *p, size_t n, int kind) { out.push_back({p, n, kind, 0}); return out.size() - 1; }
    void layout()
    {
        size_t o = 0;
        for (Item &i : in) { i.off = o; o = align_up(o + i.bytes, NTTM_STAGE_ALIGN); }
        for (Item &i : out) { i.off = o; o = align_up(o + i.bytes, NTTM_STAGE_ALIGN); }
        bytes = o ? o : NTTM_STAGE_ALIGN;
    }
    const uint64_t *din(size_t k) const { return (const uint64_t *)(g.stage + in[k].off); }
    uint64_t *dout(size_t k) const { return (uint64_t *)(g.stage + out[k].off); }
};

/* bytes per window of the copies through the bounce buffer: a quarter of the call's, so that the host's copies, the DMA
 * and (downloads) the copies out overlap, within the buffer's halves */
static size_t bounce_window(size_t total) { return std::min(g.bounce_half, std::max<size_t>((size_t)256 << 10, align_up(total / 4, 4096))); }

/* the inputs into g.stage: consecutive inputs are packed into a window of a bounce half, and a full window goes to the
 * device by one DMA while the host fills the other half (the alignment gaps are not copied over: stale, never read) */
static int stage_upload(const StageSet &st, hipStream_t s)
{
    if (st.in.empty()) return 0;
    RCK(bounce_need());
    const size_t half = g.bounce_half;
    size_t total = 0;
    for (const StageSet::Item &i : st.in) if (!(i.kind == MEM_PINNED && i.bytes >= half)) total += i.bytes;
    const size_t win = bounce_window(total);
    CopyTeam team(total, NTTM_COPY_THREADS);
    std::vector<CopyPiece> pc;
    int h = 0;
    size_t fill = 0, base = 0;                                   /* half h is to hold fill bytes for g.stage + base */
    auto flush = [&]() -> int {
        if (!fill) return 0;
        RCK(bounce_wait(h));
        team.run(pc);
        pc.clear();
        HIPCK(hipMemcpyAsync(g.stage + base, g.bounce + h * half, fill, hipMemcpyHostToDevice, s));
        HIPCK(hipEventRecord(g.bev[h], s)); g.bev_live[h] = 1;
        h ^= 1; fill = 0;
        return 0;
    };
    for (const StageSet::Item &i : st.in) {
        if (!i.bytes) continue;
        if (i.kind == MEM_PINNED && i.bytes >= half) {           /* pinned and large: one direct DMA */
            RCK(flush());
            HIPCK(hipMemcpyAsync(g.stage + i.off, i.p, i.bytes, hipMemcpyHostToDevice, s));
            continue;
        }
        const char *src = (const char *)i.p;
        size_t left = i.bytes, off = i.off;
        while (left) {
            if (fill && off - base >= win) RCK(flush());
            if (!fill) base = off;
            fill = off - base;                                   /* (past an alignment gap) */
            const size_t take = std::min(left, win - fill);
            pc.push_back({g.bounce + h * half + fill, src, take});
            fill += take; src += take; off += take; left -= take;
            if (fill == win) RCK(flush());
        }
    }
    return flush();
}

/* the results out of g.stage: windows DMA'd into alternating halves, each landed window copied to its host arrays while
 * the next one is in flight; pinned results of at least a half by DMA directly.  Returns after the stream has drained. */
static int stage_download(const StageSet &st, hipStream_t s)
{
    if (st.out.empty()) return nttm_hip_check(hipStreamSynchronize(s), "staging");
    RCK(bounce_need());
    const size_t half = g.bounce_half;
    struct Piece { char *dst; size_t off, bytes; };
    struct Win { size_t w0, w1, p0, p1; };                       /* device range, pieces [p0, p1) */
    size_t total = 0;
    for (const StageSet::Item &o : st.out) if (!(o.kind == MEM_PINNED && o.bytes >= half)) total += o.bytes;
    const size_t wmax = bounce_window(total);
    std::vector<Piece> pc;
    for (const StageSet::Item &o : st.out) {
        if (!o.bytes) continue;
        if (o.kind == MEM_PINNED && o.bytes >= half) {
            HIPCK(hipMemcpyAsync((void *)o.p, g.stage + o.off, o.bytes, hipMemcpyDeviceToHost, s));
            continue;
        }
        for (size_t k = 0; k < o.bytes; k += wmax) pc.push_back({(char *)o.p + k, o.off + k, std::min(wmax, o.bytes - k)});
    }
    std::vector<Win> win;
    for (size_t k = 0; k < pc.size(); k++) {
        if (!win.empty() && pc[k].off + pc[k].bytes - win.back().w0 <= wmax) { win.back().w1 = pc[k].off + pc[k].bytes; win.back().p1 = k + 1; }
        else win.push_back({pc[k].off, pc[k].off + pc[k].bytes, k, k + 1});
    }
    RCK(bounce_wait(0)); RCK(bounce_wait(1));
    CopyTeam team(total, NTTM_COPY_THREADS);
    std::vector<CopyPiece> cp;
    auto scatter = [&](size_t w) {
        const Win &x = win[w];
        const char *hb = g.bounce + (w & 1) * half;
        cp.clear();
        for (size_t k = x.p0; k < x.p1; k++) cp.push_back({pc[k].dst, hb + (pc[k].off - x.w0), pc[k].bytes});
        team.run(cp);
    };
    for (size_t w = 0; w < win.size(); w++) {
        const int h = (int)(w & 1);
        HIPCK(hipMemcpyAsync(g.bounce + h * half, g.stage + win[w].w0, win[w].w1 - win[w].w0, hipMemcpyDeviceToHost, s));
        HIPCK(hipEventRecord(g.bev[h], s)); g.bev_live[h] = 1;
        if (w) { RCK(bounce_wait(h ^ 1)); scatter(w - 1); }
    }
    if (!win.empty()) { RCK(bounce_wait((int)((win.size() - 1) & 1))); scatter(win.size() - 1); }
    return nttm_hip_check(hipStreamSynchronize(s), "staging");
}

/* one large device array to host memory.  Pinned destinations take one DMA.  Pageable ones above 1 MiB go through two
 * pinned halves: the DMA of chunk k overlaps the host copy of chunk k - 1, which is split over up to 8 threads (the
 * destination's pages are first touched there, so their faults are taken in parallel).  A chunk is an eighth of the array,
 * 1 to 64 MiB.  (The runtime's own copy to pageable memory moves 8 GB/s: 5.6 ms for 44 MB.)  Synchronizes. */
#define NTTM_DL_MIN ((size_t)1 << 20)
#define NTTM_DL_HALF ((size_t)64 << 20)
size_t nttm_copy_to_host_min(void) { return NTTM_DL_MIN; }
static size_t dl_chunk(size_t bytes) { return std::min(NTTM_DL_HALF, std::max(NTTM_DL_MIN, align_up(bytes / 8, 4096))); }
/* the pinned halves of nttm_copy_to_host for an array of that size, allocated ahead of the copy (pinning 128 MiB takes
 * milliseconds; a caller can run this on another host thread while the device works) */
int nttm_copy_to_host_prepare(size_t bytes)
{
    const size_t H = dl_chunk(bytes);
    if (g.dl && g.dl_half >= H) return 0;
    if (g.dl) { char *old = g.dl; g.dl = nullptr; g.dl_half = 0; HIPCK(hipHostFree(old)); }      /* (idle between copies) */
    char *dl = nullptr;
    HIPCK(hipHostMalloc((void **)&dl, 2 * H, hipHostMallocDefault));
    memset(dl, 0, 2 * H);                                        /* its pages touched here, not during the copy */
    for (int k = 0; k < 2; k++) if (!g.dlev[k]) HIPCK(hipEventCreateWithFlags(&g.dlev[k], hipEventDisableTiming));
    g.dl = dl; g.dl_half = H;
    return 0;
}
int nttm_copy_to_host(void *dst, const void *src, size_t bytes, hipStream_t s)
{
    if (!bytes) return nttm_hip_check(hipStreamSynchronize(s), "copy to host");
    MemMap mm;
    if (mm.kind(dst, bytes) == MEM_PINNED || bytes <= NTTM_DL_MIN) {
        HIPCK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
        return nttm_hip_check(hipStreamSynchronize(s), "copy to host");
    }
    RCK(nttm_copy_to_host_prepare(bytes));
    const size_t H = dl_chunk(bytes), nch = (bytes + H - 1) / H;
    CopyTeam team(bytes, 8);
    std::vector<CopyPiece> pc(1);
    auto host_copy = [&](size_t c) {
        const size_t off = c * H, len = std::min(H, bytes - off);
        pc[0] = {(char *)dst + off, g.dl + (c & 1) * g.dl_half, len};
        team.run(pc);
    };
    for (size_t c = 0; c < nch; c++) {
        const size_t off = c * H, len = std::min(H, bytes - off);
        HIPCK(hipMemcpyAsync(g.dl + (c & 1) * g.dl_half, (const char *)src + off, len, hipMemcpyDeviceToHost, s));
        HIPCK(hipEventRecord(g.dlev[c & 1], s));
        if (c) { HIPCK(hipEventSynchronize(g.dlev[(c - 1) & 1])); host_copy(c - 1); }
    }
    HIPCK(hipEventSynchronize(g.dlev[(nch - 1) & 1]));
    host_copy(nch - 1);
    return nttm_hip_check(hipStreamSynchronize(s), "copy to host");
}

/* the four pointers of a product classed (a, b, x, c with their byte counts); NTTM_EINVAL for memory no entry can use */
static int prod_kinds(MemMap &mm, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, const uint64_t *x, size_t nx,
                      const uint64_t *c, size_t nout, int *k, size_t idx)
{
    static const char *const nm[4] = {"a", "b", "x", "c"};
    k[0] = mm.kind(a, na * 8); k[1] = mm.kind(b, nb * 8); k[2] = x ? mm.kind(x, nx * 8) : MEM_DEV; k[3] = mm.kind(c, nout * 8);
    for (int j = 0; j < 4; j++)
        if (k[j] == MEM_BAD) return nttm_fail(NTTM_EINVAL, "product %zu: operand %s %s", idx, nm[j], mm.why);
    return 0;
}
static bool any_host(const int *k) { return k[0] != MEM_DEV || k[1] != MEM_DEV || k[2] != MEM_DEV || k[3] != MEM_DEV; }

/* one product with host memory among its operands (kinds k): staged, then formed on the device copies */
static int mul_staged(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, const uint64_t *x,
                      size_t nx, hipStream_t s, size_t lowcut, size_t w, const int *k)
{
    const size_t nc_full = na + nb + (x ? 1 : 0), nout = nc_full < w ? nc_full : w;
    StageSet st;
    const size_t ia = k[0] != MEM_DEV ? st.add_in(a, na * 8, k[0]) : SIZE_MAX;
    const size_t ib = k[1] != MEM_DEV ? st.add_in(b, nb * 8, k[1]) : SIZE_MAX;
    const size_t ix = k[2] != MEM_DEV ? st.add_in(x, nx * 8, k[2]) : SIZE_MAX;
    const size_t ic = k[3] != MEM_DEV ? st.add_out(c, nout * 8, k[3]) : SIZE_MAX;
    st.layout();
    RCK(stage_need(st.bytes));
    RCK(stage_upload(st, s));
    RCK(mul_full(ic == SIZE_MAX ? c : st.dout(ic), ia == SIZE_MAX ? a : st.din(ia), na, ib == SIZE_MAX ? b : st.din(ib), nb,
                 ix == SIZE_MAX ? x : st.din(ix), nx, s, lowcut, w));
    return stage_download(st, s);
}

/* the entry of the single products: device operands in place, host ones staged */
static int mul_entry(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, const uint64_t *x,
                     size_t nx, hipStream_t s, size_t lowcut = 0, size_t w = SIZE_MAX)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (x && nx > na + nb) return nttm_fail(NTTM_EINVAL, "nx = %zu exceeds na + nb = %zu", nx, na + nb);
    const size_t nc_full = na + nb + (x ? 1 : 0), nout = nc_full < w ? nc_full : w;
    MemMap mm;
    int k[4];
    RCK(prod_kinds(mm, a, na, b, nb, x, nx, c, nout, k, 0));
    if (!any_host(k)) return mul_full(c, a, na, b, nb, x, nx, s, lowcut, w);
    return mul_staged(c, a, na, b, nb, x, nx, s, lowcut, w, k);
}

extern "C" int nttm_mul(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, void *stream)
{
    return mul_entry(c, a, na, b, nb, nullptr, 0, (hipStream_t)stream);
}
extern "C" int nttm_mul_add(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, const uint64_t *x,
                            size_t nx, void *stream)
{
    if (!x) return nttm_fail(NTTM_EINVAL, "nttm_mul_add: null x");
    return mul_entry(c, a, na, b, nb, x, nx, (hipStream_t)stream);
}
/* the cut product (E/rns_dist.c:581-589,684-693; E/rns_mul.c rns_mul_local): the operands cut to their low w limbs,
 * the low min(na + nb, w) limbs of the product written.  A product that fits one transform is formed whole (the
 * reference skips no piece of it either); a grid skips the pieces ending at or below lowcut. */
extern "C" int nttm_mul_cut(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, size_t lowcut,
                            size_t w, void *stream)
{
    const size_t nout = na + nb < w ? na + nb : w;
    if (lowcut > nout) return nttm_fail(NTTM_EINVAL, "nttm_mul_cut: lowcut %zu above the %zu limbs written", lowcut, nout);
    return mul_entry(c, a, na < w ? na : w, b, nb < w ? nb : w, nullptr, 0, (hipStream_t)stream, lowcut, w);
}

/* c = a b with no allocation: the same product as nttm_mul on device memory, its planes, CRT descriptor and CRT scratch
 * in the file-scope array `scratch` of this GPU (NTTM_NOALLOC_BYTES = 40 MiB: one transform of at most 2^20 points on
 * three primes, e.g. 2^19 x 2^19 limbs).  No hipMalloc, hipFree or other allocating call: the operands are classed by
 * pointer queries without the per-call cache, live kernel timing is paused for the call, and a product that would
 * need more (a larger transform, four primes beyond the array, a grid, host operands) is refused with NTTM_EINVAL.
 * Nothing in the array must start at zero: the limb passes write every plane point before any read, and every CRT
 * block writes its status word and the carry scan its control words.  Calls that overlap on one GPU share the array
 * and race; calls in one stream or one after another are safe.  Synchronizes the stream. */
static int noalloc_dev_ok(const void *p, size_t bytes)
{
    if (!p || !bytes) return 1;
    hipPointerAttribute_t at;
    memset(&at, 0, sizeof at);
    if (hipPointerGetAttributes(&at, p) != hipSuccess) { (void)hipGetLastError(); return 0; }
    if (at.type != hipMemoryTypeDevice || at.device != g.dev) return 0;
    hipDeviceptr_t base = nullptr; size_t sz = 0;
    if (hipMemGetAddressRange(&base, &sz, (hipDeviceptr_t)p) != hipSuccess) { (void)hipGetLastError(); return 1; }
    return (uintptr_t)p + bytes <= (uintptr_t)base + sz;
}
extern "C" int nttm_mul_noalloc(uint64_t *c, const uint64_t *a, size_t na, const uint64_t *b, size_t nb, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    hipStream_t s = (hipStream_t)stream;
    if (g.dev >= NTTM_NOALLOC_MAX_DEV || !g_scratch_dev[g.dev]) return nttm_fail(NTTM_ESTATE, "nttm_mul_noalloc: no workspace on device %d", g.dev);
    if ((na && !a) || (nb && !b) || (na + nb && !c)) return nttm_fail(NTTM_EINVAL, "nttm_mul_noalloc: null pointer");
    if (!noalloc_dev_ok(a, na * 8) || !noalloc_dev_ok(b, nb * 8) || !noalloc_dev_ok(c, (na + nb) * 8))
        return nttm_fail(NTTM_EINVAL, "nttm_mul_noalloc: operands must be device memory of this device, inside their allocations");
    if (na && nb) {
        if (!fits_one(na, nb, na + nb)) return nttm_fail(NTTM_EINVAL, "nttm_mul_noalloc: a %zu x %zu-limb product needs a grid", na, nb);
        CoreLayout L; RCK(core_layout(na, nb, false, SIZE_MAX, &L));
        if (L.bytes > NTTM_NOALLOC_BYTES)
            return nttm_fail(NTTM_EINVAL, "nttm_mul_noalloc: a %zu x %zu-limb product needs %zu bytes of workspace, above the "
                             "%zu-byte maximum (one transform of at most 2^20 points on three primes)", na, nb, L.bytes,
                             (size_t)NTTM_NOALLOC_BYTES);
    }
    const int prof0 = g_prof_on;
    g_prof_on = 0;                                               /* event records could create events */
    const int rc = mul_core(c, a, na, b, nb, nullptr, 0, s, SIZE_MAX, g_scratch_dev[g.dev], NTTM_NOALLOC_BYTES);
    g_prof_on = prof0;
    return rc;
}

/* the residue post-condition on demand: c (nc limbs) = a b + x modulo NTTM_CHECK_Q; device memory; synchronizes */
extern "C" int nttm_check_product(const uint64_t *c, size_t nc, const uint64_t *a, size_t na, const uint64_t *b, size_t nb,
                                  const uint64_t *x, size_t nx, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if ((nc && !c) || (na && !a) || (nb && !b) || (nx && !x)) return nttm_fail(NTTM_EINVAL, "nttm_check_product: null pointer");
    DEVCK(c, nc * 8, "c"); DEVCK(a, na * 8, "a"); DEVCK(b, nb * 8, "b"); DEVCK(x, nx * 8, "x");
    const uint64_t *arr[4] = {a, b, x, c};
    const size_t len[4] = {na, nb, x ? nx : 0, nc};
    uint64_t r[4];
    RCK(residues_q(r, arr, len, 4, (hipStream_t)stream));
    if ((uint64_t)(((u128)r[0] * r[1] + r[2]) % NTTM_CHECK_Q) != r[3])
        return nttm_fail(NTTM_ECHECK, "c differs from a b + x modulo %llu (the residue post-condition)", (unsigned long long)NTTM_CHECK_Q);
    return 0;
}

extern "C" int nttm_mul_batch(nttm_prod *P, size_t N, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (!N) return 0;
    if (!P) return nttm_fail(NTTM_EINVAL, "nttm_mul_batch: null P");
    hipStream_t s = (hipStream_t)stream;
    MemMap mm;
    std::vector<int> k(4 * N);
    std::vector<size_t> est(N, 0);                               /* staged bytes per product */
    bool host = false;
    for (size_t i = 0; i < N; i++) {
        const nttm_prod &q = P[i];
        if (q.x && q.nx > q.na + q.nb) return nttm_fail(NTTM_EINVAL, "product %zu: nx exceeds na + nb", i);
        const size_t nc = q.na + q.nb + (q.x ? 1 : 0);
        int *ki = &k[4 * i];
        RCK(prod_kinds(mm, q.a, q.na, q.b, q.nb, q.x, q.nx, q.c, nc, ki, i));
        if (!any_host(ki)) continue;
        host = true;
        const size_t by[4] = {q.na * 8, q.nb * 8, q.x ? q.nx * 8 : 0, nc * 8};
        for (int j = 0; j < 4; j++) if (ki[j] != MEM_DEV) est[i] += align_up(by[j], NTTM_STAGE_ALIGN);
    }
    if (!host) return mul_batch_dev(P, N, s);
    /* sub-batches of at most NTTM_STAGE_CHUNK staged bytes */
    std::vector<size_t> idx;
    auto run = [&]() -> int {
        StageSet st;
        std::vector<size_t> ia(idx.size()), ib(idx.size()), ix(idx.size()), ic(idx.size());
        for (size_t j = 0; j < idx.size(); j++) {
            const nttm_prod &q = P[idx[j]];
            const int *ki = &k[4 * idx[j]];
            const size_t nc = q.na + q.nb + (q.x ? 1 : 0);
            ia[j] = ki[0] != MEM_DEV ? st.add_in(q.a, q.na * 8, ki[0]) : SIZE_MAX;
            ib[j] = ki[1] != MEM_DEV ? st.add_in(q.b, q.nb * 8, ki[1]) : SIZE_MAX;
            ix[j] = ki[2] != MEM_DEV ? st.add_in(q.x, q.nx * 8, ki[2]) : SIZE_MAX;
            ic[j] = ki[3] != MEM_DEV ? st.add_out(q.c, nc * 8, ki[3]) : SIZE_MAX;
        }
        st.layout();
        RCK(stage_need(st.bytes));
        RCK(stage_upload(st, s));
        std::vector<nttm_prod> D(idx.size());
        for (size_t j = 0; j < idx.size(); j++) {
            D[j] = P[idx[j]];
            if (ia[j] != SIZE_MAX) D[j].a = st.din(ia[j]);
            if (ib[j] != SIZE_MAX) D[j].b = st.din(ib[j]);
            if (ix[j] != SIZE_MAX) D[j].x = st.din(ix[j]);
            if (ic[j] != SIZE_MAX) D[j].c = st.dout(ic[j]);
        }
        RCK(mul_batch_dev(D.data(), D.size(), s));
        RCK(stage_download(st, s));
        for (size_t j = 0; j < idx.size(); j++) P[idx[j]].ncn = D[j].ncn;
        idx.clear();
        return 0;
    };
    size_t bytes = 0;
    for (size_t i = 0; i < N; i++) {
        if (!idx.empty() && bytes + est[i] > g.stage_chunk) { RCK(run()); bytes = 0; }
        idx.push_back(i); bytes += est[i];
    }
    return idx.empty() ? 0 : run();
}

/* the same N products, one product call each (the unbatched baseline of the batch tier); host memory staged per
 * product.  Every call synchronizes, and the normalized lengths are read back limb by limb. */
extern "C" int nttm_mul_each(nttm_prod *P, size_t N, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (N && !P) return nttm_fail(NTTM_EINVAL, "nttm_mul_each: null P");
    hipStream_t s = (hipStream_t)stream;
    MemMap mm;
    std::vector<int> k(4 * N);
    for (size_t i = 0; i < N; i++) {
        const nttm_prod &q = P[i];
        if (q.x && q.nx > q.na + q.nb) return nttm_fail(NTTM_EINVAL, "product %zu: nx exceeds na + nb", i);
        const size_t nc = q.na + q.nb + (q.x ? 1 : 0);
        int *ki = &k[4 * i];
        RCK(prod_kinds(mm, q.a, q.na, q.b, q.nb, q.x, q.nx, q.c, nc, ki, i));
        if (any_host(ki)) RCK(mul_staged(q.c, q.a, q.na, q.b, q.nb, q.x, q.nx, s, 0, SIZE_MAX, ki));
        else RCK(mul_full(q.c, q.a, q.na, q.b, q.nb, q.x, q.nx, s));
        P[i].ncn = nc;
    }
    /* normalized lengths: the top limbs read back */
    for (size_t i = 0; i < N; i++) {
        size_t n = P[i].ncn;
        if (k[4 * i + 3] != MEM_DEV) { while (n && !P[i].c[n - 1]) n--; }
        else while (n) {
            uint64_t v; HIPCK(hipMemcpy(&v, P[i].c + n - 1, 8, hipMemcpyDeviceToHost));
            if (v) break;
            n--;
        }
        P[i].ncn = n;
    }
    return 0;
}

/* the same N products, one product call each, launched back to back: no synchronization between products, one at the
 * end for every product's CRT flags, and the normalized lengths by one k_norm launch over all N.  Device memory only;
 * a product above one transform (a grid) runs synchronously inside the sequence. */
extern "C" int nttm_mul_each_async(nttm_prod *P, size_t N, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (!N) return 0;
    if (!P) return nttm_fail(NTTM_EINVAL, "nttm_mul_each_async: null P");
    hipStream_t s = (hipStream_t)stream;
    MemMap mm;
    size_t ws_max = 0;
    for (size_t i = 0; i < N; i++) {
        const nttm_prod &q = P[i];
        if (q.x && q.nx > q.na + q.nb) return nttm_fail(NTTM_EINVAL, "product %zu: nx exceeds na + nb", i);
        const size_t nc = q.na + q.nb + (q.x ? 1 : 0);
        int ki[4];
        RCK(prod_kinds(mm, q.a, q.na, q.b, q.nb, q.x, q.nx, q.c, nc, ki, i));
        if (any_host(ki)) return nttm_fail(NTTM_EINVAL, "nttm_mul_each_async: product %zu: host memory (device memory only)", i);
        if (q.na && q.nb && fits_one(q.na, q.nb, nc)) {                /* (with every prime's B plane) */
            CoreLayout L;
            RCK(core_layout(q.na, q.nb, q.x != nullptr, SIZE_MAX, &L, true, !result_over_operands(q.c, nc, q.a, q.na, q.b, q.nb)));
            ws_max = std::max(ws_max, L.bytes);
        }
    }
    const size_t off_ncn = align_up(N * sizeof(CrtDesc), 256);
    const int rcw = ws_need(ws_max);                             /* sized once: no reallocation between launches, but */
    if (rcw && rcw != NTTM_ENOMEM) return rcw;                   /* on a device nearly full, where each takes what it needs */
    RCK(hpin_need(128 * N + 8 * N + 256));
    RCK(stage_need(off_ncn + N * 8));
    std::vector<char> fl(N, 0);                                  /* 1: flags in pinned slot i */
    /* an x under its result is copied at its product's turn (x_apart): the products before it may have written it */
    std::vector<nttm_prod> Q(P, P + N);
    RCK(xc_need(x_limbs(P, N, false)));
    uint64_t *xd = g.xc;
    for (size_t i = 0; i < N; i++) {
        if (x_to_copy(P[i], false)) { RCK(copy_x(&Q[i], 1, false, xd, s)); xd += Q[i].nx; }
        const nttm_prod &q = Q[i];
        const size_t nc = q.na + q.nb + (q.x ? 1 : 0);
        if (q.na && q.nb && !fits_one(q.na, q.nb, nc)) RCK(mul_any(q.c, q.a, q.na, q.b, q.nb, q.x, q.nx, s));
        else { RCK(mul_core(q.c, q.a, q.na, q.b, q.nb, q.x, q.nx, s, SIZE_MAX, nullptr, 0, 0, i)); fl[i] = 1; }
    }
    std::vector<CrtDesc> cd(N);
    for (size_t i = 0; i < N; i++) { memset(&cd[i], 0, sizeof(CrtDesc)); cd[i].c = P[i].c; cd[i].nc = P[i].na + P[i].nb + (P[i].x ? 1 : 0); }
    HIPCK(hipMemcpyAsync(g.stage, cd.data(), N * sizeof(CrtDesc), hipMemcpyHostToDevice, s));
    RCK(nttm_run_norm(g.stage, N, (uint64_t *)(g.stage + off_ncn), s));
    uint64_t *hn = (uint64_t *)((char *)g.hpin + 128 * N);
    HIPCK(hipMemcpyAsync(hn, g.stage + off_ncn, N * 8, hipMemcpyDeviceToHost, s));
    HIPCK(hipStreamSynchronize(s));
    for (size_t i = 0; i < N; i++) {
        if (fl[i] && (((const uint32_t *)((char *)g.hpin + 128 * i + 96))[1] & 1))
            return nttm_fail(NTTM_ECHECK, "product %zu: crt: non-zero carry beyond the top limb (wrong residues)", i);
        P[i].ncn = hn[i];
    }
    return g.cfg.check ? check_products(Q.data(), N, s) : 0;
}

/* ---- the binary-splitting product tree ----------------------------------------------------------------------------------- */
static int bsp_need(int k, size_t limbs, bool defer = false)
{
    if (limbs <= g.bsp_limbs[k]) return 0;
    if (g.bsp[k]) { RCK(drop_dev(g.bsp[k], defer)); g.bsp[k] = nullptr; g.bsp_limbs[k] = 0; }
    if (hipMalloc(&g.bsp[k], limbs * 8) != hipSuccess) { (void)hipGetLastError(); return nttm_fail(NTTM_ENOMEM, "hipMalloc of %zu limbs failed", limbs); }
    g.bsp_limbs[k] = limbs;
    return 0;
}
/* ---- the binary-splitting tree planned on the host ---------------------------------------------------------------------
 * Every level's products take their operands' unnormalized lengths: a parent's P has |P_L| + |Q_R| + 1 limbs and its Q
 * |Q_L| + |Q_R| (top limbs possibly 0, which changes no value).  So every level's shape, grouping and pool layout is
 * known before any product runs, and the levels follow each other on the stream with no synchronization: the host
 * builds level k's descriptors while the device runs level k - 1 (a level's large groups in chunks of TREE_CHUNK
 * products), and copies them from a pinned image that no later group reuses.  One synchronization at the end reads every group's CRT flags and the root's top limbs (normalized
 * there).  The reference's level loop reads each level's lengths back before the next (E/binsplit.c:1583-1651).
 * Returns 1, having launched nothing, when a pair's |P_R| exceeds |P_L| + |Q_R| on the planned lengths or the residue
 * post-condition is configured (the level-by-level path handles both). */
int nttm_run_top_nonzero(const uint64_t *x, uint64_t n, uint64_t *out_dev, hipStream_t s);
static int tpin_need(size_t bytes, bool defer = false)
{
    if (bytes <= g.tpin_bytes) return 0;
    if (g.tpin) { RCK(drop_host(g.tpin, defer)); g.tpin = nullptr; g.tpin_bytes = 0; }
    HIPCK(hipHostMalloc((void **)&g.tpin, bytes, hipHostMallocDefault));
    g.tpin_bytes = bytes;
    return 0;
}
/* products per launched group: a level's large length group is launched in chunks, so that the device starts on the
 * first chunk while the host builds the next (the lowest levels have 10^5 products) */
#define TREE_CHUNK 16384
#define TREE_NKEY (2 * (NTTM_LOGN_MAX + 1))       /* transform-length classes: 2^logn at logn, 3 2^logn at 33 + logn */
/* the transform-length class of a product of ncoef coefficients.  choose_len depends on ncoef only through
 * lg = max(ceil_log2(ncoef), NTTM_PRODUCT_LOGN_MIN) and whether ncoef <= 3 2^(lg - 2), so each of those pairs is
 * resolved once, on a representative ncoef of the pair */
struct LenClass {
    int8_t key[65][2];
    LenClass() { memset(key, -1, sizeof key); }
    int operator()(uint64_t ncoef)
    {
        int lg = 63 - __builtin_clzll(ncoef | 1); if (((uint64_t)1 << lg) < ncoef) lg++;
        if (lg < NTTM_PRODUCT_LOGN_MIN) lg = NTTM_PRODUCT_LOGN_MIN;
        const int f = ncoef <= ((uint64_t)3 << (lg - 2));
        if (key[lg][f] < 0) {
            int logn, r3;
            choose_len(f ? (uint64_t)3 << (lg - 2) : (uint64_t)1 << lg, &logn, &r3);
            key[lg][f] = (int8_t)(r3 * (NTTM_LOGN_MAX + 1) + logn);
        }
        return key[lg][f];
    }
};
static_assert(TREE_NKEY <= 127, "length classes fit int8_t");
static int bs_tree_planned(const nttm_bs_node *leaves, size_t n, uint64_t *p, size_t p_cap, size_t *pn, uint64_t *q,
                           size_t q_cap, size_t *qn, hipStream_t s)
{
    if (g.cfg.check || n < 2) return 1;
    struct Len { size_t pn, qn; };
    std::vector<std::vector<Len>> len(1, std::vector<Len>(n));
    for (size_t i = 0; i < n; i++) len[0][i] = {leaves[i].pn, leaves[i].qn};
    while (len.back().size() > 1) {
        const std::vector<Len> &c = len.back();
        const size_t npairs = c.size() / 2;
        std::vector<Len> nx(npairs + (c.size() & 1));
        for (size_t i = 0; i < npairs; i++) {
            const Len &l = c[2 * i], &r = c[2 * i + 1];
            if (r.pn > l.pn + r.qn) return 1;
            nx[i] = {l.pn + r.qn + 1, l.qn + r.qn};
        }
        if (c.size() & 1) nx.back() = c.back();
        len.push_back(std::move(nx));
    }
    const int nlev = (int)len.size() - 1;                        /* levels of products */
    /* resources for every level, sized before the first launch: pools by level parity, planes, descriptors; each
     * product's length class kept for its level's grouping (-1: an empty operand) */
    size_t cap = g.cfg.workspace_bytes, pool_max[2] = {1, 1}, desc_total = 0, img_total = 0, ngroups = 0;
    struct Need { int np; uint64_t n, cnt; };
    std::vector<Need> need;                                      /* the groups with planes */
    std::vector<int> lev_np(nlev + 1, 3);
    std::vector<std::vector<int8_t>> keys(nlev + 1);
    std::vector<std::array<uint64_t, TREE_NKEY>> lev_cnt(nlev + 1);
    LenClass lclass;
    for (int k = 1; k <= nlev; k++) {
        size_t tot = 0;
        for (const Len &x : len[k]) tot += x.pn + x.qn;
        pool_max[k & 1] = std::max(pool_max[k & 1], tot);
        const std::vector<Len> &c = len[k - 1];
        const size_t npairs = c.size() / 2;
        size_t mn_max = 1;
        uint64_t *cnt = lev_cnt[k].data(), blk[TREE_NKEY];     /* per class: products, CRT blocks */
        for (int j = 0; j < TREE_NKEY; j++) cnt[j] = blk[j] = 0;
        std::vector<int8_t> &kk = keys[k];
        kk.resize(2 * npairs);
        for (size_t i = 0; i < npairs; i++) {
            const Len &l = c[2 * i], &r = c[2 * i + 1];
            const size_t pr[2][2] = {{l.pn, r.qn}, {l.qn, r.qn}};
            for (int t = 0; t < 2; t++) {
                const size_t na = pr[t][0], nb = pr[t][1];
                if (!na || !nb) { kk[2 * i + t] = -1; continue; }
                mn_max = std::max(mn_max, std::min(na, nb));
                const int key = lclass(na + nb - 1);
                const int logn = key % (NTTM_LOGN_MAX + 1), r3 = key > NTTM_LOGN_MAX;
                const uint64_t npts = (uint64_t)(r3 ? 3 : 1) << logn;
                kk[2 * i + t] = (int8_t)key;
                cnt[key]++;
                blk[key] += prod_crt_blocks(logn, r3, npts, na + nb + (t == 0 ? 1 : 0));
            }
        }
        RCK(choose_np(mn_max, &lev_np[k]));
        for (int key = 0; key < TREE_NKEY; key++) {
            if (!cnt[key]) continue;
            const int logn = key % (NTTM_LOGN_MAX + 1), r3 = key > NTTM_LOGN_MAX;
            const uint64_t npts = (uint64_t)(r3 ? 3 : 1) << logn, cnt_all = cnt[key];
            if (logn > NTTM_LOGN_MAX) return 1;
            for (uint64_t c0 = 0; c0 < cnt_all; c0 += TREE_CHUNK) {   /* the group's chunks (below) */
                const uint64_t cn = std::min<uint64_t>(TREE_CHUNK, cnt_all - c0), tb = r3 ? 3 * cn : cn;
                if (!small_len(logn, r3)) need.push_back({lev_np[k], npts, cn});
                const size_t img = align_up(cn * sizeof(CrtDesc), 256) + 2 * align_up(cn * sizeof(LoadDesc), 256) +
                                   align_up(tb * 4, 256) + 256 + 256;
                img_total += img;
                desc_total += img + align_up(cn * 8, 256) + align_up(nttm_crt_scratch_words(blk[key]) * 4, 256) + 256;
                ngroups++;
            }
        }
    }
    /* the root's P and Q go straight to p and q when their planned lengths fit there and no operand of the last level
     * lies in them (its operands are pool slots above the leaves) */
    const Len &rl = len[nlev][0];
    bool root_direct = rl.pn <= p_cap && rl.qn <= q_cap;
    if (root_direct && nlev == 1) {
        for (size_t i = 0; i < 2 && root_direct; i++) {
            const nttm_bs_node &L = leaves[i];
            const uint64_t *arr[2] = {L.p, L.q};
            const size_t nn[2] = {L.pn, L.qn};
            for (int t = 0; t < 2; t++)
                for (int o = 0; o < 2; o++) {
                    const uint64_t *d = o ? q : p;
                    const size_t dn = o ? rl.qn : rl.pn;
                    if (nn[t] && dn && arr[t] < d + dn && d < arr[t] + nn[t]) root_direct = false;
                }
        }
    }
    /* grown without waiting for the work queued before the tree (the caller's leaves): the outgrown buffers are freed
     * after the tree's final synchronization (a failed call's, at the next call's start) */
    if (g.ndfree || g.nhfree) { HIPCK(hipDeviceSynchronize()); free_deferred(); }
    RCK(bsp_need(0, pool_max[0], true)); RCK(bsp_need(1, pool_max[1], true));
    RCK(ws_need_least(&cap, [&](size_t c) {
        size_t most = 256;
        for (const Need &x : need) most = std::max(most, group_shape(x.np, x.n, x.cnt, c).bytes(x.np, x.n));
        return most;
    }, true));
    RCK(tdesc_need(desc_total + 512, true));
    RCK(tpin_need(img_total + 8 * ngroups + 2048, true));
    RCK(side_stream());
    HIPCK(hipStreamSynchronize(g.tcs));                           /* (a failed call's copies) before the image is reused */
    /* the levels */
    std::vector<nttm_bs_node> cur(leaves, leaves + n), nxt;
    std::vector<nttm_prod> prods;
    std::vector<const char *> flag_at;                          /* each group's CRT flag word in device memory */
    size_t dpos = 0, ipos = 0, ncopy = 0;
    for (int k = 1; k <= nlev; k++) {
        const size_t npairs = cur.size() / 2, odd = cur.size() & 1;
        const bool top = k == nlev && root_direct;
        uint64_t *pool = g.bsp[k & 1];
        nxt.assign(npairs + odd, nttm_bs_node());
        prods.resize(2 * npairs);
        size_t off = 0;
        for (size_t i = 0; i < npairs; i++) {                    /* P = P_L Q_R + P_R, Q = Q_L Q_R: Q_R shared */
            const nttm_bs_node &L = cur[2 * i], &R = cur[2 * i + 1];
            uint64_t *pc = top ? p : pool + off; off += L.pn + R.qn + 1;
            uint64_t *qc = top ? q : pool + off; off += L.qn + R.qn;
            nttm_prod &a = prods[2 * i], &b = prods[2 * i + 1];
            a.a = L.p; a.na = L.pn; a.b = R.q; a.nb = R.qn; a.c = pc; a.x = R.pn ? R.p : pc; a.nx = R.pn; a.ncn = 0;
            b.a = L.q; b.na = L.qn; b.b = R.q; b.nb = R.qn; b.c = qc; b.x = nullptr; b.nx = 0; b.ncn = 0;
            nxt[i].p = pc; nxt[i].pn = L.pn + R.qn + 1; nxt[i].q = qc; nxt[i].qn = L.qn + R.qn;
        }
        if (odd) {                                               /* the last node moves up (into this level's pool) */
            const nttm_bs_node &L = cur.back();
            uint64_t *pc = pool + off; off += L.pn;
            uint64_t *qc = pool + off; off += L.qn;
            if (L.pn) HIPCK(hipMemcpyAsync(pc, L.p, L.pn * 8, hipMemcpyDeviceToDevice, s));
            if (L.qn) HIPCK(hipMemcpyAsync(qc, L.q, L.qn * 8, hipMemcpyDeviceToDevice, s));
            nxt[npairs] = L; nxt[npairs].p = pc; nxt[npairs].q = qc;
        }
        /* zero-operand products (c = x, zero-extended); the others by length class */
        const std::vector<int8_t> &kk = keys[k];
        std::vector<std::vector<size_t>> groups(TREE_NKEY);
        for (int key = 0; key < TREE_NKEY; key++) groups[key].reserve(lev_cnt[k][key]);
        for (size_t i = 0; i < prods.size(); i++) {
            if (kk[i] >= 0) { groups[kk[i]].push_back(i); continue; }
            const nttm_prod &pq = prods[i];
            const size_t nc = pq.na + pq.nb + (pq.x ? 1 : 0);
            if (nc) HIPCK(hipMemsetAsync(pq.c, 0, nc * 8, s));
            if (pq.x && pq.nx) HIPCK(hipMemcpyAsync(pq.c, pq.x, pq.nx * 8, hipMemcpyDeviceToDevice, s));
        }
        for (int gi = 0; gi < TREE_NKEY; gi++) {
            const std::vector<size_t> &Gall = groups[gi];
            for (size_t c0 = 0; c0 < Gall.size(); c0 += TREE_CHUNK) {
                const std::vector<size_t> G(Gall.begin() + c0, Gall.begin() + std::min(Gall.size(), c0 + TREE_CHUNK));
                const int r3 = gi > NTTM_LOGN_MAX, logn = gi % (NTTM_LOGN_MAX + 1);
                GroupBuild gb;
                group_build(gb, prods.data(), G, lev_np[k], r3, logn, g.cfg.tile_log, batch_pts(logn), cap);
                if (dpos + gb.desc_bytes > g.tdesc_bytes || ipos + gb.off_ncn > img_total || gb.planes_bytes > g.ws_bytes)
                    return nttm_fail(NTTM_EINVAL, "internal: tree plan exceeds its sizing (level %d)", k);
                char *img = g.tpin + ipos, *dbase = g.tdesc + dpos;
                group_image(gb, (double *)g.ws, img);
                /* the descriptors copied on the side stream, which runs ahead of the launches (their region of the
                 * image and of tdesc is this group's alone): the caller's stream waits on the copy, not behind it */
                hipEvent_t ev = g.tev[ncopy++ % 8];
                HIPCK(hipMemcpyAsync(dbase, img, gb.off_ncn, hipMemcpyHostToDevice, g.tcs));
                HIPCK(hipEventRecord(ev, g.tcs));
                HIPCK(hipStreamWaitEvent(s, ev, 0));
                RCK(group_launch(gb, lev_np[k], (double *)g.ws, dbase, s, nullptr, (uint32_t *)(dbase + (gb.small ? gb.off_ctl : gb.off_crt))));
                flag_at.push_back(dbase + (gb.small ? gb.off_ctl : gb.off_crt) + 4);
                ipos = align_up(ipos + gb.off_ncn, 256);
                dpos = align_up(dpos + gb.desc_bytes, 256);
            }
        }
        cur.swap(nxt);
    }
    /* every group's flags and the root's normalized lengths (its leading zero limbs found on the device), then one
     * synchronization */
    const nttm_bs_node root = cur[0];
    char *hf = g.tpin + align_up(ipos, 256);
    uint64_t *hlen = (uint64_t *)(hf + align_up(flag_at.size() * 4, 64));
    if ((size_t)((char *)(hlen + 2) - g.tpin) > g.tpin_bytes || dpos + 16 > g.tdesc_bytes)
        return nttm_fail(NTTM_EINVAL, "internal: tree flags exceed their staging");
    uint64_t *dlen = (uint64_t *)(g.tdesc + dpos);
    RCK(nttm_run_top_nonzero(root.p, root.pn, dlen, s));
    RCK(nttm_run_top_nonzero(root.q, root.qn, dlen + 1, s));
    HIPCK(hipMemcpyAsync(hlen, dlen, 16, hipMemcpyDeviceToHost, s));
    for (size_t j = 0; j < flag_at.size(); j++) HIPCK(hipMemcpyAsync(hf + 4 * j, flag_at[j], 4, hipMemcpyDeviceToHost, s));
    HIPCK(hipStreamSynchronize(s));
    free_deferred();
    for (size_t j = 0; j < flag_at.size(); j++)
        if (((const uint32_t *)hf)[j] & 1) return nttm_fail(NTTM_ECHECK, "crt: non-zero carry beyond a top limb (wrong residues)");
    const size_t rp = hlen[0], rq = hlen[1];
    if (rp > p_cap || rq > q_cap)
        return nttm_fail(NTTM_EINVAL, "nttm_bs_tree: the root needs %zu and %zu limbs (capacities %zu, %zu)", rp, rq,
                         p_cap, q_cap);
    if (!root_direct) {
        if (rp) HIPCK(hipMemcpyAsync(p, root.p, rp * 8, hipMemcpyDeviceToDevice, s));
        if (rq) HIPCK(hipMemcpyAsync(q, root.q, rq * 8, hipMemcpyDeviceToDevice, s));
        HIPCK(hipStreamSynchronize(s));
    }
    *pn = rp; *qn = rq;
    return 0;
}
extern "C" int nttm_bs_tree(const nttm_bs_node *leaves, size_t n, uint64_t *p, size_t p_cap, size_t *pn, uint64_t *q,
                            size_t q_cap, size_t *qn, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (!leaves || !n || !pn || !qn || (p_cap && !p) || (q_cap && !q)) return nttm_fail(NTTM_EINVAL, "nttm_bs_tree arguments");
    hipStream_t s = (hipStream_t)stream;
    MemMap mm;
    for (size_t i = 0; i < n; i++) {
        if ((leaves[i].pn && !leaves[i].p) || (leaves[i].qn && !leaves[i].q)) return nttm_fail(NTTM_EINVAL, "leaf %zu: null limbs", i);
        if (mm.kind(leaves[i].p, leaves[i].pn * 8) != MEM_DEV || mm.kind(leaves[i].q, leaves[i].qn * 8) != MEM_DEV)
            return nttm_fail(NTTM_EINVAL, "nttm_bs_tree: leaf %zu is not device memory of this device", i);
    }
    if (mm.kind(p, p_cap * 8) != MEM_DEV || mm.kind(q, q_cap * 8) != MEM_DEV)
        return nttm_fail(NTTM_EINVAL, "nttm_bs_tree: p or q is not device memory of this device");
    if (!g_tree_levelwise) {
        const int rc = bs_tree_planned(leaves, n, p, p_cap, pn, q, q_cap, qn, s);
        if (rc <= 0) return rc;
    }
    std::vector<nttm_bs_node> cur(leaves, leaves + n), nxt;
    std::vector<nttm_prod> prods;
    for (int level = 0; cur.size() > 1; level++) {
        const size_t npairs = cur.size() / 2, odd = cur.size() & 1;
        size_t total = 0;                                        /* the parents' limbs (the odd node copied) */
        for (size_t i = 0; i < npairs; i++) total += cur[2 * i].pn + cur[2 * i + 1].qn + 1 + cur[2 * i].qn + cur[2 * i + 1].qn;
        if (odd) total += cur.back().pn + cur.back().qn;
        RCK(bsp_need(level & 1, total ? total : 1));
        uint64_t *pool = g.bsp[level & 1];
        nxt.assign(npairs + odd, nttm_bs_node());
        prods.assign(2 * npairs, nttm_prod());
        size_t off = 0;
        for (size_t i = 0; i < npairs; i++) {                    /* P = P_L Q_R + P_R, Q = Q_L Q_R: Q_R shared */
            const nttm_bs_node &L = cur[2 * i], &R = cur[2 * i + 1];
            if (R.pn > L.pn + R.qn)
                return nttm_fail(NTTM_EINVAL, "nttm_bs_tree: level %d pair %zu: |P_R| = %zu exceeds |P_L| + |Q_R| = %zu",
                                 level, i, R.pn, L.pn + R.qn);
            uint64_t *pc = pool + off; off += L.pn + R.qn + 1;
            uint64_t *qc = pool + off; off += L.qn + R.qn;
            nttm_prod &a = prods[2 * i], &b = prods[2 * i + 1];
            a.a = L.p; a.na = L.pn; a.b = R.q; a.nb = R.qn; a.c = pc; a.x = R.pn ? R.p : nullptr; a.nx = R.pn;
            b.a = L.q; b.na = L.qn; b.b = R.q; b.nb = R.qn; b.c = qc; b.x = nullptr; b.nx = 0;
            if (!a.x) { a.x = pc; a.nx = 0; }                     /* P_R = 0: an empty x keeps the carry limb */
            nxt[i].p = pc; nxt[i].q = qc;
        }
        if (odd) {                                               /* the last node moves up (into this level's pool) */
            const nttm_bs_node &L = cur.back();
            uint64_t *pc = pool + off; off += L.pn;
            uint64_t *qc = pool + off; off += L.qn;
            if (L.pn) HIPCK(hipMemcpyAsync(pc, L.p, L.pn * 8, hipMemcpyDeviceToDevice, s));
            if (L.qn) HIPCK(hipMemcpyAsync(qc, L.q, L.qn * 8, hipMemcpyDeviceToDevice, s));
            nxt[npairs].p = pc; nxt[npairs].pn = L.pn; nxt[npairs].q = qc; nxt[npairs].qn = L.qn;
        }
        RCK(nttm_mul_batch(prods.data(), prods.size(), stream));
        for (size_t i = 0; i < npairs; i++) { nxt[i].pn = prods[2 * i].ncn; nxt[i].qn = prods[2 * i + 1].ncn; }
        cur.swap(nxt);
    }
    const nttm_bs_node &root = cur[0];
    if (root.pn > p_cap || root.qn > q_cap)
        return nttm_fail(NTTM_EINVAL, "nttm_bs_tree: the root needs %zu and %zu limbs (capacities %zu, %zu)", root.pn,
                         root.qn, p_cap, q_cap);
    if (root.pn) HIPCK(hipMemcpyAsync(p, root.p, root.pn * 8, hipMemcpyDeviceToDevice, s));
    if (root.qn) HIPCK(hipMemcpyAsync(q, root.q, root.qn * 8, hipMemcpyDeviceToDevice, s));
    HIPCK(hipStreamSynchronize(s));
    *pn = root.pn; *qn = root.qn;
    return 0;
}

/* ---- transform primitives on canonical uint64 residues ---------------------------------------------------------------- */
/* the arguments of a transform primitive: x holds batch transforms of (3 if r3) 2^logn residues in device memory */
static int prim_check(int prime, const void *x, int logn, size_t batch, int r3 = 0)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (prime < 0 || prime >= NTTM_MAX_PRIMES) return nttm_fail(NTTM_EINVAL, "prime %d", prime);
    if (logn < 1 || logn > NTTM_LOGN_MAX) return nttm_fail(NTTM_EINVAL, "logn %d outside [1, %d]", logn, NTTM_LOGN_MAX);
    if (!x || !batch) return nttm_fail(NTTM_EINVAL, "empty transform");
    DEVCK(x, ((uint64_t)batch << logn) * (r3 ? 3 : 1) * 8, "x");
    return 0;
}
/* the residues are converted in a transform's first and last pass: passes of their own (16 B a point each) took 40% of a
 * product formed from the primitives at 2^22 points */
extern "C" int nttm_ntt_fwd(int prime, uint64_t *x, int logn, size_t batch, void *stream)
{
    RCK(prim_check(prime, x, logn, batch));
    return fwd_planes(prime, (double *)x, logn, batch, (hipStream_t)stream, 1, 1);
}
extern "C" int nttm_ntt_inv(int prime, uint64_t *x, int logn, size_t batch, void *stream)
{
    RCK(prim_check(prime, x, logn, batch));
    return inv_planes(prime, (double *)x, nullptr, NTTM_Y_FULL, logn, batch, 1, (hipStream_t)stream, 0, 1, 0, 1);
}
/* y as the fused inverse reads it: in place (canonical residues), or, where it shares memory with x other than element for
 * element, an FP64 copy made first (the inverse's first pass overwrites x tile by tile) */
static int pw_operand(const uint64_t *x, uint64_t cnt, const uint64_t *y, uint64_t ycnt, int ymode, hipStream_t s,
                      const double **yp, int *y_u64)
{
    *yp = (const double *)y; *y_u64 = 1;
    if (!(x < y + ycnt && y < x + cnt) || (ymode == NTTM_Y_FULL && x == y)) return 0;
    RCK(ws_need(ycnt * 8));
    RCK(nttm_run_cvt_u64_f64((double *)g.ws, y, ycnt, s));
    *yp = (const double *)g.ws; *y_u64 = 0;
    return 0;
}
extern "C" int nttm_ntt_inv_pw(int prime, uint64_t *x, const uint64_t *y, int ymode, int logn, size_t batch, void *stream)
{
    RCK(prim_check(prime, x, logn, batch));
    if (!y) return nttm_fail(NTTM_EINVAL, "null y");
    if (ymode < NTTM_Y_FULL || ymode > NTTM_Y_PAIR) return nttm_fail(NTTM_EINVAL, "ymode %d", ymode);
    hipStream_t s = (hipStream_t)stream;
    const uint64_t cnt = (uint64_t)batch << logn;
    const uint64_t ycnt = ymode == NTTM_Y_FULL ? cnt : ymode == NTTM_Y_BCAST ? ((uint64_t)1 << logn)
                                                     : ((uint64_t)((batch + 1) / 2) << logn);
    DEVCK(y, ycnt * 8, "y");
    const double *yp; int y_u64;
    RCK(pw_operand(x, cnt, y, ycnt, ymode, s, &yp, &y_u64));
    return inv_planes(prime, (double *)x, yp, ymode, logn, batch, 1, s, 0, 1, y_u64, 1);
}

/* the forward transform with its first four levels as one radix-16 stage on INT8 matrix cores (mfma.hip), the
 * remaining levels on the FP64 engine as 16 transforms of n/16 points each: the same canonical output as nttm_ntt_fwd */
extern "C" int nttm_ntt_fwd_mfma(int prime, uint64_t *x, int logn, size_t batch, void *stream)
{
    RCK(prim_check(prime, x, logn, batch));
    if (logn < 8) return nttm_fail(NTTM_EINVAL, "nttm_ntt_fwd_mfma: 2^%d points (at least 2^8)", logn);
    hipStream_t s = (hipStream_t)stream;
    const uint64_t p = NTTM_PRIMES[prime], n = (uint64_t)1 << logn, cnt = (uint64_t)batch << logn;
    const uint64_t w = nttm_root(prime, logn), W = nttm_root(prime, 4);
    /* host tables: the 15 x 2 A operands (30720 bytes), w^i and w^(4096 i), the recombination constants */
    const uint64_t nhi = ((n >> 4) + 4095) / 4096;
    std::vector<uint8_t> et(15 * 2 * 64 * 16, 0);
    uint64_t Wp[16];
    for (int i = 0; i < 16; i++) Wp[i] = h_powmod(W, i, p);
    for (int sh = 0; sh < 15; sh++)
        for (int h = 0; h < 2; h++)
            for (int l = 0; l < 64; l++)
                for (int by = 0; by < 16; by++) {
                    const int k = l & 15, t = 2 * (l >> 4) + by / 8 + 8 * h, b = by % 8, c = sh - b;
                    if (c < 0 || c > 7) continue;
                    et[((sh * 2 + h) * 64 + l) * 16 + by] = (uint8_t)((Wp[(t * k) & 15] >> (7 * c)) & 127);
                }
    std::vector<double> tw(4096 + nhi + 4);
    const uint64_t w4096 = h_powmod(w, 4096, p);
    for (uint64_t i = 0, v = 1; i < 4096; i++, v = h_mulmod(v, w, p)) tw[i] = h_bal(v, p);
    for (uint64_t i = 0, v = 1; i < nhi; i++, v = h_mulmod(v, w4096, p)) tw[4096 + i] = h_bal(v, p);
    const double2 c35 = h_shoup(h_powmod(2, 35, p), p), c70 = h_shoup(h_powmod(2, 70, p), p);
    double *cs = tw.data() + 4096 + nhi;
    cs[0] = c35.x; cs[1] = c35.y; cs[2] = c70.x; cs[3] = c70.y;
    const size_t off_e = align_up(cnt * 8, 256), off_t = align_up(off_e + et.size(), 256);
    RCK(ws_need(off_t + tw.size() * 8 + 256));
    HIPCK(hipMemcpyAsync(g.ws + off_e, et.data(), et.size(), hipMemcpyHostToDevice, s));
    HIPCK(hipMemcpyAsync(g.ws + off_t, tw.data(), tw.size() * 8, hipMemcpyHostToDevice, s));
    double *y = (double *)g.ws;
    const double *dt = (const double *)(g.ws + off_t);
    RCK(nttm_run_dft16_mfma(x, y, logn, batch, g.ws + off_e, dt, dt + 4096, cs, (double)p, s));   /* cs: host copy */
    RCK(fwd_planes(prime, y, logn - 4, 16 * (uint64_t)batch, s));
    HIPCK(hipMemcpyAsync(x, y, cnt * 8, hipMemcpyDeviceToDevice, s));
    RCK(nttm_run_f64_to_canon((double *)x, cnt, g.pk[prime], s));
    return nttm_hip_check(hipStreamSynchronize(s), "nttm_ntt_fwd_mfma");                 /* the host tables */
}

/* transforms of 3 2^logk points: the radix-3 layer (nttm_run_r3) and the 2^logk engine on the thirds (batch 3) */
extern "C" int nttm_ntt_fwd3(int prime, uint64_t *x, int logk, size_t batch, void *stream)
{
    RCK(prim_check(prime, x, logk, batch, 1));
    hipStream_t s = (hipStream_t)stream;
    JobSet r; memset(&r, 0, sizeof r);
    r.n = 1; r.j[0] = prime_job(prime, (double *)x, batch, false);
    RCK(nttm_run_r3(false, logk, r, s, nullptr, true));
    return fwd_planes(prime, (double *)x, logk, 3 * (uint64_t)batch, s, 0, 1);
}
/* the inverse: the engine's inverses scale by 2^-logk, the radix-3 layer by 3^-1 */
static int inv3_planes(int prime, double *x, const double *y, int y_u64, int ymode, int logk, uint64_t batch, hipStream_t s)
{
    const uint64_t p = NTTM_PRIMES[prime];
    RCK(inv_planes(prime, x, y, ymode, logk, 3 * batch, 1, s, 1, 1, y_u64, 0));
    JobSet r; memset(&r, 0, sizeof r);
    r.n = 1; r.j[0] = prime_job(prime, x, batch, true);
    r.j[0].in_scale = h_shoup(h_inv(3, p), p); r.j[0].do_in_scale = 1;
    return nttm_run_r3(true, logk, r, s, nullptr, true);
}
extern "C" int nttm_ntt_inv3(int prime, uint64_t *x, int logk, size_t batch, void *stream)
{
    RCK(prim_check(prime, x, logk, batch, 1));
    return inv3_planes(prime, (double *)x, nullptr, 0, NTTM_Y_FULL, logk, batch, (hipStream_t)stream);
}
extern "C" int nttm_ntt_inv3_pw(int prime, uint64_t *x, const uint64_t *y, int ymode, int logk, size_t batch, void *stream)
{
    RCK(prim_check(prime, x, logk, batch, 1));
    if (!y) return nttm_fail(NTTM_EINVAL, "null y");
    if (ymode < NTTM_Y_FULL || ymode > NTTM_Y_PAIR) return nttm_fail(NTTM_EINVAL, "ymode %d", ymode);
    hipStream_t s = (hipStream_t)stream;
    const uint64_t n3 = (uint64_t)3 << logk, cnt = n3 * batch;
    const uint64_t ycnt = ymode == NTTM_Y_FULL ? cnt : ymode == NTTM_Y_BCAST ? n3 : (uint64_t)((batch + 1) / 2) * n3;
    DEVCK(y, ycnt * 8, "y");
    const double *yp; int y_u64;
    RCK(pw_operand(x, cnt, y, ycnt, ymode, s, &yp, &y_u64));
    return inv3_planes(prime, (double *)x, yp, y_u64, ymode, logk, batch, s);
}
extern "C" int nttm_pw(int prime, uint64_t *x, const uint64_t *y, size_t count, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (prime < 0 || prime >= NTTM_MAX_PRIMES || !x || !y) return nttm_fail(NTTM_EINVAL, "nttm_pw arguments");
    if (!count) return 0;
    DEVCK(x, count * 8, "x");
    DEVCK(y, count * 8, "y");
    return nttm_run_pw_u64(x, y, count, g.pk[prime], (hipStream_t)stream);
}
extern "C" int nttm_load(int prime, uint64_t *dst, const uint64_t *src, size_t nlimbs, size_t npoints, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (prime < 0 || prime >= NTTM_MAX_PRIMES || !dst || (nlimbs && !src) || nlimbs > npoints)
        return nttm_fail(NTTM_EINVAL, "nttm_load arguments");
    if (!npoints) return 0;
    DEVCK(dst, npoints * 8, "dst");
    DEVCK(src, nlimbs * 8, "src");
    return nttm_run_load_planes((double *)dst, npoints, src, nlimbs, npoints, 1, &g.pk[prime], nullptr, 1, (hipStream_t)stream);
}
extern "C" int nttm_crt(uint64_t *c, size_t nc, const uint64_t *const *planes, int np, size_t ncoef, const uint64_t *x,
                        size_t nx, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (np < 3 || np > NTTM_MAX_PRIMES || !planes || (nc && !c) || (nx && !x)) return nttm_fail(NTTM_EINVAL, "nttm_crt arguments");
    if (ncoef > nc) return nttm_fail(NTTM_EINVAL, "nttm_crt: ncoef %zu exceeds nc %zu", ncoef, nc);
    if (!nc) return 0;
    DEVCK(c, nc * 8, "c");
    DEVCK(x, nx * 8, "x");
    for (int i = 0; i < np; i++) DEVCK(planes[i], ncoef * 8, "plane");
    hipStream_t s = (hipStream_t)stream;
    for (int i = 0; i < np; i++) if (!planes[i] && ncoef) return nttm_fail(NTTM_EINVAL, "null plane %d", i);
    /* the planes are read in place as canonical residues, unless c shares memory with one of them (the CRT's blocks write
     * c while others still read): then through FP64 copies */
    bool copy = false;
    for (int i = 0; i < np; i++) copy = copy || (ncoef && c < planes[i] + ncoef && planes[i] < c + nc);
    const size_t pbytes = copy ? align_up((size_t)np * ncoef * 8, 256) : 0;
    const size_t crt_words = nttm_crt_scratch_words(nttm_crt_blocks(nc));
    RCK(ws_need(pbytes + 256 + crt_words * 4 + 256));
    if (shares(c, nc, x, nx)) {                                  /* (x_apart) */
        RCK(xc_need(nx));
        nttm_prod q; memset(&q, 0, sizeof q);
        q.na = nc; q.c = c; q.x = x; q.nx = nx;
        RCK(copy_x(&q, 1, true, g.xc, s));
        x = q.x;
    }
    CrtDesc hd; memset(&hd, 0, sizeof hd);
    hd.ncoef = ncoef; hd.x = x; hd.nx = x ? nx : 0; hd.c = c; hd.nc = nc; hd.first_block = 0;
    if (copy) {
        double *pl = (double *)g.ws;
        hd.pl = pl; hd.plane = ncoef;
        for (int i = 0; i < np; i++) RCK(nttm_run_cvt_u64_f64(pl + (size_t)i * ncoef, planes[i], ncoef, s));
    }
    uint32_t *ctl = (uint32_t *)((char *)g.hpin + 96);
    RCK(nttm_crt_launch_one(hd, nttm_crt_blocks(nc), np, g.cc, (uint32_t *)(g.ws + pbytes + 256), ctl, s,
                            8.0 * np * (double)ncoef + 8.0 * (double)nc + 8.0 * (double)(x ? nx : 0), nullptr,
                            copy ? nullptr : planes));
    HIPCK(hipStreamSynchronize(s));
    const uint32_t flags = ctl[1];
    if (flags & 1) return nttm_fail(NTTM_ECHECK, "crt: the value needs more than nc limbs");
    return 0;
}

/* ---- live kernel timing ------------------------------------------------------------------------------------------------ */
struct ProfRec { const char *name; double bytes; hipEvent_t a, b; };
static std::vector<ProfRec> g_prof;
static std::vector<hipEvent_t> g_evpool;
static hipEvent_t ev_get(void)
{
    if (!g_evpool.empty()) { hipEvent_t e = g_evpool.back(); g_evpool.pop_back(); return e; }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
    return e;
}
void prof_begin(const char *name, double alg_bytes, hipStream_t s)
{
    if (!g_prof_on) return;
    ProfRec r; r.name = name; r.bytes = alg_bytes; r.a = ev_get(); r.b = ev_get();
    if (!r.a || !r.b) return;
    (void)hipEventRecord(r.a, s);
    g_prof.push_back(r);
}
void prof_end(hipStream_t s)
{
    if (!g_prof_on || g_prof.empty()) return;
    (void)hipEventRecord(g_prof.back().b, s);
}
static void prof_clear(void)
{
    for (auto &r : g_prof) { g_evpool.push_back(r.a); g_evpool.push_back(r.b); }
    g_prof.clear();
}
static void prof_release(void)
{
    prof_clear();
    for (hipEvent_t e : g_evpool) (void)hipEventDestroy(e);
    g_evpool.clear();
    g_prof_on = 0;
}
extern "C" int nttm_profile(int enable)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    HIPCK(hipDeviceSynchronize());
    prof_clear();
    g_prof_on = enable != 0;
    return 0;
}
extern "C" int nttm_profile_read(nttm_kstat *out, int cap)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    HIPCK(hipDeviceSynchronize());
    int n = 0;
    for (auto &r : g_prof) {
        float ms = 0;
        if (hipEventElapsedTime(&ms, r.a, r.b) != hipSuccess) { (void)hipGetLastError(); continue; }
        int k = 0;
        while (k < n && strcmp(out[k].name, r.name)) k++;
        if (k == n) {
            if (n >= cap) continue;
            memset(&out[n], 0, sizeof out[n]);
            snprintf(out[n].name, sizeof out[n].name, "%s", r.name);
            n++;
        }
        out[k].launches++; out[k].total_ms += ms; out[k].alg_bytes += r.bytes;
    }
    return n;
}

/* ---- batch plans: a batch's whole schedule as one hipGraph, each group's schedule chosen by measurement -------------
 * The binary-splitting leaves of the reference go through rns_mul_batch again and again with the same shapes
 * (E/rns_mul.c:792-1028).  A plan fixes one batch: it groups the products, chooses per length class whether the
 * products that fit 3 2^k points take that length or 2^(k+2), and per group the strided-pass tile (2^12 or 2^13
 * points) and the points per thread (8 or 16) by timing every candidate on the batch's own operands; uploads every
 * descriptor once; and captures all groups' launches (transforms, CRT, carry scan, lengths) as one graph that a run
 * launches with one call. */
struct nttm_batch_plan {
    size_t N = 0;
    uint64_t gen = 0;                                            /* the nttm_init it was made under */
    int np = 3;
    std::vector<GroupBuild> gb;
    std::vector<std::vector<size_t>> gidx;
    std::vector<double> gms;                                     /* each group's measured time (ms; 0 untuned) */
    std::vector<size_t> goff;                                    /* descriptor bases in blob */
    std::vector<size_t> zidx;                                    /* products with an empty operand */
    size_t off_z = 0;
    char *blob = nullptr;
    size_t blob_bytes = 0;
    uint64_t *xc = nullptr;                                      /* the copies of x operands under their results */
    uint64_t *hstage = nullptr;                                  /* pinned: the lengths and flags, written by the runs */
    size_t hstage_words = 0;
    hipStream_t cs = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    double tune_ms = 0;
    int candidates = 0;
    int reused = 0;                                              /* groups that took a remembered choice */
};

static void plan_free(nttm_batch_plan *pl)
{
    if (!pl) return;
    if (pl->exec) (void)hipGraphExecDestroy(pl->exec);
    if (pl->graph) (void)hipGraphDestroy(pl->graph);
    if (pl->cs) (void)hipStreamDestroy(pl->cs);
    if (pl->blob) (void)hipFree(pl->blob);
    if (pl->xc) (void)hipFree(pl->xc);
    if (pl->hstage) (void)hipHostFree(pl->hstage);
    delete pl;
}

/* a device buffer that grows (the autotuner's trial runs) */
struct TuneBuf {
    char *p = nullptr; size_t bytes = 0;
    ~TuneBuf() { release(); }
    void release() { if (p) { (void)hipDeviceSynchronize(); (void)hipFree(p); } p = nullptr; bytes = 0; }
    int need(size_t b)
    {
        if (b <= bytes) return 0;
        if (p) { (void)hipDeviceSynchronize(); (void)hipFree(p); p = nullptr; bytes = 0; }
        if (hipMalloc(&p, b) != hipSuccess) { (void)hipGetLastError(); return nttm_fail(NTTM_ENOMEM, "plan: %zu bytes", b); }
        bytes = b;
        return 0;
    }
};
/* the autotuner's choices, kept across plans: per prime count, transform length (2^logn, or 3 2^logn with r3) and group
 * size (its products), the (tile, points per thread) that won and its time per product.  Each entry belongs to the
 * nttm_init it was timed under.  Plans created with autotune == 2 take the entry of the same size, else the nearest
 * size of the same power-of-two class, instead of timing the candidates again */
struct TuneMemo { uint64_t gen; int np, r3, logn; uint64_t cnt; int tile, pts; double ms_per; };
#define TUNE_MEMO_MAX 4096
static TuneMemo g_memo[TUNE_MEMO_MAX];
static int g_nmemo = 0;
static const TuneMemo *memo_find(int np, int r3, int logn, uint64_t cnt)
{
    const TuneMemo *best = nullptr;
    uint64_t dbest = 0;
    for (int i = 0; i < g_nmemo; i++) {
        const TuneMemo &m = g_memo[i];
        if (m.gen != g.gen || m.np != np || m.r3 != r3 || m.logn != logn || ceil_log2(m.cnt) != ceil_log2(cnt)) continue;
        const uint64_t d = m.cnt > cnt ? m.cnt - cnt : cnt - m.cnt;
        if (!best || d < dbest) { best = &m; dbest = d; }
    }
    return best;
}
static void memo_put(const TuneMemo &e)
{
    TuneMemo *slot = nullptr;
    for (int i = 0; i < g_nmemo && !slot; i++) {                 /* the same key, or an entry of an earlier nttm_init */
        TuneMemo &m = g_memo[i];
        if (m.gen != g.gen || (m.np == e.np && m.r3 == e.r3 && m.logn == e.logn && m.cnt == e.cnt)) slot = &m;
    }
    if (!slot && g_nmemo < TUNE_MEMO_MAX) slot = &g_memo[g_nmemo++];
    if (slot) *slot = e;                                         /* (a full table keeps its entries) */
}
/* the fastest (tile, points per thread) for one group of products, timed on the stream; *ms its time.  reuse: a
 * remembered choice for the same class is taken untimed (*ms scaled from its time per product; *nreused counts it) */
static int tune_group(const nttm_prod *P, const std::vector<size_t> &G, int np, int r3, int logn, size_t cap, bool tune, TuneBuf &tb,
                      std::vector<char> &img, hipStream_t s, GroupBuild &best, double *ms, int *ntried, bool reuse = false,
                      int *nreused = nullptr)
{
    static const int cand[4][2] = {{12, 16}, {13, 16}, {12, 8}, {13, 8}};
    *ms = 0;
    if (!tune) { group_build(best, P, G, np, r3, logn, g.cfg.tile_log, batch_pts(logn), cap); return 0; }
    if (reuse) {
        if (const TuneMemo *m = memo_find(np, r3, logn, G.size())) {
            group_build(best, P, G, np, r3, logn, m->tile, m->pts, cap);
            *ms = m->ms_per * (double)G.size();
            if (nreused) (*nreused)++;
            return 0;
        }
    }
    double best_ms = 1e30;
    hipEvent_t e0 = g.ev[0], e1 = g.ev[1];
    /* the one-kernel products know neither tile nor points per thread: all four candidates are one launch, timed once for the
     * choice of length, and the group keeps the configured values */
    const bool one = small_len(logn, r3);
    for (int c = 0; c < (one ? 1 : 4); c++) {
        GroupBuild gb;
        if (one) group_build(gb, P, G, np, r3, logn, g.cfg.tile_log, batch_pts(logn), cap);
        else group_build(gb, P, G, np, r3, logn, cand[c][0], cand[c][1], cap);
        const size_t off_d = align_up(gb.planes_bytes, 256);
        RCK(tb.need(off_d + gb.desc_bytes + 256));
        img.resize(gb.desc_bytes);
        group_image(gb, (double *)tb.p, img.data());
        HIPCK(hipMemcpyAsync(tb.p + off_d, img.data(), gb.desc_bytes, hipMemcpyHostToDevice, s));
        uint64_t *const tn = (uint64_t *)(tb.p + off_d + gb.off_ncn);
        uint32_t *const tc = (uint32_t *)(tb.p + off_d + gb.off_crt);
        RCK(group_launch(gb, np, (double *)tb.p, tb.p + off_d, s, tn, tc));       /* warm */
        double t = 1e30;
        for (int r = 0; r < 2; r++) {
            HIPCK(hipEventRecord(e0, s));
            RCK(group_launch(gb, np, (double *)tb.p, tb.p + off_d, s, tn, tc));
            HIPCK(hipEventRecord(e1, s));
            HIPCK(hipEventSynchronize(e1));
            float f = 0; HIPCK(hipEventElapsedTime(&f, e0, e1));
            t = std::min(t, (double)f);
        }
        *ntried += one ? 4 : 1;
        if (t < best_ms) { best_ms = t; best = std::move(gb); }
    }
    *ms = best_ms;
    memo_put(TuneMemo{g.gen, np, r3, logn, (uint64_t)G.size(), best.tile, best.pts, best_ms / (double)G.size()});
    return 0;
}

/* a plan whose groups' planes take at most cap bytes where they can (0: any) */
static int plan_create(const nttm_prod *P, size_t N, int autotune, size_t cap, nttm_batch_plan **out, hipStream_t s)
{
    /* the graph has the operands' addresses built in: device memory only */
    {
        MemMap mm;
        for (size_t i = 0; i < N; i++) {
            const nttm_prod &q = P[i];
            int k[4];
            RCK(prod_kinds(mm, q.a, q.na, q.b, q.nb, q.x, q.nx, q.c, q.na + q.nb + (q.x ? 1 : 0), k, i));
            if (any_host(k)) return nttm_fail(NTTM_EINVAL, "plan: product %zu: host memory (a plan takes device memory)", i);
        }
    }
    nttm_batch_plan *pl = new nttm_batch_plan();
    pl->N = N;
    pl->gen = g.gen;
    auto fail = [&](int rc) { plan_free(pl); return rc; };
    /* validate and class the products by their 2^k length */
    size_t mn_max = 0;
    std::vector<std::vector<size_t>> cls(NTTM_LOGN_MAX + 1);
    std::vector<size_t> segs;
    for (size_t i = 0; i < N; i++) {
        const nttm_prod &q = P[i];
        if (q.x && q.nx > q.na + q.nb) return fail(nttm_fail(NTTM_EINVAL, "product %zu: nx exceeds na + nb", i));
        if (!q.c || (q.na && !q.a) || (q.nb && !q.b) || (q.nx && !q.x)) return fail(nttm_fail(NTTM_EINVAL, "product %zu: null pointer", i));
        if (!q.na || !q.nb) { pl->zidx.push_back(i); continue; }
        mn_max = std::max(mn_max, (size_t)std::min(q.na, q.nb));
        int logn, r3;
        choose_len(q.na + q.nb - 1, NTTM_R3_NEVER, g.cfg.tile_log, &logn, &r3);
        if (logn > NTTM_LOGN_MAX) return fail(nttm_fail(NTTM_EBOUND, "product %zu: transform above 2^%d", i, NTTM_LOGN_MAX));
        int ln, r3b;
        choose_len(q.na + q.nb - 1, &ln, &r3b);
        if (batch_segments(q, ln, r3b)) segs.push_back(i);
        else cls[logn].push_back(i);
    }
    int rc = choose_np(mn_max ? mn_max : 1, &pl->np);
    if (rc) return fail(rc);
    const int np = pl->np;
    /* an x under its result: every run copies it first (x_apart) */
    const nttm_prod *const P0 = P;
    std::vector<nttm_prod> Q;
    if (const size_t n = x_limbs(P, N, true)) {
        if (hipMalloc(&pl->xc, n * 8) != hipSuccess) {
            (void)hipGetLastError(); pl->xc = nullptr;
            return fail(nttm_fail(NTTM_ENOMEM, "plan: copies of x: %zu limbs", n));
        }
        Q.assign(P, P + N);
        if ((rc = copy_x(Q.data(), N, true, pl->xc, s))) return fail(rc);
        P = Q.data();
    }
    /* the schedule: per class k the radix-3 subset (products of at most 3 2^(k-2) coefficients) either takes 3 2^(k-2)
     * points or stays at 2^k; per group the tile and points per thread */
    TuneBuf tb;
    std::vector<char> img;
    const bool tune = autotune != 0, reuse = autotune == 2;
    auto t_start = std::chrono::steady_clock::now();
    for (int k = 0; k <= NTTM_LOGN_MAX; k++) {
        const std::vector<size_t> &C = cls[k];
        if (C.empty()) continue;
        std::vector<size_t> S3, S2;
        for (size_t i : C) {
            int logn, r3;
            choose_len(P[i].na + P[i].nb - 1, tune ? NTTM_R3_FIT : g.cfg.radix3, g.cfg.tile_log, &logn, &r3);
            (r3 ? S3 : S2).push_back(i);
        }
        GroupBuild a, b3, b2;
        double ta = 0, t3 = 0, t2 = 0;
        if (tune && !S3.empty()) {                               /* both variants timed */
            if ((rc = tune_group(P, C, np, 0, k, cap, true, tb, img, s, a, &ta, &pl->candidates, reuse, &pl->reused))) return fail(rc);
            if ((rc = tune_group(P, S3, np, 1, k - 2, cap, true, tb, img, s, b3, &t3, &pl->candidates, reuse, &pl->reused)))
                return fail(rc);
            if (!S2.empty() && (rc = tune_group(P, S2, np, 0, k, cap, true, tb, img, s, b2, &t2, &pl->candidates, reuse, &pl->reused)))
                return fail(rc);
            if (ta <= t3 + t2) { pl->gb.push_back(std::move(a)); pl->gidx.push_back(C); pl->gms.push_back(ta); continue; }
        } else if (S3.empty()) {
            if ((rc = tune_group(P, C, np, 0, k, cap, tune, tb, img, s, a, &ta, &pl->candidates, reuse, &pl->reused))) return fail(rc);
            pl->gb.push_back(std::move(a)); pl->gidx.push_back(C); pl->gms.push_back(ta);
            continue;
        } else {                                                 /* untuned: the library's rule */
            if ((rc = tune_group(P, S3, np, 1, k - 2, cap, false, tb, img, s, b3, &t3, &pl->candidates))) return fail(rc);
            if (!S2.empty() && (rc = tune_group(P, S2, np, 0, k, cap, false, tb, img, s, b2, &t2, &pl->candidates))) return fail(rc);
        }
        pl->gb.push_back(std::move(b3)); pl->gidx.push_back(S3); pl->gms.push_back(t3);
        if (!S2.empty()) { pl->gb.push_back(std::move(b2)); pl->gidx.push_back(S2); pl->gms.push_back(t2); }
    }
    if (!segs.empty()) {
        seg_sort(segs, P);
        GroupBuild b;
        group_build(b, P, segs, np, 2, SEG_CLASS % (NTTM_LOGN_MAX + 1), g.cfg.tile_log, 16);
        pl->gb.push_back(std::move(b)); pl->gidx.push_back(segs); pl->gms.push_back(0);
    }
    pl->tune_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
    /* one device blob: the planes (the largest group's; groups run one after another), then every descriptor */
    size_t planes = 0;
    for (const GroupBuild &x : pl->gb) planes = std::max(planes, x.planes_bytes);
    size_t off = align_up(std::max(planes, (size_t)256), 256);
    for (const GroupBuild &x : pl->gb) { pl->goff.push_back(off); off = align_up(off + x.desc_bytes, 256); }
    pl->off_z = off; off = align_up(off + pl->zidx.size() * sizeof(CrtDesc), 256);
    pl->blob_bytes = off;
    tb.release();
    if (hipMalloc(&pl->blob, pl->blob_bytes) != hipSuccess) {
        (void)hipGetLastError(); pl->blob = nullptr;
        return fail(nttm_fail(NTTM_ENOMEM, "plan: %zu bytes", pl->blob_bytes));
    }
    const size_t first = pl->goff.empty() ? pl->off_z : pl->goff[0];         /* the descriptors, after the planes */
    std::vector<char> himg(pl->blob_bytes - first, 0);
    double *A = (double *)pl->blob;
    for (size_t i = 0; i < pl->gb.size(); i++) group_image(pl->gb[i], A, himg.data() + (pl->goff[i] - first));
    for (size_t z = 0; z < pl->zidx.size(); z++) {
        const nttm_prod &q = P[pl->zidx[z]];
        CrtDesc c{}; c.c = q.c; c.nc = q.na + q.nb + (q.x ? 1 : 0); c.x = q.x; c.nx = q.x ? q.nx : 0;
        memcpy(himg.data() + (pl->off_z - first) + z * sizeof(CrtDesc), &c, sizeof c);
    }
    if ((rc = nttm_hip_check(hipMemcpy(pl->blob + first, himg.data(), himg.size(), hipMemcpyHostToDevice),
                             "plan descriptors"))) return fail(rc);
    size_t words = pl->zidx.size() + 2 * pl->gb.size();           /* per group its lengths and its flags; the empty products' */
    for (const GroupBuild &x : pl->gb) words += x.cnt;
    pl->hstage_words = words + 1;
    if (hipHostMalloc((void **)&pl->hstage, pl->hstage_words * 8, 0) != hipSuccess) {
        (void)hipGetLastError(); pl->hstage = nullptr; return fail(nttm_fail(NTTM_ENOMEM, "plan: pinned staging"));
    }
    memset(pl->hstage, 0, pl->hstage_words * 8);                  /* (lengths asked for before any run: 0, and no flag) */
    /* capture every group's launches on a stream of the plan's own (default priority) */
    if ((rc = nttm_hip_check(hipStreamCreate(&pl->cs), "plan stream"))) return fail(rc);
    if ((rc = nttm_hip_check(hipStreamSynchronize(s), "plan tuning"))) return fail(rc);
    const int prof0 = g_prof_on;
    g_prof_on = 0;                                               /* no event records inside the graph */
    if ((rc = nttm_hip_check(hipStreamBeginCapture(pl->cs, hipStreamCaptureModeRelaxed), "begin capture"))) { g_prof_on = prof0; return fail(rc); }
    uint64_t *hw = pl->hstage;
    if (pl->xc) {
        Q.assign(P0, P0 + N);
        rc = copy_x(Q.data(), N, true, pl->xc, pl->cs);
    }
    for (size_t i = 0; i < pl->gb.size() && !rc; i++) {
        const uint64_t cnt = pl->gb[i].cnt;
        rc = group_launch(pl->gb[i], np, A, pl->blob + pl->goff[i], pl->cs, hw, (uint32_t *)(hw + cnt));
        hw += cnt + 2;
    }
    if (!rc) rc = nttm_run_fill_x(pl->blob + pl->off_z, pl->zidx.size(), pl->cs);
    if (!rc) rc = nttm_run_norm(pl->blob + pl->off_z, pl->zidx.size(), hw, pl->cs);
    hipGraph_t gr = nullptr;
    const int rc_end = nttm_hip_check(hipStreamEndCapture(pl->cs, &gr), "end capture");
    g_prof_on = prof0;
    pl->graph = gr;
    if (rc || rc_end) return fail(rc ? rc : rc_end);
    if ((rc = nttm_hip_check(hipGraphInstantiate(&pl->exec, pl->graph, nullptr, nullptr, 0), "graph instantiate"))) return fail(rc);
    *out = pl;
    return 0;
}

extern "C" int nttm_batch_plan_create(const nttm_prod *P, size_t N, int autotune, nttm_batch_plan **out, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (!out || (N && !P)) return nttm_fail(NTTM_EINVAL, "nttm_batch_plan_create arguments");
    *out = nullptr;
    const int rc = plan_create(P, N, autotune, 0, out, (hipStream_t)stream);
    return rc == NTTM_ENOMEM ? plan_create(P, N, autotune, 1, out, (hipStream_t)stream) : rc;   /* (the least planes) */
}

extern "C" int nttm_batch_plan_run(nttm_batch_plan *pl, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (!pl) return nttm_fail(NTTM_EINVAL, "null plan");
    if (pl->gen != g.gen) return nttm_fail(NTTM_ESTATE, "plan made before the last nttm_shutdown: its tables are gone");
    if (!pl->exec) return 0;
    return nttm_hip_check(hipGraphLaunch(pl->exec, (hipStream_t)stream), "graph launch");
}

extern "C" int nttm_batch_plan_ncn(nttm_batch_plan *pl, size_t *ncn, void *stream)
{
    if (!g.init) return nttm_fail(NTTM_ESTATE, "not initialised");
    if (!pl || !ncn) return nttm_fail(NTTM_EINVAL, "nttm_batch_plan_ncn arguments");
    if (pl->gen != g.gen) return nttm_fail(NTTM_ESTATE, "plan made before the last nttm_shutdown: its tables are gone");
    hipStream_t s = (hipStream_t)stream;
    HIPCK(hipStreamSynchronize(s));
    const uint64_t *h = pl->hstage;                               /* written by the run itself (pinned) */
    size_t w = 0;
    for (size_t i = 0; i < pl->gb.size(); i++) {
        const GroupBuild &x = pl->gb[i];
        if (group_lengths(x, h + w, (const uint32_t *)(h + w + x.cnt), [&](uint64_t j, uint64_t n) { ncn[pl->gidx[i][j]] = n; }))
            return nttm_fail(NTTM_ECHECK, "crt: non-zero carry beyond a top limb (wrong residues)");
        w += x.cnt + 2;
    }
    for (size_t z = 0; z < pl->zidx.size(); z++) ncn[pl->zidx[z]] = h[w + z];
    return 0;
}

/* the chosen schedule as text: one line per group, then the tuning summary */
extern "C" int nttm_batch_plan_info(const nttm_batch_plan *pl, char *buf, size_t cap)
{
    if (!pl || !buf || !cap) return nttm_fail(NTTM_EINVAL, "nttm_batch_plan_info arguments");
    size_t k = 0;
    buf[0] = 0;
    for (size_t i = 0; i < pl->gb.size() && k < cap; i++) {
        const GroupBuild &x = pl->gb[i];
        k += snprintf(buf + k, cap - k, "group points=%llu r3=%d logn=%d products=%llu shared_b=%llu tile=%d pts=%d ms=%.4f\n",
                      (unsigned long long)x.n, x.r3, x.logn, (unsigned long long)x.cnt,
                      (unsigned long long)(x.share ? x.cnt - x.cnt_b : 0), x.tile, x.pts, pl->gms[i]);
    }
    if (k < cap) k += snprintf(buf + k, cap - k, "plan products=%zu empty=%zu primes=%d candidates=%d reused=%d tune_ms=%.1f "
                               "blob_bytes=%zu\n", pl->N, pl->zidx.size(), pl->np, pl->candidates, pl->reused, pl->tune_ms,
                               pl->blob_bytes);
    return k < cap ? 0 : nttm_fail(NTTM_EINVAL, "nttm_batch_plan_info: buffer too small");
}

extern "C" void nttm_batch_plan_destroy(nttm_batch_plan *pl)
{
    if (pl && pl->cs) (void)hipStreamSynchronize(pl->cs);
    (void)hipDeviceSynchronize();                                /* no replay still reading the plan's memory */
    plan_free(pl);
}

/* ---- host-side introspection for tests: the pass plan and the tile -> element map ---------------------------------- */
extern "C" int nttm_debug_plan(int logn, uint64_t batch, int tile_log, int last_log, int *out, int cap)
{
    if (tile_log <= 0) tile_log = NTTM_TILE_LOG_DEFAULT;
    if (tile_log > NTTM_TILE_LOG || last_log > NTTM_TILE_LOG) return nttm_fail(NTTM_EINVAL, "tile logs above %d", NTTM_TILE_LOG);
    Plan pl; plan_make2(&pl, logn, batch, tile_log, last_log > 0 ? last_log : tile_log);
    int k = 0;
    for (int i = 0; i < pl.npass && k + 4 <= cap; i++) { out[k++] = pl.p[i].lo; out[k++] = pl.p[i].m; out[k++] = pl.p[i].logw; out[k++] = pl.p[i].logh; }
    return pl.npass;
}
extern "C" int nttm_debug_product_plan(int logn, uint64_t batch, int tile_log, int *out, int cap)
{
    if (tile_log <= 0) tile_log = NTTM_TILE_LOG_DEFAULT;
    if (tile_log != 12 && tile_log != 13) return nttm_fail(NTTM_EINVAL, "tile_log %d", tile_log);
    if (logn < 1 || logn > NTTM_LOGN_MAX || !batch) return nttm_fail(NTTM_EINVAL, "nttm_debug_product_plan arguments");
    Plan pl; product_plan(&pl, logn, batch, product_tile_log(logn, tile_log));
    int k = 0;
    for (int i = 0; i < pl.npass && k + 4 <= cap; i++) { out[k++] = pl.p[i].lo; out[k++] = pl.p[i].m; out[k++] = pl.p[i].logw; out[k++] = pl.p[i].logh; }
    return pl.npass;
}
extern "C" int nttm_debug_product_len(size_t ncoef, int radix3, int tile_log, int *logn, int *r3)
{
    if (!ncoef || !logn || !r3) return nttm_fail(NTTM_EINVAL, "nttm_debug_product_len arguments");
    if (radix3 < NTTM_R3_AUTO || radix3 > NTTM_R3_FIT) return nttm_fail(NTTM_EINVAL, "radix3 mode %d", radix3);
    if (tile_log <= 0) tile_log = NTTM_TILE_LOG_DEFAULT;
    if (tile_log != 12 && tile_log != 13) return nttm_fail(NTTM_EINVAL, "tile_log %d", tile_log);
    choose_len(ncoef, radix3, tile_log, logn, r3);
    return 0;
}
extern "C" int nttm_debug_tile_indices(int lo, int m, int logw, int logh, uint64_t tile, uint64_t *out)
{
    PassGeom gg; gg.lo = lo; gg.m = m; gg.logw = logw; gg.logh = logh;
    const int T = 1 << (m + logw + logh);
    for (int e = 0; e < T; e++) out[e] = plan_gidx(gg, tile, e);
    return T;
}
