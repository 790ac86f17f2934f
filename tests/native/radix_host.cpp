/* the radix steps of ntt_amd/csrc/radix.h on the host, their modular products and reductions watched: the largest operand
 * each was given, the largest output, and every output's residue against exact integers */
#include <stdint.h>
#include <math.h>
#include "../../ntt_amd/csrc/arith.h"

struct double2 { double x, y; };
static inline double2 make_double2(double x, double y) { return double2{x, y}; }
struct HTab { const double2 *w; };
static inline double2 tw_at(HTab t, uint32_t lane, uint32_t fixed) { return t.w[lane + fixed]; }

static double t_mul, t_red;                      /* largest |operand| of a product, of a reduction */
static bool t_triv;
static inline double watched_mul(double a, double w, double wq, double p) { t_mul = fmax(t_mul, fabs(a)); return mul_shoup(a, w, wq, p); }
static inline double watched_red(double s, double p, double pinv) { t_red = fmax(t_red, fabs(s)); return reduce(s, p, pinv); }
#define mul_shoup watched_mul
#define reduce watched_red
#define NTTM_TRIVIAL_W(rlow, jj) ((jj) == 0 && t_triv)
#include "../../ntt_amd/csrc/radix.h"
#undef mul_shoup
#undef reduce

typedef __int128 i128;
static uint64_t rng;
static uint64_t next(void) { rng ^= rng << 13; rng ^= rng >> 7; rng ^= rng << 17; return rng; }
static int64_t posmod(i128 v, int64_t p) { int64_t r = (int64_t)(v % p); return r < 0 ? r + p : r; }

template <int LOGR> static int run(int inv, int wide_in, int wide_out, int64_t p, uint64_t pat, double *out)
{
    constexpr int R = 1 << LOGR;
    double2 w[2 * R];
    double v[R];
    int64_t e[R];
    const int64_t lim = wide_in ? 4 * p : p;
    for (int j = 0; j < 2 * R; j++) {            /* any |w| <= p / 2 will do for the bounds: the ends, and between */
        const uint64_t r = next();
        const int64_t x = r % 4 == 0 ? p / 2 : r % 4 == 1 ? -(p / 2) : (int64_t)(next() % (uint64_t)p) - p / 2;
        w[j] = make_double2((double)x, (double)x / (double)p);
    }
    for (int j = 0; j < R; j++) {
        const int64_t x = next() % 8 ? lim : (int64_t)(next() % (uint64_t)lim);
        e[j] = (pat >> j) & 1 ? -x : x;
        v[j] = (double)e[j];
    }
    if (inv) dit_group<LOGR, HTab>(v, 0, 0, HTab{w}, (double)p, 1.0 / (double)p, wide_in != 0, wide_out != 0);
    else dif_group<LOGR, HTab>(v, 0, 0, HTab{w}, (double)p, 1.0 / (double)p);
    for (int lev = 0; lev < LOGR; lev++) {
        const int k = inv ? lev : LOGR - 1 - lev, h = 1 << k;
        for (int jj = 0; jj < h; jj++)
            for (int j = jj; j < R; j += 2 * h) {
                const bool one = t_triv && jj == 0 && (!inv || lev == 0);
                const int64_t tw = one ? 1 : (int64_t)w[h + jj].x;
                const i128 u = e[j], x = e[j + h];
                if (inv) { const i128 y = posmod(x * tw, p); e[j] = posmod(u + y, p); e[j + h] = posmod(u - y, p); }
                else { e[j] = posmod(u + x, p); e[j + h] = posmod(posmod(u - x, p) * (i128)tw, p); }
            }
    }
    int bad = 0;
    for (int j = 0; j < R; j++) {
        *out = fmax(*out, fabs(v[j]));
        bad += v[j] != floor(v[j]) || fabs(v[j]) >= 9007199254740992.0 || posmod((i128)v[j], p) != posmod(e[j], p);
    }
    return bad;
}
extern "C" {
uint64_t r_prime(int i) { return NTTM_PRIMES[i]; }
/* `count` sign patterns from `first` on; most[3]: largest operand of a product, of a reduction, largest output.  Returns the
 * number of wrong outputs */
int r_radix(int logr, int inv, int triv, int wide_in, int wide_out, int prime, uint64_t first, uint64_t count, double *most)
{
    const int64_t p = (int64_t)NTTM_PRIMES[prime];
    t_mul = t_red = 0; t_triv = triv != 0;
    rng = 0x9E3779B97F4A7C15ULL + first;
    double out = 0;
    int bad = 0;
    for (uint64_t i = first; i < first + count; i++)
        bad += logr == 1 ? run<1>(inv, wide_in, wide_out, p, i, &out) : logr == 2 ? run<2>(inv, wide_in, wide_out, p, i, &out)
             : logr == 3 ? run<3>(inv, wide_in, wide_out, p, i, &out) : run<4>(inv, wide_in, wide_out, p, i, &out);
    most[0] = t_mul; most[1] = t_red; most[2] = out;
    return bad;
}
/* the outputs that the DIF reduces at level lev (DifRed) */
uint32_t r_mask(int logr, int triv, int lev)
{
    switch (logr) {
    case 1: return triv ? DifRed<1, true>().mask[lev] : DifRed<1, false>().mask[lev];
    case 2: return triv ? DifRed<2, true>().mask[lev] : DifRed<2, false>().mask[lev];
    case 3: return triv ? DifRed<3, true>().mask[lev] : DifRed<3, false>().mask[lev];
    default: return triv ? DifRed<4, true>().mask[lev] : DifRed<4, false>().mask[lev];
    }
}
}
