/* segrule.h - the rules of the dispatch that count workgroups against the device's CUs (host code, plain C++).  Times in
 * microseconds; a CU has room for one workgroup of k_segments. */
#ifndef NTTM_SEGRULE_H
#define NTTM_SEGRULE_H
#include <math.h>
#include <stddef.h>
#include <stdint.h>

#define NTTM_CUS 256               /* CUs of the device the times and rates of the rules were measured on (all of an MI355X) */
#define SEG_PER_MAX 8              /* segments of a workgroup of k_segments */
#define SEG_B_US 13.0              /* a workgroup of k_segments: the short operand's transforms, ... */
static inline double seg_us(uint64_t S) { return 21.0 + 10.0 * (double)S / 4096; }   /* ... and each segment of S limbs */
/* the launch's time in workgroups of `per` segments, n workgroups in all */
static inline double seg_launch_us(uint64_t n, uint32_t per, uint64_t S, int ncu)
{
    const double r = (double)n / ncu;
    return (r <= 4 ? ceil(r) : r + 0.5) * (SEG_B_US + seg_us(S) * per);
}
/* one product of `segs` segments of S limbs: the segments of a workgroup that give it the least time, if that is below `most`;
 * else 0 (forced: 1 at least) */
static inline uint32_t seg_choose(uint64_t segs, uint64_t S, double most, int ncu, bool forced)
{
    uint32_t best = 0;
    for (uint32_t per = 1; per <= SEG_PER_MAX; per++) {
        const double us = 17.0 + seg_launch_us((segs + per - 1) / per, per, S, ncu);
        if (us < most || (forced && !best)) { most = us; best = per; }
    }
    return best;
}
/* a batch of cnt products of blocks[i] segments of len[i] limbs: segments of a workgroup, at most.  A product's are shared out
 * evenly, the products come longest first, and the launch ends within about a quarter of its longest workgroup.  (Every
 * workgroup taken for a full one, in the callers' order: the 4096 leaves' plan 4.70 ms, so 4.50.) */
static inline uint32_t seg_batch_per(const uint64_t *blocks, const uint64_t *len, size_t cnt, int ncu)
{
    double least = 0;
    uint32_t best = 1;
    for (uint32_t per = 1; per <= SEG_PER_MAX; per++) {
        double sum = 0, longest = 0;
        uint64_t n = 0;
        for (size_t i = 0; i < cnt; i++) {
            const uint64_t sb = blocks[i], k = (sb + per - 1) / per;
            const double us = SEG_B_US + seg_us(len[i]) * (double)((sb + k - 1) / k);
            sum += us * (double)k; n += k; longest = us > longest ? us : longest;
        }
        const double r = (double)n / ncu, us = r <= 4 ? ceil(r) * longest : sum / ncu + longest / 4;
        if (per == 1 || us < least) { least = us; best = per; }
    }
    return best;
}
/* one-kernel products of 2^logn points, cnt of them: few enough for a block each, spread over more waves (2^11 points a CU) */
static inline bool small_few(uint64_t cnt, int logn, int ncu) { return cnt <= ((uint64_t)ncu << 11) >> logn; }
#endif
