/* the dispatch rules of ntt_amd/csrc/segrule.h for the host tests */
#include "../../ntt_amd/csrc/segrule.h"
extern "C" {
double t_seg_launch_us(uint64_t n, uint32_t per, uint64_t S, int ncu) { return seg_launch_us(n, per, S, ncu); }
uint32_t t_seg_choose(uint64_t segs, uint64_t S, double most, int ncu, int forced) { return seg_choose(segs, S, most, ncu, forced != 0); }
uint32_t t_seg_batch_per(const uint64_t *blocks, const uint64_t *len, size_t cnt, int ncu) { return seg_batch_per(blocks, len, cnt, ncu); }
int t_small_few(uint64_t cnt, int logn, int ncu) { return small_few(cnt, logn, ncu); }
}
