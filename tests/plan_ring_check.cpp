// Host program of tests/test_ring_plan.py: every plan plan_ring makes over a sweep of launches must be one the kernel
// has, with no empty K slice and partial sums that fit the fixed workspace of t12_gemm_noalloc.
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "ring_plan.h"

static uint64_t state = 0x9e3779b97f4a7c15ull;
static uint32_t rnd()
{
    state ^= state << 13;
    state ^= state >> 7;
    state ^= state << 17;
    return (uint32_t)(state >> 11);
}

int main(int argc, char** argv)
{
    const long cases = argc > 1 ? atol(argv[1]) : 100000;
    const int cu_choices[] = {1, 7, 64, 228, 256, 304};
    long plans = 0, form[9] = {}, split = 0, none = 0;
    for (long c = 0; c < cases; c++) {
        const int nseg = 1 + (int)(rnd() % 8), B = 3 + (int)(rnd() % (RING_MAX_B - 2)), K = 128 * (1 + (int)(rnd() % (rnd() % 4 ? 128 : 600)));
        const int cus = cu_choices[rnd() % 6];
        int M[8];
        long long total = 0;
        for (int i = 0; i < nseg; i++) total += M[i] = 1 + (int)(rnd() % (rnd() % 3 ? 5000 : 140000));
        const RingPlan r = plan_ring(M, nseg, K, B, cus);
        if (r.rw == 0) {
            if (B > 32) { printf("no kernel for B %d\n", B); return 1; }
            none++;
            continue;
        }
        plans++;
        const int nbt = ring_batch_tiles(B), windows = K / 128;
        if (r.rw * r.kw != 8 || (r.kw == 4 && nbt > 2) || (r.kw == 8 && nbt > 1) || r.kw < 1) { printf("form %d x %d, %d batch tiles\n", r.rw, r.kw, nbt); return 1; }
        if (r.ks < 1 || r.ks > 16 || (B <= 8 && r.ks > 1)) { printf("ks %d at B %d\n", r.ks, B); return 1; }
        const int per = (windows + r.ks - 1) / r.ks;
        if ((r.ks - 1) * per >= windows) { printf("an empty slice: %d windows, %d slices\n", windows, r.ks); return 1; }
        if (r.ks > 1 && cus <= 256 && (long long)r.ks * B * total * 4 > (32 << 20)) { printf("%lld bytes of partial sums\n", (long long)r.ks * B * total * 4); return 1; }
        form[r.kw]++;
        split += r.ks > 1;
    }
    printf("ok: %ld plans (%ld %ld %ld %ld, %ld split), %ld left to the sweep\n", plans, form[1], form[2], form[4], form[8], split, none);
    return form[1] && form[2] && form[4] && form[8] && split && none ? 0 : 2;
}
