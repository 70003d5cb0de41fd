// Which form of the ring kernel (gemm_ring.h) a medium-batch launch takes, if any (host only).
#pragma once

// rw row waves of 16 rows and kw K waves per workgroup, K cut into ks slices (partial sums when > 1).  rw == 0: the
// launch stays with the whole-row sweep (gemm_dense16_kernel).
struct RingPlan {
    int rw, kw, ks;
    float us;
};

constexpr int RING_MAX_B = 64;
constexpr int ring_batch_tiles(int B) { return B <= 16 ? 1 : (B <= 32 ? 2 : 4); }

// The time of a launch of one batch tile is modelled as
//     first + next x (rounds - 1) + grid x fill + run x (c x rounds + d x fill)
// with rounds of one workgroup per CU, fill = workgroups per CU, `run` windows of 128 columns that a wave takes one after the other.
// Fits to 460 launches of 1 .. 4 tensors (500 .. 32000 rows, 512 .. 14592 columns, 3 .. 16 rows of activations, one MI355X of 256
// CUs), 1.5 % off on average with one or two K waves, 2.6 and 4 % with four and eight.
inline float ring_one_tile_us(int tiles, int kw, int windows, int ks, int B, int cus)
{
    const int per = (windows + ks - 1) / ks, run = (per + kw - 1) / kw;
    const int groups = tiles * ((windows + per - 1) / per), rounds = (groups + cus - 1) / cus;
    const float fill = (float)groups / cus;
    if (kw == 1) return 4.68f + 2.13f * (rounds - 1) + 1.91f * fill + run * (0.868f * rounds + 0.022f * fill);
    if (kw == 2) return 5.70f + 3.13f * (rounds - 1) + 1.14f * fill + run * (0.854f * rounds + 0.069f * fill);
    if (kw == 4) return 4.95f + 2.30f * (rounds - 1) + 1.47f * fill + run * (1.034f * rounds);
    return 5.18f + 2.43f * (rounds - 1) + 0.99f * fill + run * ((0.906f + 0.0127f * B) * rounds + 0.145f * fill);
}

// Two and four batch tiles: rounds x (fix + run x c), less with a part of a round.  c grows with the activations a window needs
// (B x kw rows): 0.95 us on a full grid is the memory's rate, 24.6 KB per CU and window at 6.6 TB/s.
inline float ring_form_us(int tiles, int kw, int windows, int ks, int B, int cus)
{
    const int nbt = ring_batch_tiles(B);
    if (nbt == 1) return ring_one_tile_us(tiles, kw, windows, ks, B, cus);
    const float fix = nbt == 4 ? 7.2f : (kw == 1 ? 6.2f : 6.6f);
    const float c = nbt == 4 ? (kw == 1 ? 1.05f : 1.17f) : (kw == 1 ? 0.975f : (kw == 2 ? 0.98f : 1.15f));
    const int per = (windows + ks - 1) / ks, run = (per + kw - 1) / kw;
    long long left = (long long)tiles * ((windows + per - 1) / per);
    float us = 0.0f;
    for (; left > 0; left -= cus) {
        const float fill = left >= cus ? 1.0f : (float)left / cus;
        us += fix + run * c * (0.64f + 0.36f * fill);
    }
    return us;
}

// 16-row groups per workgroup of the sweep with two batch tiles (17 .. 32 rows), 0 where it does not take the launch: at most
// one round, every workgroup reads all B activation rows.
inline int sweep_row_groups(int groups16, int groups32, int K, int B, int cus)
{
    const long long kb = (long long)K * B;
    if (groups16 <= cus && kb <= 4096 * 48) return 1;
    if (groups32 <= cus && kb <= 5120 * 32) return 2;
    return 0;
}

// The whole-row sweep on the same launch (B <= 32); up to 16 rows a fit to the launches above, 5 % off on average, of the sweep as it was before
// its loads were turned through LDS.  As it is now, 70 launches that this leaves to it (one to three tensors, 500 .. 16000 rows, 512 .. 14592 columns, 3 .. 32
// rows of activations, replayed from a graph) are predicted 17 % too slow on average, 13 % too fast to 59 % too slow; 4096 x 4096 at 24 / 32 rows
// 12.3 / 13.6 against 11.0 / 11.3 measured.  So some launches near the line still go to the ring that the sweep would be quicker at; none is slower than
// it was.  Negative: not a launch of its.
inline float sweep_us(int groups16, int groups32, int K, int B, int cus)
{
    const float k = (float)K / 4096.0f;
    if (B <= 16) {
        const int more = (groups16 + cus - 1) / cus - 1;
        return 3.79f + k * (3.03f + 0.204f * B + 0.223f * k) + more * (2.14f + k * (1.14f + 0.135f * B + 1.24f * (k < 2.0f ? k : 2.0f)));
    }
    if (B > 32) return -1.0f;
    const int rg = sweep_row_groups(groups16, groups32, K, B, cus);
    return rg == 1 ? 5.0f + k * (3.2f + 0.17f * B) : (rg == 2 ? 6.0f + 1.35f * k * (3.2f + 0.17f * B) : -1.0f);
}

// Ring or sweep.  Two tensors of as many rows as each other and more rows than columns are gate and up of a feed-forward layer:
// up to 8 rows their gated unit is taken into whichever kernel this names (t12_gemm_glu), and the sweep's paired form works in
// whole rounds of 32 + 32 rows, so where the two are close that form decides.  11008 x 4096 at 5 rows: unpaired 34.1 (sweep) and
// 34.0 us, gated 40.6 and 36.4; 8192 x 2048: 15.1 and 14.5, gated 14.6 and 15.9.
inline bool prefers_sweep(const RingPlan& ring, float sweep, const int* rows, int nseg, int K, int B, int cus)
{
    if (nseg == 2 && rows[0] == rows[1] && rows[0] > K && B >= 5 && B <= 8 && ring.us > 0.88f * sweep && ring.us < 1.06f * sweep) {
        const int sets = (rows[0] + 31) / 32, rounds = (sets + cus - 1) / cus;
        const float k = (float)K / 4096.0f, fill = (float)sets / (rounds * cus);
        return ring.us + 1.4f > rounds * (7.2f + k * (13.8f + 4.5f * k * fill * fill * fill));
    }
    return ring.us > 0.97f * sweep;
}

// rows[nseg]: the tensors of the launch; K a multiple of 128, 3 <= B <= RING_MAX_B.
//
// A K split leaves partial sums, which the caller's next kernel (t12_gemm_deferred) or a reduction launch has to read: 2.5 us and
// their traffic above 32 rows, where most are taken by the former, 4.0 us + 0.43 us per MB, what the latter was measured at, below.
// No split:
//   * up to 8 rows, where t12_gemm_swiglu has to add in the same order as t12_gemm;
//   * where t12_gemm and t12_gemm_noalloc promise none (t12_abi.h: no workspace, no second launch): up to 16 rows, and up to 32
//     on rows of at most RING_SHORT_K columns that the sweep takes in one round.  (There the reduction eats the gain anyway:
//     2048 x 4096 at 21 rows 12.5 us by the sweep, 8.6 + 7.7 in 16 slices; longer rows gain, 1024 x 8192 20.0 against 16.4.)
//     t12_gemm_deferred adds in t12_gemm's order, so it has none there either: 1 .. 2 % of a decode step of 9 .. 16 sequences.
constexpr int RING_SHORT_K = 5120;
inline RingPlan plan_ring(const int* rows, int nseg, int K, int B, int cus)
{
    const int windows = K / 128, nbt = ring_batch_tiles(B);
    long long m = 0;
    int groups16 = 0, groups32 = 0;
    for (int i = 0; i < nseg; i++) {
        m += rows[i];
        groups16 += (rows[i] + 15) / 16;
        groups32 += (rows[i] + 31) / 32;
    }
    const float sweep = sweep_us(groups16, groups32, K, B, cus);
    const bool may_split = B > 32 || (B > 16 && (sweep < 0.0f || K > RING_SHORT_K));
    const float sum_us = B > 32 ? 2.5f : 4.0f, sum_us_per_mb = B > 32 ? 0.25f : 0.43f;
    RingPlan best = {0, 0, 1, 1e30f};
    for (int kw = 1; kw <= 8; kw *= 2) {
        if ((kw == 4 && nbt > 2) || (kw == 8 && nbt > 1)) continue;      // the activations of kw windows must fit LDS
        const int rw = 8 / kw;
        int tiles = 0;
        for (int i = 0; i < nseg; i++) tiles += (rows[i] + 16 * rw - 1) / (16 * rw);
        for (int ks = 1; ks <= 16; ks++) {
            if (ks > 1 && (!may_split || (long long)tiles * ks > cus || windows / ks < 2 * kw)) break;
            const int per = (windows + ks - 1) / ks;
            if ((windows + per - 1) / per != ks) continue;
            float us = ring_form_us(tiles, kw, windows, ks, B, cus);
            if (ks > 1) us += sum_us + (float)ks * B * m * 4e-6f * sum_us_per_mb;
            if (us < best.us) best = {rw, kw, ks, us};
        }
    }
    if (sweep >= 0.0f && prefers_sweep(best, sweep, rows, nseg, K, B, cus)) return {0, 0, 1, sweep};
    return best;
}
