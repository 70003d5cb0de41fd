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

// The time of a launch is modelled as  F + rounds x windows x c:  F the part that does not depend on K (launch, first
// requests, escape list, stores), rounds of one workgroup per CU, `windows` of 128 columns a wave takes one after the
// other, c the time of one.  F and c are fits to 2048 .. 14336 columns x 1024 .. 40000 rows, B = 3 .. 64, on one
// MI355X (256 CUs), good to about 1 us: with a full grid c is the memory's (24.6 KB per CU and window: 0.95 us =
// 6.6 TB/s), with half of it 0.82 of that, and it grows with the activations a window needs (B x kw rows).
inline float ring_form_us(int tiles, int kw, int windows, int ks, int B, int cus)
{
    const int t = ring_batch_tiles(B) == 1 ? 0 : (ring_batch_tiles(B) == 2 ? 1 : 2);
    const float fix[3] = {kw == 1 ? 5.6f : 6.5f, kw == 1 ? 6.2f : 6.6f, 7.2f};
    const float c1[3] = {0.95f, 0.975f, 1.05f}, c2[3] = {0.90f, 0.98f, 1.17f}, c4[3] = {0.95f, 1.15f, 1e9f};
    float c = kw == 1 ? c1[t] : (kw == 2 ? c2[t] : c4[t]);
    if (kw == 8) c = t ? 1e9f : 0.95f + 0.02f * B;
    const int per = (windows + ks - 1) / ks, run = (per + kw - 1) / kw;
    long long left = (long long)tiles * ((windows + per - 1) / per);
    float us = 0.0f;
    for (; left > 0; left -= cus) {
        const float fill = left >= cus ? 1.0f : (float)left / cus;
        us += fix[t] + run * c * (0.64f + 0.36f * fill);
    }
    return us;
}

// The whole-row sweep on the same launch (B <= 32): fits as above; its second and later rounds cost 1.7 of the first, and
// with two batch tiles it takes at most one round (of 16-row, or of 32-row workgroups).  Negative: not a launch of its.
inline float sweep_us(int groups16, int groups32, int K, int B, int cus)
{
    const float k = (float)K / 4096.0f;
    if (B <= 16) {
        const int rounds = (groups16 + cus - 1) / cus;
        float kk = k;                                       // K^1.2 without a pow: k^(6/5) ~ k (1 + ln(k) / 5)
        float ln = 0.0f;
        for (float x = k; x > 1.05f; x /= 1.05f) ln += 0.0488f;
        for (float x = k; x < 0.95f; x *= 1.05f) ln -= 0.0488f;
        kk = k * (1.0f + ln / 5.0f + ln * ln / 50.0f);
        return 5.6f + (1.0f + 1.7f * (rounds - 1)) * kk * (2.7f + 0.1f * B);
    }
    if (B > 32) return -1.0f;
    const long long kb = (long long)K * B;
    if (groups16 <= cus && kb <= 4096 * 48) return 5.0f + k * (3.2f + 0.17f * B);
    if (groups32 <= cus && kb <= 5120 * 32) return 6.0f + 1.35f * k * (3.2f + 0.17f * B);
    return -1.0f;
}

// rows[nseg]: the tensors of the launch; K a multiple of 128, 3 <= B <= RING_MAX_B.  A K split leaves partial sums, which
// a reduction launch (4.2 us + 0.3 us per MB) or the caller's next kernel has to read: it is charged 2.5 us and their
// traffic, and is not taken up to 8 rows, where t12_gemm_swiglu has to add in the same order as t12_gemm.
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
    RingPlan best = {0, 0, 1, 1e30f};
    for (int kw = 1; kw <= 8; kw *= 2) {
        if ((kw == 4 && nbt > 2) || (kw == 8 && nbt > 1)) continue;      // the activations of kw windows must fit LDS
        const int rw = 8 / kw;
        int tiles = 0;
        for (int i = 0; i < nseg; i++) tiles += (rows[i] + 16 * rw - 1) / (16 * rw);
        for (int ks = 1; ks <= 16; ks++) {
            if (ks > 1 && (B <= 8 || (long long)tiles * ks > cus || windows / ks < 2 * kw)) break;
            const int per = (windows + ks - 1) / ks;
            if ((windows + per - 1) / per != ks) continue;
            float us = ring_form_us(tiles, kw, windows, ks, B, cus);
            if (ks > 1) us += 2.5f + (float)ks * B * m * 4.0f / 4e6f;
            if (us < best.us) best = {rw, kw, ks, us};
        }
    }
    const float sweep = sweep_us(groups16, groups32, K, B, cus);
    if (sweep >= 0.0f && best.us > 0.97f * sweep) return {0, 0, 1, sweep};
    return best;
}
