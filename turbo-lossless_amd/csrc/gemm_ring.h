// Decode+GEMM for 3 .. 64 rows (included by gemm.hip): bound by the weight stream, so everything here serves to keep it
// running at the memory's rate.
//   * Planes and activations are copied global -> LDS without passing through registers (global_load_lds, 16 bytes per
//     lane), in windows of 128 columns: a copy instruction takes whole lines of a plane, two rounds of windows are in
//     flight per wave (48 KB per CU and more), and no register ring limits it.  The copies are swizzled through their
//     source addresses, so that the 16-byte reads of the MFMA operands touch every LDS bank once.
//   * A wave owns 16 weight rows and reads its own part of the ring: no barrier for the planes.  The activations of a
//     window are shared by the workgroup (one barrier per window, three buffers).  KW > 1: the waves are split into
//     groups that take every KW-th window and are added up at the end, for launches of few rows.
//   * Weights are rebuilt in registers in the order the activations have in memory (t12_decode8_seq) and go straight into
//     v_mfma_f32_16x16x32_bf16: no bf16 copy of W anywhere, no shuffling of X.  The next window is decoded between the
//     products of this one, each step's registers right behind the products that read them.
//   * Escapes are exact: the tile's list lies in LDS, each lane holds its row's next entry and puts the exact value over
//     the decoded one in its register; the entry behind it is read along with the planes.
// Measured (28672 x 4096, us, B = 16 / 32 / 64): 34.4 / 34.3 / 39.9 = 5.1 / 5.1 / 4.4 TB/s; the whole-row sweep and the
// tile kernel, which took these launches before, 44.3 / 46.9 / 48.2.  A plain read of the same planes in the same
// order takes 27.5 .. 33.  Experts (DEV: a group's rows are read from device memory, batch tiles in a loop): gate|up and down
// of eight of 4096 / 14336 at 40 tokens 232 + 118 us = 6.1 and 6.0 TB/s, the tile kernel 333 + 158.  4096 x 14336 at B = 16 unsplit 23.8,
// the sweep 28.5; at B = 32 / 64 in 4 / 8 K slices 21.4 / 23.6 and 4 .. 5.5 us for their sum, before 26.6 / 27.8 and the same.
#pragma once
#include <type_traits>

#include "gemm_params.h"

namespace {

constexpr int RING_WC = 128;                 // columns of a window
constexpr int RING_W_BYTES = 16 * RING_WC * 3 / 2;    // one wave's window: 16 rows of both planes

typedef const __attribute__((address_space(1))) void* ring_gptr;
typedef __attribute__((address_space(3))) void* ring_lptr;

__device__ __forceinline__ uint32_t ring_lds_at(const void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t*)p; }

// s_waitcnt immediate: at most n vector memory operations outstanding, nothing else waited for.
constexpr int ring_vmcnt(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }

// LDS reads of the planes' ring.  What is outstanding of the copies is counted by hand below (they run two rounds ahead
// and their slots are picked at run time); a plain LDS read would make the compiler drain every copy in flight first, so
// these are asm, with their own wait.
struct RingRaw {
    t12_u32x4 s0, s1, g;         // 32 columns of a row: sign/mantissa bytes, nibbles
};
__device__ __forceinline__ void ring_read(RingRaw& r, uint32_t sa0, uint32_t sa1, uint32_t ga, uint32_t& next, uint32_t na)
{
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b32 %3, %7\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(r.s0), "=&v"(r.s1), "=&v"(r.g), "=&v"(next)
                 : "v"(sa0), "v"(sa1), "v"(ga), "v"(na)
                 : "memory");
}
__device__ __forceinline__ uint32_t ring_read32(uint32_t at)
{
    uint32_t v;
    asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v) : "v"(at) : "memory");
    return v;
}

// LDS of a workgroup: the planes' ring (two windows per wave), the activations' ring (three windows per K wave), the
// escape list.
template <int RW, int KW, int NBT, bool DEV = false>
struct RingLds {
    static constexpr int W = RW * KW * 2 * RING_W_BYTES;
    static constexpr int XWIN = 16 * NBT * RING_WC * 2;
    static constexpr int X = KW * XWIN;                                // one round's
    static constexpr int ROWS = 16 * RW;
    static constexpr int TABLE = ROWS + 4;                             // row offsets into the list
    // (a launch over experts has many rounds of workgroups: two per CU, so that one starts while the other streams.  Its table
    // lies in the third activation buffer, which is first written behind round 0's barrier: so 17 .. 32 rows hold 2048 entries)
    static constexpr bool TABLE_IN_X = DEV;
    static constexpr int ROOM = ((DEV && NBT <= 2 ? 80 : 160) * 1024 - W - 3 * X - (TABLE_IN_X ? 0 : TABLE * 4)) / 4;
    static constexpr int CAP = ROOM > 8192 ? 8192 : (ROOM & ~63);      // escape entries held
    static_assert(CAP >= 2048, "room for the escapes of a tile");
    static_assert(!TABLE_IN_X || (TABLE * 4 <= X && RW > 1), "the table in the third activation buffer");
    static_assert((KW - 1) * RW * NBT * 64 * 16 <= W, "the sums of the K waves reuse the rings");
};

// GLU: a wave's 16 rows are 8 rows of gate and the same 8 rows of up.
template <int RW, int KW, int NBT, bool GLU, bool DEV>
__device__ __forceinline__ bool gemm_ring_body(const GemmParams& p, const int bt, uint8_t* const x0, uint8_t* const x1, uint8_t* const x2,
                                               uint8_t* const wr, int* const lrow, uint32_t* const lpat, t12_f32x4* const red)
{
    using L = RingLds<RW, KW, NBT, DEV>;
    constexpr int NT = RW * KW * 64, BP = 16 * NBT;
    constexpr int NXI = 4 * NBT;                              // activation copies of a window (4 rows of 256 bytes each)
    constexpr int NX = (NXI + RW - 1) / RW;                   // of them, per wave (the last may be one less)
    constexpr int WR = GLU ? 8 : 16;                          // rows of a tensor per wave
    constexpr int NA = NBT >= 4 ? 1 : 4 / NBT;                // accumulators per batch tile
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rw = wave % RW, kw = wave / RW;
    const int n = lane & 15, g = lane >> 4;

    const int tile = blockIdx.x;
    const int pair = GLU ? find_pair(p, tile) : 0;
    const int s = GLU ? 2 * pair : find_segment(p, tile);
    const T12Segment& sg = p.seg[s];
    const T12Segment& sg1 = p.seg[GLU ? s + 1 : s];
    const int M = sg.M, K = p.K;
    const int B = DEV ? p.dev_counts[p.group_of_seg[s]] : p.seg_B[s];
    const int b0 = bt * BP;
    if (b0 >= B) return false;
    const int row_base = DEV ? p.dev_base[p.group_of_seg[s]] : 0;
    const int act_stride = p.seg_act_stride[s];
    const uint16_t* const act = p.seg_act[s] + (size_t)row_base * act_stride;
    const int m0 = (tile - p.blk_start[GLU ? pair : s]) * (WR * RW);
    const int k_begin = blockIdx.z * p.kslice;
    const int nwin = (min(K, k_begin + p.kslice) - k_begin) / RING_WC;
    const int T = (nwin + KW - 1) / KW;                       // rounds: wave kw takes windows kw, kw + KW, ...
    // Where in its slice a workgroup begins: four rounds further for every 1024 rows, wrapping around.  Rows lie K bytes
    // apart; with K a power of two and every workgroup at the same columns the chip as a whole reads a few memory
    // channels at a time (28672 x 4096: 32.5 us in phase, 27.5 us rotated, plain reads of the planes).  A function of the
    // row alone, so that a row's sums are taken in the same order whatever else the launch holds.
    const int rot = T >= 8 ? (int)((unsigned)(m0 >> 10) * 4u % (unsigned)T) : 0;
    auto window = [&](int t) __attribute__((always_inline)) {              // t < T
        int r = t + rot;
        r = r >= T ? r - T : r;
        return KW > 1 ? min(kw + r * KW, nwin - 1) : r;
    };

    // ---- this lane's part of the copies
    const int wm0 = m0 + WR * rw;                             // first row of this wave
    const uint8_t* s_src[2];
    {
        const int q = lane & 7;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int r = 8 * i + (lane >> 3);
            const int piece = q ^ (r & 7) ^ (r >> 3);         // swizzle: see the reads below
            const uint8_t* plane = GLU && i ? sg1.sm : sg.sm;
            s_src[i] = plane + (size_t)min(wm0 + (GLU ? r & 7 : r), M - 1) * K + k_begin + 16 * piece;
        }
    }
    const uint8_t* g_src;
    {
        const int r = lane >> 2, piece = (lane & 3) ^ ((r >> 1) & 3) ^ (r >> 3);
        const uint8_t* plane = GLU && (r >> 3) ? sg1.gr : sg.gr;
        g_src = plane + (((size_t)min(wm0 + (GLU ? r & 7 : r), M - 1) * K + k_begin) >> 1) + 16 * piece;
    }
    const uint16_t* x_src[NX];
    uint32_t x_dst[NX];
    int nx = 0;
#pragma unroll
    for (int j = 0; j < NX; j++) {
        const int i = j * RW + rw;                            // copy number: rows 4 i .. 4 i + 3
        if (i < NXI) nx = j + 1;
        const int r = 4 * min(i, NXI - 1) + (lane >> 4);
        const int piece = (lane & 15) ^ (r & 15);
        x_src[j] = act + (size_t)min(b0 + r, B - 1) * act_stride + k_begin + 8 * piece;
        x_dst[j] = kw * L::XWIN + 1024 * min(i, NXI - 1);
    }
    auto copy_x = [&](uint8_t* to, int t) __attribute__((always_inline)) {
        const int win = window(t);
#pragma unroll
        for (int j = 0; j < NX; j++)
            if (j < nx)
                __builtin_amdgcn_global_load_lds((ring_gptr)(x_src[j] + (size_t)win * RING_WC), (ring_lptr)(to + x_dst[j]), 16, 0, 0);
    };
    auto copy_w = [&](int t, int slot) __attribute__((always_inline)) {
        const int win = window(t);
        const uint32_t to = (wave * 2 + slot) * RING_W_BYTES;
#pragma unroll
        for (int i = 0; i < 2; i++)
            __builtin_amdgcn_global_load_lds((ring_gptr)(s_src[i] + (size_t)win * RING_WC), (ring_lptr)(wr + to + 1024 * i), 16, 0, 2);
        // (a window takes half a line of the nibble plane; its other half is due a round later and must stay in L2 until then,
        // so this copy is not a streaming one: with the hint the plane came in twice, 202 MB for 176 MB of 28672 x 4096)
        __builtin_amdgcn_global_load_lds((ring_gptr)(g_src + (size_t)win * (RING_WC / 2)), (ring_lptr)(wr + to + 2048), 16, 0, 0);
    };
    copy_w(0, 0);
    copy_x(x0, 0);
    copy_w(min(1, T - 1), 1);                                 // (past the last round: the last one again, not used)

    // ---- the escape list of the workgroup's rows -> LDS (esc_mode as TileList's mode)
    int esc_mode = 0;
    if (GLU) {
        const int r_lo = min(m0, M), r_hi = min(m0 + WR * RW, M);
        const int e0 = sg.row_off ? sg.row_off[r_lo] : 0, e1 = sg1.row_off ? sg1.row_off[r_lo] : 0;
        const int n0 = sg.row_off ? sg.row_off[r_hi] - e0 : 0, n1 = sg1.row_off ? sg1.row_off[r_hi] - e1 : 0;
        if (sg.row_off || sg1.row_off) esc_mode = (n0 + n1 <= L::CAP && K <= 65536) ? 1 : 2;
        if (esc_mode == 1) {
            for (int t = tid; t < n0; t += NT) lpat[t] = (uint32_t)sg.cols[e0 + t] | ((uint32_t)(uint16_t)sg.correct[e0 + t] << 16);
            for (int t = tid; t < n1; t += NT) lpat[n0 + t] = (uint32_t)sg1.cols[e1 + t] | ((uint32_t)(uint16_t)sg1.correct[e1 + t] << 16);
            for (int t = tid; t <= WR * RW; t += NT) {
                lrow[t] = sg.row_off ? sg.row_off[min(m0 + t, M)] - e0 : 0;
                lrow[WR * RW + 1 + t] = n0 + (sg1.row_off ? sg1.row_off[min(m0 + t, M)] - e1 : 0);
            }
        }
    } else if (sg.row_off) {
        const int e0 = sg.row_off[min(m0, M)], e1 = sg.row_off[min(m0 + WR * RW, M)];
        esc_mode = (e1 - e0 <= L::CAP && K <= 65536) ? 1 : 2;
        if (esc_mode == 1) {
            for (int t = tid; t < e1 - e0; t += NT) lpat[t] = (uint32_t)sg.cols[e0 + t] | ((uint32_t)(uint16_t)sg.correct[e0 + t] << 16);
            for (int t = tid; t <= WR * RW; t += NT) lrow[t] = sg.row_off[min(m0 + t, M)] - e0;
        }
    }
    const uint32_t at_pat = ring_lds_at(lpat);
    uint32_t e_at = 0, e_end = 0;                             // byte offsets of this lane's row's entries
    int e_col = 0x7FFFFFFF;                                   // column of the next one
    uint32_t e_val = 0;
    uint32_t e_at0 = 0, e_val0 = 0;                           // the slice's first one, for the way around its end
    int e_col0 = 0x7FFFFFFF;
    if (esc_mode == 1) {
        __syncthreads();
        const int li = GLU ? (n >> 3) * (WR * RW + 1) + WR * rw + (n & 7) : WR * rw + n;
        const int q0 = lrow[li], q1 = lrow[li + 1];
        auto first_from = [&](int q, int col) __attribute__((always_inline)) {
            int hi = q1;
            while (q < hi) {
                const int mid = (q + hi) >> 1;
                if ((int)(lpat[mid] & 0xFFFFu) < col) q = mid + 1;
                else hi = mid;
            }
            return q;
        };
        int q = k_begin > 0 ? first_from(q0, k_begin) : q0;
        e_end = 4 * q1;
        e_at = e_at0 = 4 * q;
        if (q < q1) {
            e_col = e_col0 = (int)(lpat[q] & 0xFFFFu);
            e_val = e_val0 = lpat[q] >> 16;
        }
        if (rot > 0) {
            q = first_from(q, k_begin + window(0) * RING_WC);
            e_at = 4 * q;
            e_col = q < q1 ? (int)(lpat[q] & 0xFFFFu) : 0x7FFFFFFF;
            e_val = q < q1 ? lpat[q] >> 16 : 0;
        }
    }

    // ---- LDS addresses of the reads.  Lane (n, g) takes row n, columns 32 g .. 32 g + 31 of a window: pieces 2 g and
    //      2 g + 1 of the row's eight 16-byte pieces of sign/mantissa, piece g of its four of nibbles.  A piece lies in
    //      slot piece ^ (row % 8) ^ (row / 8) (nibbles: ^ ((row / 2) % 4) ^ (row / 8)), so that 16 neighbouring lanes
    //      reading one piece of 16 rows touch every LDS bank once.  Activations: row b of a tile, piece 4 g + step, in
    //      slot piece ^ b of the row's sixteen.
    const int sw = (n & 7) ^ (n >> 3);
    const uint32_t at_w = ring_lds_at(wr) + wave * (2 * RING_W_BYTES);
    const uint32_t sa0 = at_w + n * 128 + 16 * ((2 * g) ^ sw);
    const uint32_t sa1 = at_w + n * 128 + 16 * ((2 * g + 1) ^ sw);
    const uint32_t ga = at_w + 2048 + n * 64 + 16 * (g ^ ((n >> 1) & 3) ^ (n >> 3));
    int xo[4];
#pragma unroll
    for (int q = 0; q < 4; q++) xo[q] = kw * L::XWIN + n * 256 + 16 * ((4 * g + q) ^ n);

    const int be = GLU && n >= 8 ? sg1.base_exp : sg.base_exp;
    const uint32_t be2 = t12_opaque(((uint32_t)be << 7) | ((uint32_t)be << 23));
    t12_f32x4 acc[NA][NBT];
#pragma unroll
    for (int a = 0; a < NA; a++)
#pragma unroll
        for (int u = 0; u < NBT; u++) acc[a][u] = t12_f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    RingRaw raw;
    uint32_t e_next = 0;                                      // the entry behind the next one, read along with the planes
    uint32_t w[16];                                           // decoded weights of the round
    auto decode = [&](int q) __attribute__((always_inline)) {
        if (q == 0) t12_decode8_seq(raw.s0.x, raw.s0.y, raw.g.x, be2, w);
        if (q == 1) t12_decode8_seq(raw.s0.z, raw.s0.w, raw.g.y, be2, w + 4);
        if (q == 2) t12_decode8_seq(raw.s1.x, raw.s1.y, raw.g.z, be2, w + 8);
        if (q == 3) t12_decode8_seq(raw.s1.z, raw.s1.w, raw.g.w, be2, w + 12);
    };
    // the escapes among the weights of round t: the lane that holds one puts the exact value in its place
    auto patch = [&](int t) __attribute__((always_inline)) {
        const int k_abs = k_begin + window(t) * RING_WC;
        bool have = true;                                     // e_next is the entry behind e_at
        if (t + rot == T) {                                   // around the end of the slice
            e_at = e_at0;
            e_col = e_col0;
            e_val = e_val0;
            have = false;
        }
        if (!__any(e_col < k_abs + RING_WC)) return;
        do {
            const int e = e_col - k_abs - 32 * g;             // 0 .. 31: one of this lane's
            const uint32_t keep = (e & 1) ? 0x0000FFFFu : 0xFFFF0000u;
            const uint32_t put = (e & 1) ? e_val << 16 : e_val;
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (__any((unsigned)(e - 8 * q) < 8u)) {
#pragma unroll
                    for (int j = 0; j < 4; j++) w[4 * q + j] = (e >> 1) == 4 * q + j ? (w[4 * q + j] & keep) | put : w[4 * q + j];
                }
            if (e_col < k_abs + RING_WC) {
                e_at += 4;
                e_col = 0x7FFFFFFF;
                if (e_at < e_end) {
                    const uint32_t v = have ? e_next : ring_read32(at_pat + e_at);
                    e_col = (int)(v & 0xFFFFu);
                    e_val = v >> 16;
                }
            }
            have = false;
        } while (__any(e_col < k_abs + RING_WC));
    };

    // The round past an uneven number of windows: the last K waves have none and take no products (the window they would
    // repeat is another wave's; with their weights at zero an infinite activation in it would still make every sum of its
    // row NaN).
    const int none = KW > 1 && kw + (T - 1) * KW >= nwin ? T - 1 - rot : -1;

    // round 0's weights
    __builtin_amdgcn_s_waitcnt(ring_vmcnt(3));
    asm volatile("" ::: "memory");
    ring_read(raw, sa0, sa1, ga, e_next, at_pat + min(e_at + 4, (uint32_t)(4 * L::CAP - 4)));
#pragma unroll
    for (int q = 0; q < 4; q++) decode(q);
    patch(0);
    copy_x(x1, min(1, T - 1));
    copy_w(min(2, T - 1), 0);

    // One round.  The activations of round t and the planes of round t + 1 have landed when only the copies requested in
    // round t - 1 (activations of t + 1, planes of t + 2) are outstanding.  Between the products of window t the wave
    // decodes window t + 1, a step's weights behind the products that used its registers.  full: every request of the
    // round is issued, without a condition around it (the compiler counts copies per path, and behind a condition it
    // would wait for all of them).
    auto round = [&](const uint8_t* xb, uint8_t* xfree, const int t, auto full_c) __attribute__((always_inline)) {
        constexpr bool full = decltype(full_c)::value;
        if (full || t + 2 < T) {
            if (nx == NX) __builtin_amdgcn_s_waitcnt(ring_vmcnt(3 + NX));
            else __builtin_amdgcn_s_waitcnt(ring_vmcnt(2 + NX));
        } else {
            __builtin_amdgcn_s_waitcnt(ring_vmcnt(0));
        }
        asm volatile("" ::: "memory");
        if (RW > 1) {
            __builtin_amdgcn_s_barrier();      // everybody's share of the activations is there, and the buffer of round t - 1 is read
            asm volatile("" ::: "memory");
        }
        if (full || t + 2 < T) copy_x(xfree, t + 2);
        t12_u32x4 x[2][NBT];
#pragma unroll
        for (int u = 0; u < NBT; u++) x[0][u] = *(const t12_u32x4*)(xb + xo[0] + 4096 * u);
        const uint32_t wo = ((t + 1) & 1) * RING_W_BYTES;
        ring_read(raw, sa0 + wo, sa1 + wo, ga + wo, e_next, at_pat + min(e_at + 4, (uint32_t)(4 * L::CAP - 4)));
        if (full || t + 3 < T) copy_w(t + 3, (t + 1) & 1);
        if (KW == 1 || t != none) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (q < 3) {
#pragma unroll
                    for (int u = 0; u < NBT; u++) x[(q + 1) & 1][u] = *(const t12_u32x4*)(xb + xo[q + 1] + 4096 * u);
                }
                const uint4 wv = make_uint4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
#pragma unroll
                for (int u = 0; u < NBT; u++)
                    acc[q % NA][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(t12_bf16x8, x[q & 1][u]),
                                                                             __builtin_bit_cast(t12_bf16x8, wv), acc[q % NA][u], 0, 0, 0);
                decode(q);
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) decode(q);
        }
        if (full || t + 1 < T) patch(t + 1);
    };
    int t = 0;
    for (; t + 6 <= T; t += 3) {
        round(x0, x2, t, std::true_type());
        round(x1, x0, t + 1, std::true_type());
        round(x2, x1, t + 2, std::true_type());
    }
    for (; t < T; t += 3) {
        round(x0, x2, t, std::false_type());
        if (t + 1 < T) round(x1, x0, t + 1, std::false_type());
        if (t + 2 < T) round(x2, x1, t + 2, std::false_type());
    }
    t12_f32x4 sum[NBT];
#pragma unroll
    for (int u = 0; u < NBT; u++) {
        sum[u] = acc[0][u];
#pragma unroll
        for (int a = 1; a < NA; a++) sum[u] += acc[a][u];
    }

    // ---- more escapes than the list holds: acc += (correct - wrong) * x, by the split and K wave that own column 0
    const int r_mat = wm0 + (GLU ? n & 7 : n);
    if (esc_mode == 2 && blockIdx.z == 0 && kw == 0 && r_mat < M) {
        const T12Segment& sr = GLU && n >= 8 ? sg1 : sg;
        if (sr.row_off) {
            const int beg = sr.row_off[r_mat], end = sr.row_off[r_mat + 1];
            for (int e = beg; e < end; e++) {
                const int col = sr.cols[e];
                const float delta = t12_bf16_to_f32((uint16_t)sr.correct[e]) - t12_bf16_to_f32((uint16_t)sr.wrong[e]);
#pragma unroll
                for (int u = 0; u < NBT; u++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        sum[u][r] += delta * t12_bf16_to_f32(act[(size_t)min(b0 + 16 * u + 4 * g + r, B - 1) * act_stride + col]);
            }
        }
    }

    // ---- the K waves' sums, added in their order by wave (rw, 0)
    if (KW > 1) {
        __syncthreads();
        if (kw > 0) {
#pragma unroll
            for (int u = 0; u < NBT; u++) red[((kw - 1) * RW + rw) * (NBT * 64) + u * 64 + lane] = sum[u];
        }
        __syncthreads();
        if (kw > 0) return true;
#pragma unroll
        for (int u = 0; u < NBT; u++)
            for (int j = 0; j < KW - 1; j++) sum[u] += red[(j * RW + rw) * (NBT * 64) + u * 64 + lane];
    }

    // ---- store: register r of lane (n, g) in batch tile u is D[batch 16 u + 4 g + r][row n]
    if (GLU) {
        uint16_t* const ob = p.out_bf16 + (size_t)row_base * p.out_bf16_ld;
        // gate in lanes n < 8, the same rows of up in lanes n + 8 (all lanes active: no branch around the exchange)
        float up[NBT][4];
#pragma unroll
        for (int u = 0; u < NBT; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) up[u][r] = __shfl_xor(sum[u][r], 8, T12_WAVE);
#pragma unroll
        for (int u = 0; u < NBT; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int b = b0 + 16 * u + 4 * g + r;
                if (n < 8 && wm0 + n < M && b < B) ob[(size_t)b * p.out_bf16_ld + wm0 + n] = t12_f32_to_bf16(t12_apply_glu(sum[u][r], up[u][r], p.glu));
            }
        return true;
    }
    const int m = wm0 + n;
    float* dst;
    size_t ld;
    if (p.ksplit > 1) {
        dst = p.ws + (size_t)blockIdx.z * p.split_stride + p.seg_ws0[s];
        ld = p.seg_ld[s];
    } else {
        dst = sg.out + (size_t)row_base * sg.out_stride;
        ld = sg.out_stride;
    }
#pragma unroll
    for (int u = 0; u < NBT; u++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int b = b0 + 16 * u + 4 * g + r;
            if (m < M && b < B) dst[(size_t)b * ld + m] = sum[u][r];
        }
    return true;
}

template <int RW, int KW, int NBT, bool GLU = false, bool DEV = false>
__global__ __launch_bounds__(RW * KW * 64, DEV && NBT <= 2 ? 4 : 2) void gemm_ring_kernel(const GemmParams p)
{
    // (arrays of their own: the compiler then knows that a read of one needs no wait for copies into another)
    using L = RingLds<RW, KW, NBT, DEV>;
    __shared__ __attribute__((aligned(16))) uint8_t x0[L::X], x1[L::X], x2[L::X], wr[L::W];
    __shared__ int table[L::TABLE_IN_X ? 1 : L::TABLE];
    __shared__ uint32_t lpat[L::CAP];
    int* const lrow = L::TABLE_IN_X ? (int*)x2 : table;
    for (int bt = blockIdx.y;; bt++) {
        if (!gemm_ring_body<RW, KW, NBT, GLU, DEV>(p, bt, x0, x1, x2, wr, lrow, lpat, (t12_f32x4*)wr) || !DEV) break;
        __syncthreads();                                   // the next tile reuses the rings
    }
}

}  // namespace
