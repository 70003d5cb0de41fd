// Decode+GEMM for more than 64 rows (and for 3 .. 64 where K is no multiple of 128 or the planes lie at odd addresses); included by gemm.hip.
//   * v_mfma_f32_32x32x16_bf16, activations as the A operand (rows = batch), weights as the B operand (columns = output features): an accumulator
//     register holds 32 consecutive features of one batch row, so stores to out[b, m] coalesce without a transpose.
//   * A stage is 64 columns.  Its activations are copied global -> LDS without passing through registers (16 bytes per lane, whole lines, swizzled
//     through the source addresses); its planes go to registers, are rebuilt there in the order the activations have in memory (t12_decode2_seq) and
//     written once per workgroup into a bf16 tile in LDS.  No bf16 copy of W ever exists in HBM, and every weight is decoded once per workgroup.
//   * The reads of one 16-column step's operands lie between the products of the step before, at a fixed place each, and the decode of the next
//     stage's weights between the later ones: what is not issued under a running product is serial time.  The barrier of a stage lies in front of its
//     last step, whose operands are in registers by then: the reads of the next stage's first step run under its products.
//   * Escapes are exact and cost no extra pass: the (column, exact bf16) pairs of the tile's rows -- one contiguous slice of the CSR list -- are staged in
//     LDS once; the thread that decoded 16 columns of a row walks that row's slice in step with the K loop and overwrites the decoded half-words.
//
// Times here and at the rules of gemm.hip: a loop of one product over copies of its weights of 600 MB, both sides in turn on one card, us, launch gap and
// the reduction of K slices included; the cards and loops of other days differ by up to 15 % either way, so only pairs compare.
//
// gemm_tile_kernel: 256 batch rows x 128 weight rows.  Four waves multiply (one per SIMD, 128 x 64 each), the four others copy the activations; all
// eight decode.  Against eight multiplying waves of half the tile that also carried the activations through registers: a quarter fewer LDS reads, two
// thirds fewer LDS writes (13 cycles per 1 KB where a read takes 4), no shuffling of activations.  Those waves -> these: 28672 x 4096 at B = 256 78.5 -> 76.2,
// 32000 x 4096 at 256 86.3 -> 82.9, 4096 x 14336 at 256 / 512 51.9 -> 50.3 / 80.6 -> 77.3, 6144 x 4096 at 256 33.9 -> 32.7.  What bounds it, per stage and CU: the matrix cores (1024 cycles), and the
// loads, which the vector cache takes in order (860 cycles of look-ups, and waiting for planes from HBM in between): 1740 together (1300 without loads of
// planes, 1100 without the decode as well).
//
// gemm_strip_kernel: 64 or 128 batch rows x 128 weight rows, the same roles, two stages between barriers.  28672 x 4096 at B = 100 / 128 56.3 -> 51.5 /
// 56.7 -> 51.7 (gated epilogue 55.8 -> 51.4 / 56.6 -> 51.3), 4096 x 14336 at 100 37.1 -> 35.3, 6144 x 4096 25.6 -> 23.9 (one stage between barriers is 3 / 9 / 0 / 5 %
// slower).  Streaming the planes and decoding them alone takes 41 (a plain read 28); loads further ahead (four windows, five to seven buffers of
// activations) are 2 .. 5 % slower.
//
// gemm_wide_kernel: 256 batch rows x 256 weight rows, eight waves of 128 x 64: half the activation traffic and half the LDS writes of activations per
// product.  28672 x 4096 at B = 512 / 1024 140 -> 124 / 271 -> 238 (gemm_tile_kernel -> here), with the gated epilogue at 512 152 -> 129 (eight multiplying waves of
// half the 256 x 128 tile -> here); 2850 cycles per stage against 2048 of the matrix cores, at 1.8 GHz (with every CU multiplying the chip runs no faster).
// Measured and not taken: four waves of 128 x 128 with 512 registers (165: nothing covers a wave's waits), the reads and the decode in other places
// between the products, wave priorities (all level or slower), the tile kernel's copies spread between the parts of its decode (2 % slower), its
// stages begun at another column in every row tile (level; with K slices, whose activations then leave L2, 15 % slower).
#pragma once
#include <type_traits>

#include "gemm_params.h"
#include "gemm_ring.h"

namespace {

constexpr int KC = 64;          // K columns of a stage
constexpr int TM = 128;         // weight rows of a tile
constexpr int PCAP = 2048;      // escape entries held for one
constexpr int NO_ESCAPE = 0x7FFFFFFF;

// How far apart two arrays lie, one value in the wave.  A lane that picks one of the two tensors of a pair adds it or not: between the
// pointers themselves the compiler would choose a pointer to load, a chain of loads per lane.
__device__ __forceinline__ int64_t apart(const void* a, const void* b)
{
    const uint64_t d = (uint64_t)(uintptr_t)b - (uint64_t)(uintptr_t)a;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)d), hi = __builtin_amdgcn_readfirstlane((uint32_t)(d >> 32));
    return (int64_t)((uint64_t)hi << 32 | lo);
}
// A word that is one value in the wave and that no kernel in flight writes.
__device__ __forceinline__ int scalar_load(const int* p) { return *(const __attribute__((address_space(4))) int*)(uintptr_t)p; }

// LDS slot of (unit, row) in a [units][rows] array of 16-byte units.  Rows change places inside their aligned block of eight by the unit's number, so that
// both access patterns are bank-conflict free: the staging writes (neighbouring lanes = the units of one row) and the fragment reads (neighbouring lanes
// = consecutive rows of one unit).  Unit u ^ 1 of a row lies at its slot ^ 1, 2 t units on at slot ^ (2 t) (and their rows on).
__device__ __forceinline__ int lds_slot(int u, int r, int rows) { return u * rows + (r ^ (u & 7)); }

// Activation row stride (so K too) up to which a tile's 32-bit offsets reach: 256 rows of activations or of weights at 2^31 bytes, half of the range.
// Rows further apart go to gemm_strip_kernel<FAR>, whose lanes hold addresses: same K slices and order of sums, so the same bits.
constexpr int TILE_MAX_STRIDE = 1 << 22;
template <class T>
__device__ __forceinline__ T global_load(const void* p) { return *(const __attribute__((address_space(1))) T*)(uintptr_t)p; }

// Workgroups go round the eight XCDs; the batch tiles of one row tile follow each other on the same one, whose L2 then holds the row tile's planes
// for all of them.
__device__ __forceinline__ void tile_of_block(int& tile, int& bt)
{
    const int nb = gridDim.y, at = blockIdx.x + gridDim.x * blockIdx.y;
    const int group = at / (8 * nb), in = at - group * (8 * nb), n = min(8, (int)gridDim.x - 8 * group);
    tile = 8 * group + in % n;
    bt = in / n;
}

__device__ __forceinline__ void tile_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
constexpr int TILE_LDS_DONE = 0xC07F;         // s_waitcnt: LDS operations done, nothing else
// The loops count the loads of planes behind a copy, those of their last round too, which nobody decodes: used here, behind the loop, they are not dropped.
__device__ __forceinline__ void tile_keep(const t12_u32x4 (&s)[2][2], const t12_u32x2 (&g)[2][2])
{
    asm volatile("" : : "v"(s[0][0]), "v"(s[0][1]), "v"(s[1][0]), "v"(s[1][1]), "v"(g[0][0]), "v"(g[0][1]), "v"(g[1][0]), "v"(g[1][1]));
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_buffer(const void* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, -1, 0x00027000); }

// Which part of a launch a workgroup computes.  SWI (two segments of equal M, gate and up): a tile of ROWS rows holds ROWS / 2 of each, in turn by
// blocks of 32 -- local rows [0,32) gate rows 0..31, [32,64) up rows 0..31, [64,96) gate 32..63, ... -- so that two neighbouring accumulator tiles of a
// wave are gate and up of the SAME 32 rows and the epilogue writes bf16( silu(gate) * up ) straight from registers: the reference's
// silu_mul_bf16 kernel (engine/kernels.hip:447-459) and the fp32 round trip of both projections folded away.
// EPI (T12_ACT_*, one segment, no K split): the unary function of every sum is stored as bf16 to out_bf16.
template <int ROWS, bool SWI, bool DEV>
struct TileJob {
    const T12Segment &sg, &sg1;               // the tensor, SWI: gate and up
    const uint16_t* act;
    int s, M, K, B, row_base, act_stride, m0, b0, k_begin, nstage;

    __device__ __forceinline__ static int segment(const GemmParams& p, int tile) { return SWI ? 2 * find_pair(p, tile) : find_segment(p, tile); }
    __device__ __forceinline__ TileJob(const GemmParams& p, int tile, int bt, int TB)
        : sg(p.seg[segment(p, tile)]), sg1(p.seg[segment(p, tile) + (SWI ? 1 : 0)]), s(segment(p, tile))
    {
        M = sg.M;
        K = p.K;
        B = DEV ? p.dev_counts[p.group_of_seg[s]] : p.seg_B[s];
        row_base = DEV ? p.dev_base[p.group_of_seg[s]] : 0;             // first row of this group in act / out
        act_stride = p.seg_act_stride[s];
        act = p.seg_act[s] + (size_t)row_base * act_stride;
        m0 = SWI ? (tile - p.blk_start[s / 2]) * (ROWS / 2) : (tile - p.blk_start[s]) * ROWS;
        b0 = bt * TB;
        k_begin = blockIdx.z * p.kslice;
        nstage = (min(K, k_begin + p.kslice) - k_begin) / KC;
    }
    // local row -> row of its tensor, from m0
    __device__ __forceinline__ static int rel(int r) { return SWI ? ((r >> 6) << 5) + (r & 31) : r; }
};

// The escape list of a tile's rows.  They are consecutive, so their entries are one slice of cols[] / correct[] per tensor.
// mode: 0 none, 1 staged in LDS, 2 too many for that (or K > 65536): wrong values multiplied, corrected in the epilogue.
// What a workgroup waits for before its first product is a chain of loads, 1 us each: the ends of the slice come by scalar loads, every row's offset is
// requested along with them.
template <int ROWS, bool SWI, int CAP>
struct TileList {
    static constexpr int ER = SWI ? ROWS / 2 : ROWS;                    // rows of a tensor
    static constexpr int TABLE = ROWS + 4;
    int mode = 0, e0 = 0, e1 = 0, n0 = 0, n1 = 0;                       // first entry and number of entries, per tensor
    int my_off = 0;                                                     // thread t: offset of row t (SWI: of up's row t - ER - 1)
    bool has0, has1;

    template <class Job>
    __device__ __forceinline__ explicit TileList(const Job& j) : has0(j.sg.row_off), has1(SWI && j.sg1.row_off)
    {
        const int tid = threadIdx.x;
        if (!has0 && !has1) return;
        // (a tensor without a list: any readable address)
        const int* r0 = has0 ? j.sg.row_off : (const int*)j.sg.sm;
        const int* r1 = has1 ? j.sg1.row_off : (const int*)j.sg.sm;
        const int lo = min(j.m0, j.M), hi = min(j.m0 + ER, j.M);
        e0 = scalar_load(r0 + (has0 ? lo : 0));
        n0 = scalar_load(r0 + (has0 ? hi : 0));
        e1 = scalar_load(r1 + (has1 ? lo : 0));
        n1 = scalar_load(r1 + (has1 ? hi : 0));
        if (SWI && tid > ER) {
            if (has1 && tid <= 2 * ER + 1) my_off = j.sg1.row_off[min(j.m0 + tid - ER - 1, j.M)];
        } else if (has0 && tid <= ER) {
            my_off = j.sg.row_off[min(j.m0 + tid, j.M)];
        }
        n0 = has0 ? n0 - e0 : 0;
        n1 = has1 ? n1 - e1 : 0;
        mode = n0 + n1 <= CAP && j.K <= 65536 ? 1 : 2;
    }
    // col | exact value << 16 of every entry, and where a row's entries begin (SWI: ER + 1 places per tensor); 512 threads
    template <class Job>
    __device__ __forceinline__ void stage(const Job& j, uint32_t* lpat, int* lrow) const
    {
        if (mode != 1) return;
        const int tid = threadIdx.x;
        const int64_t cols_apart = SWI ? apart(j.sg.cols, j.sg1.cols) : 0, exact_apart = SWI ? apart(j.sg.correct, j.sg1.correct) : 0;
        for (int t = tid; t < n0 + n1; t += 512) {
            const bool second = SWI && t >= n0;
            const int64_t e = second ? e1 + t - n0 : e0 + t;
            const uint32_t col = *(const uint32_t*)((const uint8_t*)j.sg.cols + ((second ? cols_apart : 0) + 4 * e));
            const uint32_t exact = *(const uint16_t*)((const uint8_t*)j.sg.correct + ((second ? exact_apart : 0) + 2 * e));
            lpat[t] = col | exact << 16;
        }
        if (tid <= ER) lrow[tid] = has0 ? my_off - e0 : 0;
        else if (SWI && tid <= 2 * ER + 1) lrow[tid] = n0 + (has1 ? my_off - e1 : 0);
    }
};

// A thread's place in one row's slice of the list: the next entry, its column, and the entry behind it, which is read when the one before
// is taken (a wave that read the list when it came to an entry held the others up).
struct TileCursor {
    int at = 0, end = 0;
    uint32_t entry = 0, behind = 0;

    __device__ __forceinline__ void start(const uint32_t* lpat, const int* row, int k_begin)
    {
        int q = row[0];
        end = row[1];
        for (int hi = end; k_begin > 0 && q < hi;) {           // K split: the first entry of the slice
            const int half = (q + hi) >> 1;
            if ((int)(lpat[half] & 0xFFFFu) < k_begin) q = half + 1;
            else hi = half;
        }
        at = q;
        entry = lpat[q];                                       // (at most two past the list: the room behind it)
        behind = lpat[q + 1];
    }
    __device__ __forceinline__ int col() const { return at < end ? (int)(entry & 0xFFFFu) : NO_ESCAPE; }
    // the entries in front of column k_end: where(e) is where the weight of column first + e lies, null if it is another thread's
    template <class F>
    __device__ __forceinline__ void take(const uint32_t* lpat, int first, int k_end, F where)
    {
        while (col() < k_end) {
            if (uint8_t* const to = where((int)(entry & 0xFFFFu) - first)) *(uint16_t*)to = (uint16_t)(entry >> 16);
            entry = behind;
            behind = lpat[++at + 1];
        }
    }
};

// The sums of a multiplying wave: acc holds 32 FB batch rows from b0 + row0 on x 64 weight rows (SWI: 32 of gate and of up), mw the first of them.
// Overflow path only: the streamed value of an escape was its "wrong" decode, so acc[b, m] += (correct - wrong) * X[b, col], added by the K split that
// owns column 0.
template <int FB, bool SWI, class Job>
__device__ __forceinline__ void tile_overflow(const GemmParams& p, const Job& j, int esc_mode, int row0, int mw, t12_f32x16 (&acc)[FB][2])
{
    const int lane = threadIdx.x & 63, ln = lane & 31, lh = lane >> 5;
    const int b0 = j.b0 + row0;
    if (blockIdx.z == 0 && esc_mode == 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const T12Segment& g = SWI && u ? j.sg1 : j.sg;
            const int m = mw + (SWI ? 0 : 32 * u) + ln;
            if (m < j.M && g.row_off) {
                const int beg = g.row_off[m], end = g.row_off[m + 1];
                for (int q = beg; q < end; q++) {
                    const float delta = t12_bf16_to_f32((uint16_t)g.correct[q]) - t12_bf16_to_f32((uint16_t)g.wrong[q]);
                    const uint16_t* xc = j.act + g.cols[q];
                    int stride = j.act_stride, row = b0;
                    asm volatile("" : "+s"(stride), "+s"(row));          // (the rows' addresses are formed anew per entry: kept, they would not fit)
#pragma unroll
                    for (int i = 0; i < 2 * FB; i++) {
#pragma unroll
                        for (int r = 8 * (i & 1); r < 8 * (i & 1) + 8; r++)          // (rows past the end: the last one again, not stored)
                            acc[i / 2][u][r] += delta * t12_bf16_to_f32(xc[(size_t)min(row + 16 * i + 8 * ((r >> 2) & 1) + 4 * lh + (r & 3), j.B - 1) * stride]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
    }
}

// Stores the sums FIRST .. END - 1 of them, number 16 i + r register r of acc[i].  Register r of lane (ln, lh) is D[row = 8*(r/4) + 4*lh + r%4][col = ln]
// (row = batch, col = m).  A row's address is the wave's, the lanes add theirs: 64 addresses and conditions of a lane each would not fit its registers.
template <int FB, bool SWI, int EPI, int FIRST, int END, class Job>
__device__ __forceinline__ void tile_store(const GemmParams& p, const Job& j, int row0, int mw, const t12_f32x16 (&acc)[FB][2])
{
    const int lane = threadIdx.x & 63, ln = lane & 31, lh = lane >> 5;
    const int b0 = j.b0 + row0;
    const bool in0 = mw + ln < j.M, in1 = !SWI && mw + 32 + ln < j.M;
    constexpr bool HALF = SWI || EPI != T12_ACT_NONE;          // bf16 results of a function of the sums
    uint8_t* dst;
    size_t ld;
    if (HALF) {
        ld = p.out_bf16_ld;
        dst = (uint8_t*)(p.out_bf16 + (size_t)j.row_base * ld + mw);
    } else if (p.ksplit > 1) {
        ld = p.seg_ld[j.s];
        dst = (uint8_t*)(p.ws + (size_t)blockIdx.z * p.split_stride + p.seg_ws0[j.s] + mw);
    } else {
        ld = j.sg.out_stride;
        dst = (uint8_t*)(j.sg.out + (size_t)j.row_base * ld + mw);
    }
    constexpr int ES = HALF ? 2 : 4;
    const size_t lane_at = ((size_t)(4 * lh) * ld + ln) * ES;
#pragma unroll
    for (int n = FIRST; n < END; n++) {
        const int i = n >> 4, r = n & 15;
        const int b = b0 + 32 * i + 8 * (r >> 2) + (r & 3);                          // of the lanes' lower half
        uint8_t* const at = dst + (size_t)b * ld * ES + lane_at;
        if (b + 4 * lh < j.B) {
            if (SWI) {
                if (in0) *(uint16_t*)at = t12_f32_to_bf16(t12_apply_glu(acc[i][0][r], acc[i][1][r], p.glu));
            } else if (HALF) {
                if (in0) *(uint16_t*)at = t12_f32_to_bf16(t12_apply_act<EPI>(acc[i][0][r], p.act_a, p.act_b));
                if (in1) *(uint16_t*)(at + 64) = t12_f32_to_bf16(t12_apply_act<EPI>(acc[i][1][r], p.act_a, p.act_b));
            } else {
                if (in0) *(float*)at = acc[i][0][r];
                if (in1) *(float*)(at + 128) = acc[i][1][r];
            }
        }
    }
}

// The end of a tile of four multiplying and four copying waves, all eight there.  Each copying wave takes half of the sums of a multiplying one, through
// the LDS of the activations (lx, free by then): four waves alone neither hide a gated unit's operations (45 a pair; gated 28672 x 512 at B = 256 24.1 -> 20.2
// us) nor have enough stores in flight where a slice along K is short (us, plain sums: 2 x 8192 x 2048 at 200 rows 40.0 -> 39.2, 6144 x 4096 at 129 / 160 / 256
// 30.9 -> 29.9, 32.1 -> 31.0, 34.4 -> 33.4, 8320 x 2048 at 512 34.4 -> 33.2, 3072 x 2048 at 200 20.4 -> 19.6).  wave: 0 .. 3 of its kind.
template <int FB, bool SWI, int EPI, class Job>
__device__ __forceinline__ void tile_finish(const GemmParams& p, const Job& j, int esc_mode, int row0, int mw, int wave, uint8_t* lx, t12_f32x16 (&acc)[FB][2])
{
    constexpr int N = 16 * FB, KEEP = N / 2;
    tile_overflow<FB, SWI>(p, j, esc_mode, row0, mw, acc);
    tile_barrier();                                            // the copies have ended
    uint8_t* const to = lx + wave * (N / 2 * 512) + (threadIdx.x & 63) * 16;
#pragma unroll
    for (int n = KEEP; n < N; n += 4)
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const t12_f32x16& a = acc[n >> 4][u];
            *(t12_f32x4*)(to + ((n - KEEP) / 4 * 2 + u) * 1024) = t12_f32x4{a[n & 15], a[(n & 15) + 1], a[(n & 15) + 2], a[(n & 15) + 3]};
        }
    __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
    tile_barrier();
    tile_store<FB, SWI, EPI, 0, KEEP>(p, j, row0, mw, acc);
}
template <int FB, bool SWI, int EPI, class Job>
__device__ __forceinline__ void tile_finish_copying(const GemmParams& p, const Job& j, int row0, int mw, int wave, const uint8_t* lx)
{
    constexpr int N = 16 * FB, KEEP = N / 2;
    __builtin_amdgcn_s_waitcnt(ring_vmcnt(0));             // no copy outlives its workgroup or reaches into its next tile
    tile_barrier();
    tile_barrier();                                        // the sums are there
    t12_f32x16 acc[FB][2];
    const uint8_t* const at = lx + wave * (N / 2 * 512) + (threadIdx.x & 63) * 16;
#pragma unroll
    for (int n = KEEP; n < N; n += 4)
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const t12_f32x4 a = *(const t12_f32x4*)(at + ((n - KEEP) / 4 * 2 + u) * 1024);
#pragma unroll
            for (int q = 0; q < 4; q++) acc[n >> 4][u][(n & 15) + q] = a[q];
        }
    tile_store<FB, SWI, EPI, KEEP, N>(p, j, row0, mw, acc);
}

// ---------------------------------------------------------------------------
// 256 x 128.  LDS: activations of three stages, [256 rows][8 units of 16 bytes], unit u of row r in slot u ^ (r % 8) ^ (r / 8 % 2); decoded
// weights of two, [8 units][128 rows] of 16 bytes, rotated (lds_slot).  Step t of a stage takes columns 16 t .. 16 t + 15, the lanes of wave half h unit 2 t + h.
//
// Loads of the planes.  A stage is 64 bytes of a row's sm plane and 32 of its gr plane, half a line and a quarter; fetched a stage at a time HBM would be
// asked for every line twice or more (the rows of a tile are K bytes apart, a power of two: they fall into a handful of L2 sets and are evicted
// before the next stage comes back for the other half).  So a window of two stages is loaded at once, both halves of a line in neighbouring
// instructions; eight lanes take two rows, rr and 64 + (rr ^ 1), four lanes the 64 columns of either (rr ^ 1: the LDS writes of the two rows meet other banks).
// Returns false when the tile lies past the segment's rows (nothing was done).
// ---------------------------------------------------------------------------
struct TileLds {
    static constexpr int TB = 256;                 // batch rows of a tile
    static constexpr int X = TB * KC * 2;          // a stage's activations
    static constexpr int W = TM * KC * 2;          // a stage's decoded weights
};

template <bool SWI, int EPI, bool DEV>
__device__ __forceinline__ bool gemm_tile_body(const GemmParams& p, const int tile, const int bt, uint8_t* const lx, uint8_t* const lw,
                                               uint32_t* const lpat, int* const lrow)
{
    using L = TileLds;
    constexpr int FB = 4;
    constexpr int NXC = L::TB / 32;                   // activation copies of a stage per copying wave (8 rows of 128 bytes each)
    constexpr int NWL = 4;                            // plane loads of a window per thread
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31, lh = lane >> 5;
    const TileJob<TM, SWI, DEV> j(p, tile, bt, L::TB);
    if (j.b0 >= j.B) return false;                    // grouped launch: this segment has fewer batch tiles than the grid
    const int nstage = j.nstage, k_begin = j.k_begin;
    const TileList<TM, SWI, PCAP> list(j);

    // ---- this thread's share of the weights: 16 columns of a row per stage (SWI: the rows of a wave are all of one tensor)
    const int c8 = tid & 7, cc = c8 & 3, rr = tid >> 3;
    const int w_row = c8 >> 2 ? 64 + (rr ^ 1) : rr;            // local row
    const T12Segment& sw = SWI && wave >= 4 ? j.sg1 : j.sg;
    const size_t first = (size_t)j.m0 * j.K + k_begin;
    const auto s_buf = tile_buffer(sw.sm + first), g_buf = tile_buffer(sw.gr + (first >> 1));
    const uint32_t s_off = (uint32_t)(min(j.m0 + j.rel(w_row), j.M - 1) - j.m0) * (uint32_t)j.K + 16u * cc;
    const uint32_t be = __builtin_amdgcn_readfirstlane(sw.base_exp);
    const uint32_t be2 = t12_opaque((be << 7) | (be << 23));
    const int w_dst = lds_slot(2 * cc, w_row, TM) * 16;           // unit 2 cc; 2 cc + 1: ^ 16, and a unit on
    t12_u32x4 rs[2][2];                                        // [window slot][stage of the window]
    t12_u32x2 rg[2][2];
    // part q (0 .. 3) of a window's loads; past the end: the last stage again
    auto load_w = [&](int slot, int win, int q) __attribute__((always_inline)) {
        const int y = q & 1, st = min(2 * win + y, nstage - 1);
        if (q < 2) rs[slot][y] = __builtin_amdgcn_raw_buffer_load_b128(s_buf, s_off, st * KC, 0);
        else rg[slot][y] = __builtin_amdgcn_raw_buffer_load_b64(g_buf, s_off >> 1, st * (KC / 2), 0);
    };
    // part q (0 .. 4) of unit h (eight columns): a pair of weights each, the first with what they share, the last the store
    uint32_t w_lo = 0, w_hi = 0, w_[4];
    auto put = [&](uint8_t* to, int slot, int y, int h, int q) __attribute__((always_inline)) {
        const t12_u32x4 sv = rs[slot][y];
        const uint32_t gv = rg[slot][y][h];
        if (q == 0) {
            w_lo = gv & 0x0F0F0F0Fu;
            w_hi = (gv >> 4) & 0x0F0F0F0Fu;
        }
        if (q < 4) w_[q] = t12_decode2_seq(sv[2 * h], sv[2 * h + 1], w_lo, w_hi, be2, q);
        else *(uint4*)(to + (w_dst ^ (16 * h)) + h * (16 * TM)) = make_uint4(w_[0], w_[1], w_[2], w_[3]);
    };
    auto put_all = [&](uint8_t* to, int slot, int y) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int q = 0; q < 5; q++) put(to, slot, y, h, q);
    };
    TileCursor cursor;
    // the escapes among this thread's 16 weights of the stage from column k on (same wave: LDS keeps the order of the writes)
    auto patch = [&](uint8_t* to, int k) __attribute__((always_inline)) {
        if (list.mode == 1)
            cursor.take(lpat, k + 16 * cc, k + KC, [&](int e) { return (unsigned)e < 16u ? to + (w_dst ^ (16 * (e >> 3))) + (e >> 3) * (16 * TM) + (e & 7) * 2 : nullptr; });
    };
    auto start_cursor = [&]() __attribute__((always_inline)) {
        if (list.mode == 1) cursor.start(lpat, lrow + (SWI && wave >= 4 ? list.ER + 1 : 0) + j.rel(w_row), k_begin);
    };
#pragma unroll
    for (int q = 0; q < 4; q++) load_w(0, 0, q);
#pragma unroll
    for (int q = 0; q < 4; q++) load_w(1, 1, q);

    if (wave >= 4) {
        // ================= waves that copy the activations, and decode =================
        const int pw = wave - 4;
        const auto x_buf = tile_buffer(j.act + (size_t)j.b0 * j.act_stride + k_begin);
        uint32_t x_off[NXC];
#pragma unroll
        for (int c = 0; c < NXC; c++) {
            const int r = 8 * (4 * c + pw) + (lane >> 3);      // (rows past the end: the last one again, not stored)
            x_off[c] = 2u * ((uint32_t)(min(j.b0 + r, j.B - 1) - j.b0) * (uint32_t)j.act_stride + 8u * ((lane & 7) ^ (r & 7) ^ ((r >> 3) & 1)));
        }
        auto copy_x = [&](int at, int st) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < NXC; c++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(x_buf, (ring_lptr)(lx + at + (4 * c + pw) * 1024), 16, x_off[c], min(st, nstage - 1) * (2 * KC), 0, 0);
        };
        copy_x(0, 0);
        copy_x(L::X, 1);
        list.stage(j, lpat, lrow);
        __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
        tile_barrier();                                        // the list is there
        start_cursor();
        put_all(lw, 0, 0);
        patch(lw, k_begin);
        __builtin_amdgcn_s_waitcnt(ring_vmcnt(NXC) & TILE_LDS_DONE);
        tile_barrier();                                        // stage 0 is there
        // interval st: the copies of stage st + 2, this half of the weights of stage st + 1; ends when both parts of stage st + 1 are there
        int xat = 2 * L::X;
        // (the copies of stage st + 1 are older than those of stage st + 2 and, in the loop, than one window's loads; behind it no window is left to load)
        auto interval = [&](auto dc, int st, auto loop) __attribute__((always_inline)) {
            constexpr int d = decltype(dc)::value;             // st % 4
            copy_x(xat, st + 2);
            __builtin_amdgcn_sched_barrier(0);                 // (in this order: the wait below counts what is behind a copy)
            xat = xat == 2 * L::X ? 0 : xat + L::X;
            uint8_t* const to = lw + ((d + 1) & 1) * L::W;
            put_all(to, ((d + 1) >> 1) & 1, (d + 1) & 1);
            if (decltype(loop)::value && (d & 1) == 0) {
#pragma unroll
                for (int q = 0; q < 4; q++) load_w((d >> 1) & 1, (st >> 1) + 2, q);
            }
            patch(to, k_begin + (st + 1) * KC);
            __builtin_amdgcn_s_waitcnt(ring_vmcnt(NXC + (decltype(loop)::value ? NWL : 0)) & TILE_LDS_DONE);
            tile_barrier();
        };
        // (no way out of the loop but at its end: with one, the compiler would wait for everything in flight once per round)
        int st = 0;
        for (; st + 4 <= nstage; st += 4) {
            interval(std::integral_constant<int, 0>(), st, std::true_type());
            interval(std::integral_constant<int, 1>(), st + 1, std::true_type());
            interval(std::integral_constant<int, 2>(), st + 2, std::true_type());
            interval(std::integral_constant<int, 3>(), st + 3, std::true_type());
        }
        if (st < nstage) {
            interval(std::integral_constant<int, 0>(), st, std::false_type());
            if (st + 1 < nstage) {
                interval(std::integral_constant<int, 1>(), st + 1, std::false_type());
                if (st + 2 < nstage) interval(std::integral_constant<int, 2>(), st + 2, std::false_type());
            }
        }
        tile_keep(rs, rg);
        tile_finish_copying<FB, SWI, EPI>(p, j, ((wave - 4) >> 1) * (FB * 32), j.m0 + (wave & 1) * (SWI ? 32 : 64), wave - 4, lx);
        return true;
    }

    // ================= waves that multiply: 2 x 2, of 32 FB batch rows x 64 weight rows =================
    const int wb = wave >> 1, wm = wave & 1;
    list.stage(j, lpat, lrow);
    __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
    tile_barrier();
    start_cursor();
    put_all(lw, 0, 0);
    patch(lw, k_begin);
    const int xo0 = (wb * (FB * 32) + ln) * 128 + ((lh ^ (ln & 7) ^ ((ln >> 3) & 1)) << 4);          // step t: ^ (t << 5)
    const int wo0 = lds_slot(lh, wm * 64 + ln, TM) * 16;       // step t of a stage: ^ (t << 5), and 2 t units on
    t12_f32x16 acc[FB][2];
#pragma unroll
    for (int i = 0; i < FB; i++)
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][u][r] = 0.0f;
    t12_u32x4 A[2][FB], W[2][2];
    // fragment number f of step t: the order in which the products need them
    auto frag = [&](int xat, int wat, int t, int f, int xo0, int wo0) __attribute__((always_inline)) {
        if (f == 0) W[t & 1][0] = *(const t12_u32x4*)(lw + wat + (wo0 ^ (t << 5)) + t * (32 * TM));
        else if (f == 1) A[t & 1][0] = *(const t12_u32x4*)(lx + xat + (xo0 ^ (t << 5)));
        else if (f == 2) W[t & 1][1] = *(const t12_u32x4*)(lw + wat + (wo0 ^ (t << 5)) + t * (32 * TM) + 512);
        else A[t & 1][f - 2] = *(const t12_u32x4*)(lx + xat + (xo0 ^ (t << 5)) + 4096 * (f - 2));
    };
    // the products of step t; behind the first three the reads for the next step (of buffers xat, wat), behind the others the five parts of `work`
    auto step = [&](int t, int xat, int wat, auto work) __attribute__((always_inline)) {
        int xo = xo0, wo = wo0;
        asm volatile("" : "+v"(xo), "+v"(wo));               // (the addresses are formed anew in every step: kept, they would not fit)
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const int i = m >> 1, u = m & 1;
            acc[i][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(t12_bf16x8, A[t & 1][i]),
                                                                __builtin_bit_cast(t12_bf16x8, W[t & 1][u]), acc[i][u], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (m < 3) {
                frag(xat, wat, (t + 1) & 3, 2 * m, xo, wo);
                frag(xat, wat, (t + 1) & 3, 2 * m + 1, xo, wo);
            } else {
                work(m - 3);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
    tile_barrier();                                            // stage 0 is there
#pragma unroll
    for (int f = 0; f < FB + 2; f++) frag(0, 0, 0, f, xo0, wo0);
    int xat = 0;
    // Stage st, and this half of the weights of stage st + 1.  (Past the last stage: the last one again, read and not used.)
    auto stage = [&](auto dc, int st) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value;                 // st % 4
        constexpr int wat = (d & 1) * L::W, wnext = L::W - wat, slot = ((d + 1) >> 1) & 1, y = (d + 1) & 1;
        step(0, xat, wat, [&](int q) __attribute__((always_inline)) { put(lw + wnext, slot, y, 0, q); });
        step(1, xat, wat, [&](int q) __attribute__((always_inline)) { put(lw + wnext, slot, y, 1, q); });
        step(2, xat, wat, [&](int q) __attribute__((always_inline)) {
            if ((d & 1) == 0 && q < 4) load_w((d >> 1) & 1, (st >> 1) + 2, q);
        });
        patch(lw + wnext, k_begin + (st + 1) * KC);
        xat = xat == 2 * L::X ? 0 : xat + L::X;
        // this stage's operands are in registers: its buffers are free, and the next stage is there
        __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
        tile_barrier();
        step(3, xat, wnext, [&](int) __attribute__((always_inline)) {});
    };
    int st = 0;
    for (; st + 4 <= nstage; st += 4) {
        stage(std::integral_constant<int, 0>(), st);
        stage(std::integral_constant<int, 1>(), st + 1);
        stage(std::integral_constant<int, 2>(), st + 2);
        stage(std::integral_constant<int, 3>(), st + 3);
    }
    if (st < nstage) {
        stage(std::integral_constant<int, 0>(), st);
        if (st + 1 < nstage) {
            stage(std::integral_constant<int, 1>(), st + 1);
            if (st + 2 < nstage) stage(std::integral_constant<int, 2>(), st + 2);
        }
    }
    tile_finish<FB, SWI, EPI>(p, j, list.mode, wb * (FB * 32), j.m0 + wm * (SWI ? 32 : 64), wave, lx, acc);
    return true;
}

// Batch tiles: one per workgroup (blockIdx.y), except when the rows per group are known on the device only: such a launch has one workgroup per row
// tile, which takes the group's batch tiles one after the other (a group within the tile -- the usual case -- is streamed once, a larger one once
// per tile; no group's rows can fall outside the grid).
template <bool SWI = false, int EPI = T12_ACT_NONE, bool DEV = false>
__global__ __launch_bounds__(512) void gemm_tile_kernel(const GemmParams p)
{
    using L = TileLds;
    __shared__ __attribute__((aligned(16))) uint8_t lx[3 * L::X], lw[2 * L::W];
    __shared__ uint32_t lpat[PCAP + 4];
    __shared__ int lrow[TileList<TM, SWI, PCAP>::TABLE];
    int tile = blockIdx.x, bt = blockIdx.y;
    if (!DEV && gridDim.y > 1) tile_of_block(tile, bt);
    for (;; bt++) {
        if (!gemm_tile_body<SWI, EPI, DEV>(p, tile, bt, lx, lw, lpat, lrow) || !DEV) break;
        __syncthreads();                                   // the next tile reuses the staging buffers
    }
}

// ---------------------------------------------------------------------------
// 64 or 128 batch rows x 128 weight rows, two stages (a window of 128 columns) between barriers: with so few products per stage what a stage cost was the
// chain barrier - decode - LDS writes - barrier, about 1000 cycles, and not the 512 of its products.  Roles as in gemm_tile_body.  (Operands read two steps
// ahead of their products instead of one, in four sets of registers: level.)
// LDS: activations of NXB windows, two stages each laid out as above; decoded weights of two windows, [16 units][128 rows] of 16 bytes.
// ---------------------------------------------------------------------------
template <int FB>
struct StripLds {
    static constexpr int TB = 64 * FB;
    static constexpr int X = TB * KC * 2, XW = 2 * X;          // a stage's, a window's activations
    static constexpr int W = 2 * TM * KC * 2;                  // a window's decoded weights
    static constexpr int NXB = FB == 2 ? 2 : 3;
};

template <int FB, bool SWI, int EPI, bool DEV, bool FAR>
__device__ __forceinline__ bool gemm_strip_body(const GemmParams& p, const int tile, const int bt, uint8_t* const lx, uint8_t* const lw,
                                                uint32_t* const lpat, int* const lrow)
{
    using L = StripLds<FB>;
    constexpr int NXC = L::TB / 32;                   // activation copies of a stage per copying wave (8 rows of 128 bytes each)
    constexpr int NWL = 4, NXB = L::NXB, XEND = (NXB - 1) * L::XW;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31, lh = lane >> 5;
    const TileJob<TM, SWI, DEV> j(p, tile, bt, L::TB);
    if (j.b0 >= j.B) return false;                    // grouped launch: this segment has fewer batch tiles than the grid
    const int nstage = j.nstage, k_begin = j.k_begin, nwin = (nstage + 1) / 2;
    const TileList<TM, SWI, PCAP> list(j);

    // ---- this thread's share of the weights: 16 columns of a row per stage (SWI: the rows of a wave are all of one tensor)
    const int c8 = tid & 7, cc = c8 & 3, rr = tid >> 3;
    const int w_row = c8 >> 2 ? 64 + (rr ^ 1) : rr;            // local row
    const T12Segment& sw = SWI && wave >= 4 ? j.sg1 : j.sg;
    const size_t first = (size_t)j.m0 * j.K + k_begin;
    const auto s_buf = tile_buffer(sw.sm + first), g_buf = tile_buffer(sw.gr + (first >> 1));
    const int w_at = min(j.m0 + j.rel(w_row), j.M - 1) - j.m0;
    const uint32_t s_off = (uint32_t)w_at * (uint32_t)j.K + 16u * cc, g_off = s_off >> 1;
    const size_t far = first + (size_t)w_at * j.K + 16 * cc;
    const uint8_t *const s_far = sw.sm + far, *const g_far = sw.gr + (far >> 1);
    const uint32_t be = __builtin_amdgcn_readfirstlane(sw.base_exp);
    const uint32_t be2 = t12_opaque((be << 7) | (be << 23));
    const int w_dst = lds_slot(2 * cc, w_row, TM) * 16;           // unit 2 cc; 2 cc + 1: ^ 16, and a unit on
    t12_u32x4 rs[2][2];                                        // [window % 2][stage of the window]
    t12_u32x2 rg[2][2];
    // part q (0 .. 3) of a window's loads; past the end: the last stage again
    auto load_w = [&](int slot, int win, int q) __attribute__((always_inline)) {
        const int y = q & 1, st = min(2 * win + y, nstage - 1);
        if (FAR && q < 2) rs[slot][y] = global_load<t12_u32x4>(s_far + (size_t)st * KC);
        else if (FAR) rg[slot][y] = global_load<t12_u32x2>(g_far + (size_t)st * (KC / 2));
        else if (q < 2) rs[slot][y] = __builtin_amdgcn_raw_buffer_load_b128(s_buf, s_off, st * KC, 0);
        else rg[slot][y] = __builtin_amdgcn_raw_buffer_load_b64(g_buf, g_off, st * (KC / 2), 0);
    };
    // part q (0 .. 4) of unit u (eight columns of stage u / 2): a pair of weights each, the first with what they share, the last the store
    uint32_t w_lo = 0, w_hi = 0, w_[4];
    auto put = [&](uint8_t* to, int slot, int u, int q) __attribute__((always_inline)) {
        const int y = u >> 1, h = u & 1;
        const t12_u32x4 sv = rs[slot][y];
        const uint32_t gv = rg[slot][y][h];
        if (q == 0) {
            w_lo = gv & 0x0F0F0F0Fu;
            w_hi = (gv >> 4) & 0x0F0F0F0Fu;
        }
        if (q < 4) w_[q] = t12_decode2_seq(sv[2 * h], sv[2 * h + 1], w_lo, w_hi, be2, q);
        else *(uint4*)(to + (w_dst ^ (16 * h)) + h * (16 * TM) + y * (L::W / 2)) = make_uint4(w_[0], w_[1], w_[2], w_[3]);
    };
    auto put_all = [&](uint8_t* to, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int q = 0; q < 5; q++) put(to, slot, u, q);
    };
    TileCursor cursor;
    // the escapes among this thread's 2 x 16 weights of the window from column k on (same wave: LDS keeps the order of the writes)
    auto patch = [&](uint8_t* to, int k) __attribute__((always_inline)) {
        if (list.mode == 1)
            cursor.take(lpat, k, k + 2 * KC, [&](int e) -> uint8_t* {
                const int c = (e & (KC - 1)) - 16 * cc;        // 0 .. 15: one of this thread's
                return (unsigned)c < 16u ? to + (w_dst ^ (16 * (c >> 3))) + (c >> 3) * (16 * TM) + (e >> 6) * (L::W / 2) + (c & 7) * 2 : nullptr;
            });
    };
    auto start_cursor = [&]() __attribute__((always_inline)) {
        if (list.mode == 1) cursor.start(lpat, lrow + (SWI && wave >= 4 ? list.ER + 1 : 0) + j.rel(w_row), k_begin);
    };
#pragma unroll
    for (int q = 0; q < 4; q++) load_w(0, 0, q);

    if (wave >= 4) {
        // ================= waves that copy the activations, and decode =================
        const int pw = wave - 4;
        const auto x_buf = tile_buffer(j.act + (size_t)j.b0 * j.act_stride + k_begin);
        uint32_t x_off[NXC];
        const uint16_t* x_far[NXC];
#pragma unroll
        for (int c = 0; c < NXC; c++) {
            const int r = 8 * (4 * c + pw) + (lane >> 3);      // (rows past the end: the last one again, not stored)
            const int row = min(j.b0 + r, j.B - 1), unit = 8 * ((lane & 7) ^ (r & 7) ^ ((r >> 3) & 1));
            x_off[c] = 2u * ((uint32_t)(row - j.b0) * (uint32_t)j.act_stride + (uint32_t)unit);
            x_far[c] = j.act + (size_t)row * j.act_stride + k_begin + unit;
        }
        auto copy_x = [&](int at, int win) __attribute__((always_inline)) {
#pragma unroll
            for (int y = 0; y < 2; y++)
#pragma unroll
                for (int c = 0; c < NXC; c++) {
                    const ring_lptr to = (ring_lptr)(lx + at + y * L::X + (4 * c + pw) * 1024);
                    const int st = min(2 * win + y, nstage - 1);
                    if (FAR) __builtin_amdgcn_global_load_lds((ring_gptr)(uintptr_t)(x_far[c] + (size_t)st * KC), to, 16, 0, 0);
                    else __builtin_amdgcn_raw_ptr_buffer_load_lds(x_buf, to, 16, x_off[c], st * (2 * KC), 0, 0);
                }
            __builtin_amdgcn_sched_barrier(0);                 // (in this order: the waits below count what is behind a copy)
        };
#pragma unroll
        for (int w = 0; w < NXB - 1; w++) copy_x(w * L::XW, w);
#pragma unroll
        for (int q = 0; q < 4; q++) load_w(1, 1, q);
        list.stage(j, lpat, lrow);
        __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
        tile_barrier();                                        // the list is there
        start_cursor();
        put_all(lw, 0);
        patch(lw, k_begin);
        __builtin_amdgcn_s_waitcnt(ring_vmcnt((NXB - 2) * 2 * NXC) & TILE_LDS_DONE);
        tile_barrier();                                        // window 0 is there
#pragma unroll
        for (int q = 0; q < 4; q++) load_w(0, 2, q);
        __builtin_amdgcn_sched_barrier(0);
        // Interval w: the copies of window w + NXB - 1, this half of the weights of window w + 1; ends when both parts of window w + 1 are there: its copies
        // are older than those of NXB - 2 windows and, in the loop, than NXB - 1 windows' loads of planes (behind it no window is left to load).
        int xat = XEND;
        auto interval = [&](auto dc, int w, auto loop) __attribute__((always_inline)) {
            constexpr int d = decltype(dc)::value;             // w % 2
            copy_x(xat, w + NXB - 1);
            xat = xat == XEND ? 0 : xat + L::XW;
            uint8_t* const to = lw + (1 - d) * L::W;
            put_all(to, 1 - d);
            if (decltype(loop)::value) {
#pragma unroll
                for (int q = 0; q < 4; q++) load_w(1 - d, w + 3, q);
            }
            patch(to, k_begin + (w + 1) * 2 * KC);
            __builtin_amdgcn_s_waitcnt(ring_vmcnt((NXB - 2) * 2 * NXC + (decltype(loop)::value ? (NXB - 1) * NWL : 0)) & TILE_LDS_DONE);
            tile_barrier();
        };
        // (no way out of the loop but at its end: with one, the compiler would wait for everything in flight once per round)
        int w = 0;
        for (; w + 2 < nwin; w += 2) {
            interval(std::integral_constant<int, 0>(), w, std::true_type());
            interval(std::integral_constant<int, 1>(), w + 1, std::true_type());
        }
        interval(std::integral_constant<int, 0>(), w, std::false_type());
        if (w + 1 < nwin) interval(std::integral_constant<int, 1>(), w + 1, std::false_type());
        tile_keep(rs, rg);
        tile_finish_copying<FB, SWI, EPI>(p, j, ((wave - 4) >> 1) * (FB * 32), j.m0 + (wave & 1) * (SWI ? 32 : 64), wave - 4, lx);
        return true;
    }

    // ================= waves that multiply: 2 x 2, of 32 FB batch rows x 64 weight rows =================
    const int wb = wave >> 1, wm = wave & 1;
#pragma unroll
    for (int q = 0; q < 4; q++) load_w(1, 1, q);
    list.stage(j, lpat, lrow);
    __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
    tile_barrier();
    start_cursor();
    put_all(lw, 0);
    patch(lw, k_begin);
#pragma unroll
    for (int q = 0; q < 4; q++) load_w(0, 2, q);
    const int xo0 = (wb * (FB * 32) + ln) * 128 + ((lh ^ (ln & 7) ^ ((ln >> 3) & 1)) << 4);          // step t of a stage: ^ (t << 5)
    const int wo0 = lds_slot(lh, wm * 64 + ln, TM) * 16;       // step t of a stage: ^ (t << 5), and 2 t units on
    t12_f32x16 acc[FB][2];
#pragma unroll
    for (int i = 0; i < FB; i++)
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][u][r] = 0.0f;
    t12_u32x4 A[2][FB], W[2][2];
    // fragment number f of step t (0 .. 7) of a window: the order in which the products need them
    auto frag = [&](int xat, int wat, int t, int f) __attribute__((always_inline)) {
        const int r = t & 3, xs = xat + (t >> 2) * L::X, ws = wat + (t >> 2) * (L::W / 2);
        if (f == 0) W[t & 1][0] = *(const t12_u32x4*)(lw + ws + (wo0 ^ (r << 5)) + r * (32 * TM));
        else if (f == 1) A[t & 1][0] = *(const t12_u32x4*)(lx + xs + (xo0 ^ (r << 5)));
        else if (f == 2) W[t & 1][1] = *(const t12_u32x4*)(lw + ws + (wo0 ^ (r << 5)) + r * (32 * TM) + 512);
        else A[t & 1][f - 2] = *(const t12_u32x4*)(lx + xs + (xo0 ^ (r << 5)) + 4096 * (f - 2));
    };
    // the products of step t; behind the first ones the reads for step t + 1 (of buffers xat, wat), behind the others the five parts of `work`
    constexpr int NF = FB + 2, NM = 2 * FB, per = NM >= 4 ? 2 : 3, M0 = (NF + per - 1) / per;
    auto step = [&](int t, int xat, int wat, auto work) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const int i = m >> 1, u = m & 1;
            acc[i][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(t12_bf16x8, A[t & 1][i]),
                                                                __builtin_bit_cast(t12_bf16x8, W[t & 1][u]), acc[i][u], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int f = 0; f < NF; f++)
                if (f / per == m) frag(xat, wat, (t + 1) & 7, f);
#pragma unroll
            for (int q = 0; q < 5; q++)
                if (M0 + q * (NM - M0) / 5 == m) work(q);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
    tile_barrier();                                            // window 0 is there
#pragma unroll
    for (int f = 0; f < NF; f++) frag(0, 0, 0, f);
    int xat = 0;
    auto none = [](int) __attribute__((always_inline)) {};
    // Window w, and this half of the weights of window w + 1.  odd: the slice ends with this window's first stage.  (Past the last window: the last
    // stage again, read and not used.)
    auto window = [&](auto dc, int w, bool odd) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value, wat = d * L::W, wnext = L::W - wat;          // w % 2
        uint8_t* const to = lw + wnext;
        step(0, xat, wat, [&](int q) __attribute__((always_inline)) { put(to, 1 - d, 0, q); });
        step(1, xat, wat, [&](int q) __attribute__((always_inline)) { put(to, 1 - d, 1, q); });
        step(2, xat, wat, [&](int q) __attribute__((always_inline)) { put(to, 1 - d, 2, q); });
        step(3, xat, wat, [&](int q) __attribute__((always_inline)) { put(to, 1 - d, 3, q); });
        if (odd) {
            __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
            tile_barrier();
            return;
        }
        patch(to, k_begin + (w + 1) * 2 * KC);
        step(4, xat, wat, [&](int q) __attribute__((always_inline)) {
            if (q < 4) load_w(1 - d, w + 3, q);
        });
        step(5, xat, wat, none);
        step(6, xat, wat, none);
        xat = xat == XEND ? 0 : xat + L::XW;
        // this window's operands are in registers: its buffers are free, and the next window is there
        __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
        tile_barrier();
        step(7, xat, wnext, none);
    };
    int w = 0;
    for (; w + 2 < nwin; w += 2) {
        window(std::integral_constant<int, 0>(), w, false);
        window(std::integral_constant<int, 1>(), w + 1, false);
    }
    const bool odd = nstage & 1;
    if (w + 1 < nwin) {
        window(std::integral_constant<int, 0>(), w, false);
        window(std::integral_constant<int, 1>(), w + 1, odd);
    } else {
        window(std::integral_constant<int, 0>(), w, odd);
    }
    tile_finish<FB, SWI, EPI>(p, j, list.mode, wb * (FB * 32), j.m0 + wm * (SWI ? 32 : 64), wave, lx, acc);
    return true;
}

template <int FB, bool SWI = false, int EPI = T12_ACT_NONE, bool DEV = false, bool FAR = false>
__global__ __launch_bounds__(512) void gemm_strip_kernel(const GemmParams p)
{
    using L = StripLds<FB>;
    __shared__ __attribute__((aligned(16))) uint8_t lx[L::NXB * L::XW], lw[2 * L::W];
    __shared__ uint32_t lpat[PCAP + 4];
    __shared__ int lrow[TileList<TM, SWI, PCAP>::TABLE];
    int tile = blockIdx.x, bt = blockIdx.y;
    if (!DEV && gridDim.y > 1) tile_of_block(tile, bt);
    for (;; bt++) {
        if (!gemm_strip_body<FB, SWI, EPI, DEV, FAR>(p, tile, bt, lx, lw, lpat, lrow) || !DEV) break;
        __syncthreads();                                   // the next tile reuses the staging buffers
    }
}

// ---------------------------------------------------------------------------
// 256 x 256.  LDS: activations and decoded weights of two stages, laid out as above.  Everything is every wave's: the products of 128 batch rows x 64
// weight rows, an eighth of the copies, 16 columns of two rows of the weights (eight lanes: rows rr and 128 + (rr ^ 1), and 64 rows on).  A stage's planes
// are loaded by themselves, two stages ahead: there are no registers for a window, and what it would save is in L2 (the other half of a line
// follows within 1.6 us).
// ---------------------------------------------------------------------------
constexpr int WIDE = 256;                     // rows of a tile, either way
constexpr int WIDE_PCAP = 4096;               // escape entries held

template <bool SWI, int EPI>
__device__ __forceinline__ void gemm_wide_body(const GemmParams& p, const int tile, const int bt, uint8_t* const x0, uint8_t* const x1, uint8_t* const w0,
                                               uint8_t* const w1, uint32_t* const lpat, int* const lrow)
{
    constexpr int FB = 4;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 31, lh = lane >> 5;
    const TileJob<WIDE, SWI, false> j(p, tile, bt, WIDE);
    if (j.b0 >= j.B) return;
    const int nstage = j.nstage, k_begin = j.k_begin;
    const TileList<WIDE, SWI, WIDE_PCAP> list(j);

    // ---- this thread's share of the weights (SWI: the rows of a wave are all of one tensor)
    const int c8 = tid & 7, cc = c8 & 3;
    const int w_row = c8 >> 2 ? 128 + ((tid >> 3) ^ 1) : tid >> 3;          // local row of item 0; item 1: 64 rows on
    const bool second = SWI && wave >= 4;
    const T12Segment& sw = second ? j.sg1 : j.sg;
    const size_t first = (size_t)j.m0 * j.K + k_begin;
    const auto s_buf = tile_buffer(sw.sm + first), g_buf = tile_buffer(sw.gr + (first >> 1));
    uint32_t s_off[2];
#pragma unroll
    for (int i = 0; i < 2; i++) s_off[i] = (uint32_t)(min(j.m0 + j.rel(w_row + 64 * i), j.M - 1) - j.m0) * (uint32_t)j.K + 16u * cc;
    const uint32_t be = __builtin_amdgcn_readfirstlane(sw.base_exp);
    const uint32_t be2 = t12_opaque((be << 7) | (be << 23));
    const int w_dst = lds_slot(2 * cc, w_row, WIDE) * 16;           // unit 2 cc; 2 cc + 1: ^ 16, and a unit on
    t12_u32x4 rs[2][2];                                        // [stage % 2][item]
    t12_u32x2 rg[2][2];
    auto load_w = [&](int slot, int st, int i) __attribute__((always_inline)) {          // past the end: the last stage again
        st = min(st, nstage - 1);
        rs[slot][i] = __builtin_amdgcn_raw_buffer_load_b128(s_buf, s_off[i], st * KC, 0);
        rg[slot][i] = __builtin_amdgcn_raw_buffer_load_b64(g_buf, s_off[i] >> 1, st * (KC / 2), 0);
    };
    // part q (0 .. 4) of unit u (eight columns of item u / 2): a pair of weights each, the first with what they share, the last the store
    uint32_t w_lo = 0, w_hi = 0, w_[4];
    auto put = [&](uint8_t* to, int slot, int u, int q) __attribute__((always_inline)) {
        const int i = u >> 1, h = u & 1;
        const t12_u32x4 sv = rs[slot][i];
        const uint32_t gv = rg[slot][i][h];
        if (q == 0) {
            w_lo = gv & 0x0F0F0F0Fu;
            w_hi = (gv >> 4) & 0x0F0F0F0Fu;
        }
        if (q < 4) w_[q] = t12_decode2_seq(sv[2 * h], sv[2 * h + 1], w_lo, w_hi, be2, q);
        else *(uint4*)(to + (w_dst ^ (16 * h)) + h * (16 * WIDE) + 1024 * i) = make_uint4(w_[0], w_[1], w_[2], w_[3]);
    };
    TileCursor cursor[2];
    auto patch = [&](uint8_t* to, int k) __attribute__((always_inline)) {
        if (list.mode != 1 || !__any(min(cursor[0].col(), cursor[1].col()) < k + KC)) return;
#pragma unroll
        for (int i = 0; i < 2; i++)
            cursor[i].take(lpat, k + 16 * cc, k + KC, [&](int e) { return (unsigned)e < 16u ? to + (w_dst ^ (16 * (e >> 3))) + (e >> 3) * (16 * WIDE) + 1024 * i + (e & 7) * 2 : nullptr; });
    };
    const auto x_buf = tile_buffer(j.act + (size_t)j.b0 * j.act_stride + k_begin);
    uint32_t x_off[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int r = 8 * (8 * c + wave) + (lane >> 3);        // (rows past the end: the last one again, not stored)
        x_off[c] = 2u * ((uint32_t)(min(j.b0 + r, j.B - 1) - j.b0) * (uint32_t)j.act_stride + 8u * ((lane & 7) ^ (r & 7) ^ ((r >> 3) & 1)));
    }
    auto copy_x = [&](uint8_t* to, int st, int c) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x_buf, (ring_lptr)(to + (8 * c + wave) * 1024), 16, x_off[c], min(st, nstage - 1) * (2 * KC), 0, 0);
    };
    const int wb = wave >> 2, wm = wave & 3;
    const int xo0 = (wb * (FB * 32) + ln) * 128 + ((lh ^ (ln & 7) ^ ((ln >> 3) & 1)) << 4);          // step t: ^ (t << 5)
    const int wo0 = lds_slot(lh, wm * 64 + ln, WIDE) * 16;     // step t: ^ (t << 5), and 2 t units on

    load_w(0, 0, 0);
    load_w(0, 0, 1);
#pragma unroll
    for (int c = 0; c < 4; c++) copy_x(x0, 0, c);
    __builtin_amdgcn_sched_barrier(0);                         // (in this order: the waits below count what is behind a copy)
    list.stage(j, lpat, lrow);
    load_w(1, 1, 0);
    load_w(1, 1, 1);
    __builtin_amdgcn_s_waitcnt(TILE_LDS_DONE);
    tile_barrier();                                            // the list is there
    if (list.mode == 1) {
#pragma unroll
        for (int i = 0; i < 2; i++) cursor[i].start(lpat, lrow + (second ? list.ER + 1 : 0) + j.rel(w_row + 64 * i), k_begin);
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int q = 0; q < 5; q++) put(w0, 0, u, q);
    load_w(0, 2, 0);
    load_w(0, 2, 1);
    patch(w0, k_begin);
    copy_x(x1, 1, 0);
    copy_x(x1, 1, 1);
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int q = 0; q < 5; q++) put(w1, 1, u, q);
    t12_f32x16 acc[FB][2];
#pragma unroll
    for (int i = 0; i < FB; i++)
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][u][r] = 0.0f;
    t12_u32x4 A[2][FB], W[2][2];
    // fragment number f of step t: the order in which the products need them
    auto frag = [&](const uint8_t* xb, const uint8_t* wbuf, int t, int f) __attribute__((always_inline)) {
        if (f == 0) W[t & 1][0] = *(const t12_u32x4*)(wbuf + (wo0 ^ (t << 5)) + t * (32 * WIDE));
        else if (f == 1) A[t & 1][0] = *(const t12_u32x4*)(xb + (xo0 ^ (t << 5)));
        else if (f == 2) W[t & 1][1] = *(const t12_u32x4*)(wbuf + (wo0 ^ (t << 5)) + t * (32 * WIDE) + 512);
        else A[t & 1][f - 2] = *(const t12_u32x4*)(xb + (xo0 ^ (t << 5)) + 4096 * (f - 2));
    };
    // the products of step t; behind the first three the reads for the next step (of buffers xb, wbuf), behind the others the five parts of `work`
    auto step = [&](int t, const uint8_t* xb, const uint8_t* wbuf, auto work) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 8; m++) {
            const int i = m >> 1, u = m & 1;
            acc[i][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(t12_bf16x8, A[t & 1][i]),
                                                                __builtin_bit_cast(t12_bf16x8, W[t & 1][u]), acc[i][u], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (m < 3) {
                frag(xb, wbuf, (t + 1) & 3, 2 * m);
                frag(xb, wbuf, (t + 1) & 3, 2 * m + 1);
            } else {
                work(m - 3);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    __builtin_amdgcn_s_waitcnt(ring_vmcnt(10) & TILE_LDS_DONE);          // (behind the copies of stage 0: planes of stages 1 and 2, two copies of stage 1)
    tile_barrier();                                            // stage 0 is there
#pragma unroll
    for (int f = 0; f < FB + 2; f++) frag(x0, w0, 0, f);
    // Stage st; half the weights and half the copies of stage st + 1 are done; these of stage st + 2 go into its own buffers once everybody has its
    // operands in registers.  The escapes of stage st + 1 are put in before the third step, not before the barrier: then its products cover a
    // wave that has some.  (Past the last stage: the last one again, read and not used; behind the loop no planes are left to load.)
    auto stage = [&](auto dc, int st, auto loop) __attribute__((always_inline)) {
        constexpr int d = decltype(dc)::value;                 // st % 2
        uint8_t* const xb = d ? x1 : x0;
        uint8_t* const xn = d ? x0 : x1;
        uint8_t* const wbuf = d ? w1 : w0;
        uint8_t* const wn = d ? w0 : w1;
        step(0, xb, wbuf, [&](int q) __attribute__((always_inline)) {
            put(wn, 1 - d, 2, q);
            if (q == 0 || q == 2) copy_x(xn, st + 1, 2 + q / 2);
        });
        step(1, xb, wbuf, [&](int q) __attribute__((always_inline)) { put(wn, 1 - d, 3, q); });
        patch(wn, k_begin + (st + 1) * KC);
        step(2, xb, wbuf, [&](int q) __attribute__((always_inline)) {
            if (decltype(loop)::value && (q == 0 || q == 2)) load_w(1 - d, st + 3, q / 2);
        });
        // this stage's operands are in registers: its buffers are free; the next stage is there (behind its copies: four loads of planes)
        __builtin_amdgcn_s_waitcnt(ring_vmcnt(4) & TILE_LDS_DONE);
        tile_barrier();
        step(3, xn, wn, [&](int q) __attribute__((always_inline)) {
#pragma unroll
            for (int part = 2 * q; part < 2 * q + 2; part++) put(wbuf, d, part / 5, part % 5);
            if (q == 1 || q == 3) copy_x(xb, st + 2, q / 2);
        });
    };
    int st = 0;
    for (; st + 2 <= nstage; st += 2) {
        stage(std::integral_constant<int, 0>(), st, std::true_type());
        stage(std::integral_constant<int, 1>(), st + 1, std::true_type());
    }
    if (st < nstage) stage(std::integral_constant<int, 0>(), st, std::false_type());
    tile_keep(rs, rg);
    __builtin_amdgcn_s_waitcnt(ring_vmcnt(0));                 // no copy outlives its workgroup
    tile_overflow<FB, SWI>(p, j, list.mode, wb * (FB * 32), j.m0 + wm * (SWI ? 32 : 64), acc);
    tile_store<FB, SWI, EPI, 0, 16 * FB>(p, j, wb * (FB * 32), j.m0 + wm * (SWI ? 32 : 64), acc);
}

template <bool SWI = false, int EPI = T12_ACT_NONE>
__global__ __launch_bounds__(512) void gemm_wide_kernel(const GemmParams p)
{
    __shared__ __attribute__((aligned(16))) uint8_t x0[WIDE * KC * 2], x1[WIDE * KC * 2], w0[WIDE * KC * 2], w1[WIDE * KC * 2];
    __shared__ uint32_t lpat[WIDE_PCAP + 4];
    __shared__ int lrow[TileList<WIDE, SWI, WIDE_PCAP>::TABLE];
    int tile = blockIdx.x, bt = blockIdx.y;
    if (gridDim.y > 1) tile_of_block(tile, bt);
    gemm_wide_body<SWI, EPI>(p, tile, bt, x0, x1, w0, w1, lpat, lrow);
}

}  // namespace
