// Split-12 fused decode + GEMM on CDNA4 matrix cores (gfx950).
//
//   out_s[b*out_stride + m] = sum_k dec(W_s[m,k]) * X[b*act_stride + k]
//
// the function of the reference's split12_fused_gemm V1/V2/V3
// (split12_gemm.cuh:99-288, split12_gemm_v2.cuh:86-240, split12_gemm_v3.cuh:111-253)
// plus nv_apply_patches_batch (nvidia_kernels.cu:295-319), re-designed for
// wave64 MFMA instead of warp-level mma.sync:
//
//   * More than 64 rows: tiles of 128 or 256 weight rows x up to 256 batch rows (gemm_tile.h).  3 .. 64 rows, where the weight stream is the
//     bound, have a kernel of their own (gemm_ring.h) and, on short or few rows, the whole-row sweep.
//   * Up to 256 batch rows live in one workgroup: every weight byte is fetched once per launch (the reference re-decodes per
//     batch tile, nvidia_kernels.cu:456).
//   * Few row tiles (small M) are split along K across workgroups; the partial
//     sums go to a workspace and a second kernel adds them in a fixed order
//     (deterministic) -- or the caller's next kernel does (t12_gemm_deferred).
//   * Escapes are EXACT and cost no extra pass: the (column, exact bf16) pairs of a workgroup's rows -- one contiguous slice of
//     the CSR list -- are staged in LDS once, and the exact values take the places of the decoded ones.
//
// Fast path requirements: K % 64 == 0, 0 <= base_exp <= 240, 16-byte aligned
// activation rows.  Everything else goes to the general kernel below.

#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

#include "t12_act.h"
#include "t12_device.h"
#include "t12_host.h"
#include "dense16_plan.h"
#include "gemm_params.h"
#include "gemm_ring.h"
#include "gemm_tile.h"
#include "ring_plan.h"

// library-internal (hidden: not part of the ABI)
extern "C" __attribute__((visibility("hidden"))) void t12_glue_release_stream(hipStream_t st);      // glue.hip
extern "C" __attribute__((visibility("hidden"))) void t12_sampler_release_stream(hipStream_t st);   // engine/sampler.cpp

namespace {

// ---------------------------------------------------------------------------
// K-split reduction: out[b, m] = sum over splits z of the partial sums of (b, m), in ascending z
// (a fixed order: the result does not depend on which workgroup finished first).
// Grid: (blocks of 256 rows of the launch, largest batch).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const GemmParams p)
{
    const int col = blockIdx.x * 256 + threadIdx.x;
    const int b = blockIdx.y;
    if (col >= p.m_total) return;
    int s = 0;
#pragma unroll
    for (int i = 1; i < GMAX; i++)
        if (i < p.nseg && col >= p.seg_row0[i]) s = i;
    if (b >= p.seg_B[s]) return;
    const int m = col - p.seg_row0[s];
    const float* src = p.ws + p.seg_ws0[s] + (size_t)b * p.seg_ld[s] + m;
    float v = 0.0f;
    for (int z = 0; z < p.ksplit; z++) v += src[(size_t)z * p.split_stride];
    const T12Segment& sg = p.seg[s];
    sg.out[(size_t)b * sg.out_stride + m] = v;
}

// The same sums four rows at a time (16-byte loads and stores): thread = rows 4 c .. 4 c + 3 of one batch row.
// Used when every segment's row count, first row, output stride and pointers are multiples of four floats.
__global__ __launch_bounds__(256) void gemm_reduce4_kernel(const GemmParams p)
{
    const int col = (blockIdx.x * 256 + threadIdx.x) * 4;
    const int b = blockIdx.y;
    if (col >= p.m_total) return;
    int s = 0;
#pragma unroll
    for (int i = 1; i < GMAX; i++)
        if (i < p.nseg && col >= p.seg_row0[i]) s = i;
    if (b >= p.seg_B[s]) return;
    const int m = col - p.seg_row0[s];
    const float* src = p.ws + p.seg_ws0[s] + (size_t)b * p.seg_ld[s] + m;
    t12_f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int z = 0; z < p.ksplit; z++) v += *(const t12_f32x4*)(src + (size_t)z * p.split_stride);
    const T12Segment& sg = p.seg[s];
    *(t12_f32x4*)(sg.out + (size_t)b * sg.out_stride + m) = v;
}

// Adds up the partial sums of a K-split launch described by p into the segments' outputs.
void launch_reduce(const GemmParams& p, int max_b, hipStream_t st)
{
    bool vec = p.split_stride % 4 == 0 && (uintptr_t)p.ws % 16 == 0;
    for (int i = 0; i < p.nseg; i++) {
        const T12Segment& g = p.seg[i];
        if (g.M % 4 || p.seg_row0[i] % 4 || p.seg_ws0[i] % 4 || p.seg_ld[i] % 4 || g.out_stride % 4 || (uintptr_t)g.out % 16) vec = false;
    }
    if (vec)
        hipLaunchKernelGGL(gemm_reduce4_kernel, dim3((p.m_total / 4 + 255) / 256, max_b), dim3(256), 0, st, p);
    else
        hipLaunchKernelGGL(gemm_reduce_kernel, dim3((p.m_total + 255) / 256, max_b), dim3(256), 0, st, p);
}

// ---------------------------------------------------------------------------
// General path: any K, any base_exp, any alignment.  One wave per (row, 8
// batch rows); scalar decode rule; escapes exact from the CSR list.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void gemm_general_kernel(const GemmParams p)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int tile = blockIdx.x;            // blk_start counts 4-row blocks
    const int s = find_segment(p, tile);
    const T12Segment& sg = p.seg[s];
    const int row = (tile - p.blk_start[s]) * 4 + wave;
    if (row >= sg.M) return;
    const int b0 = blockIdx.y * 8;
    const int nb = min(8, p.B - b0);
    const int K = p.K;
    const size_t base = (size_t)row * K;
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int k = lane; k < K; k += T12_WAVE) {
        const size_t i = base + k;
        const uint32_t g = (sg.gr[i >> 1] >> (4 * (i & 1))) & 0xFu;
        if (g == 0 && sg.row_off) continue;            // taken from the list below
        const float w = t12_bf16_to_f32(t12_decode_scalar(sg.sm[i], g, sg.base_exp));
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (j < nb) acc[j] += w * t12_bf16_to_f32(p.act[(size_t)(b0 + j) * p.act_stride + k]);
    }
    if (sg.row_off) {
        const int beg = sg.row_off[row], end = sg.row_off[row + 1];
        for (int q = beg + lane; q < end; q += T12_WAVE) {
            const float w = t12_bf16_to_f32((uint16_t)sg.correct[q]);
            const int k = sg.cols[q];
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (j < nb) acc[j] += w * t12_bf16_to_f32(p.act[(size_t)(b0 + j) * p.act_stride + k]);
        }
    }
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float v = t12_wave_sum(acc[j]);
        if (lane == 0 && j < nb) sg.out[(size_t)(b0 + j) * sg.out_stride + row] = v;
    }
}

// ---------------------------------------------------------------------------
// Small batches (B <= 16): the dense-sweep kernel.  At these sizes the product is bound by the weight stream, and
// what the memory system streams fastest is what the B = 1 kernel gives it: workgroups in launch order, each
// sweeping a few whole rows quickly, so that the chip as a whole reads one dense window of the planes.  (Kernels
// whose waves walk many rows slowly in parallel -- a K-split grid of 128-row tiles, a wave per 16 rows -- measure
// 3.5-4.5 TB/s on the same bytes.)
//   * a workgroup owns 16 consecutive weight rows and all of K; its NW waves take the 128-column blocks of the rows
//     in turn (wave w: blocks w, w + NW, ...), so the workgroup as a whole reads its rows' planes front to back;
//   * v_mfma_f32_16x16x32_bf16, activations = A operand (rows = batch), weights = B operand: lane (n, g) =
//     (lane % 16, lane / 16) holds row n, so the planes go straight from HBM into the operand registers -- per
//     block a lane loads 2 x 16 bytes of sign/mantissa (columns 32g .. 32g+15 and 32g+16 .. 32g+31: the four lanes
//     of a row cover its 128-byte line in two back-to-back instructions) and 16 bytes of nibbles, rebuilds them
//     with t12_decode8 and feeds four MFMAs;
//   * the activations are not shared between waves: lane (b, g) takes the 8 columns an MFMA needs (they are
//     B x K bf16, resident in L2) and pairs them in registers to match t12_decode8's order;
//   * with one row group or two batch tiles the loads are turned through LDS on their way to these lanes (NX below);
//   * no barrier until the end, where the waves' partial 16 x 16 tiles are added through LDS in wave order;
//   * escapes: the streamed value of a group-0 weight is its "wrong" value; wave w adds (correct - wrong) * x[b, col]
//     for the entries w, w + NW, ... of each row (the four lanes of a row each for their four batch rows).
// Requires K % 128 == 0, 0 <= base_exp <= 240, B <= 16 NBT (NBT batch tiles of 16 rows share every weight load and
// decode; accumulators, activation registers and the reduction buffer grow with NBT).  blk_start counts the workgroups
// (16 RG rows each) per segment.
// Rows per group known on the device only (dev_counts, the experts of a mixture-of-experts layer at a few tokens):
// the segment's group has dev_counts[g] batch rows starting dev_base[g] rows into the activations and the outputs; a
// workgroup of a group without rows exits at once, one of a group above 16 rows sweeps its weight rows once per 16.
// ---------------------------------------------------------------------------
// SWI (a launch of ONE gate / up pair, segments 0 and 1 of equal row count): the first RG / 2 row groups of a workgroup
// are 16 RG / 2 rows of gate, the others the same rows of up, and the thread that finishes an element of both stores
// bf16( silu(gate) * up ) to out_bf16 instead of the two sums (the arithmetic of silu_mul_kernel, so the result is
// what t12_gemm + launch_silu_mul_bf16_batch give, bit for bit).
// NX > 0 (at most 4 NX batch rows per batch tile): neighbouring lanes load neighbouring bytes, and the operands' lanes get theirs by way of LDS, a buffer of
// D16_TURN bytes per wave at `turn` (rows of 144, 80 and 272 bytes: sixteen lanes reading 16 bytes of sixteen rows meet no bank twice).
// Loaded as the operands lie, sixteen lanes touch sixteen rows: 64 cache lines per load instruction, 448 per block against 48 .. 64, and a
// CU's cache looks up one per clock.  us per call, as the operands lie -> turned: 4096 x 14336 at 4 / 8 / 16 rows 20.7 / 23.4 / 23.0 -> 18.5 / 19.9 / 23.1,
// 2048 x 8192 at 8 13.6 -> 11.0, 4096 x 4096 at 16 / 24 / 32 10.2 / 13.1 / 14.4 -> 9.2 / 11.0 / 11.3, 4096 x 2048 at 24 10.5 -> 7.7; many rows are level
// (28672 x 4096 at 4: 34).  Three to six blocks ahead instead of two are no faster (19.9 -> 20.5 .. 21.3), nor are sixteen waves.  Row
// counts known on the device only keep the other form: level within 0.5 % (experts of 1 .. 6 rows stream at the rate of memory).
constexpr int D16_SM = 144, D16_GR = 80, D16_ACT = 272;
constexpr int d16_turn_bytes(int nx) { return 16 * (D16_SM + D16_GR) + 4 * nx * D16_ACT; }
template <int NW, int D, int RG, bool DEV, int NBT = 1, bool SWI = false, int NX = 0>
__device__ __forceinline__ void gemm_dense16_body(const GemmParams& p, t12_f32x4 (*red)[NW][64], uint8_t* turn = nullptr)
{
    static_assert(NX == 0 || (!SWI && !DEV && (NBT == 1 || NX == 4)), "no turned form");
    constexpr bool TURN = NX > 0;
    static_assert(!SWI || (RG % 2 == 0 && !DEV && NBT == 1), "the SwiGLU form pairs row groups");
    constexpr int RH = SWI ? RG / 2 : RG;             // row groups of one tensor
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, g = lane >> 4;

    const int blk = blockIdx.x;
    const int s = SWI ? 0 : find_segment(p, blk);
    const T12Segment& sg = p.seg[s];
    const int M = sg.M, K = p.K;
    // DEV: the group's rows from the device tables; otherwise one pass over the launch's B <= 16 rows
    const int b_all = DEV ? p.dev_counts[p.group_of_seg[s]] : 1;
    const int row_base = DEV ? p.dev_base[p.group_of_seg[s]] : 0;
    for (int b_first = 0; b_first < b_all; b_first += 16 * NBT) {
    const int B = DEV ? min(16 * NBT, b_all - b_first) : p.B;
    const uint16_t* const act = DEV ? p.act + (size_t)(row_base + b_first) * p.act_stride : p.act;
    float* const outp = DEV ? sg.out + (size_t)(row_base + b_first) * sg.out_stride : sg.out;
    const int m0 = (blk - p.blk_start[s]) * (16 * RH);               // RG groups of 16 rows share every activation load
    const int nblk = K >> 7;                          // 128-column blocks per row
    const int mine = nblk > wave ? (nblk - wave + NW - 1) / NW : 0;      // blocks of this wave
    // A wave without a block (K < NW * 128) still issues the first D fetches below and drops them: it aims them at
    // block 0, because its own first block would lie past the end of the row -- and, in the last rows of a plane or
    // of the activations, past the end of the allocation.
    const int wblk = mine > 0 ? wave : 0;
    uint32_t be2r[RG];
#pragma unroll
    for (int rg = 0; rg < RG; rg++) {
        const int be = p.seg[SWI && rg >= RH ? 1 : s].base_exp;
        be2r[rg] = t12_opaque(((uint32_t)be << 7) | ((uint32_t)be << 23));
    }

    // CSR pointers of this lane's rows (used after the stream)
    int e_beg[RG], e_end[RG];
    const uint8_t* smp[RG];
    const uint8_t* grp[RG];
    const uint8_t* smp8[RG];                          // TURN: rows 8 .. 15
#pragma unroll
    for (int rg = 0; rg < RG; rg++) {
        const T12Segment& sr = p.seg[SWI && rg >= RH ? 1 : s];      // (SWI: gate for the first half, up for the second)
        const int row = m0 + 16 * (rg % RH) + n;
        e_beg[rg] = e_end[rg] = 0;
        if (sr.row_off && row < M) {
            e_beg[rg] = sr.row_off[row];
            e_end[rg] = sr.row_off[row + 1];
        }
        const size_t e0 = (size_t)min(row, M - 1) * K;              // rows past the end are clamped, never stored
        smp[rg] = sr.sm + e0 + 32 * g + (size_t)wblk * 128;
        grp[rg] = sr.gr + (e0 >> 1) + 16 * g + (size_t)wblk * 64;
        if (TURN) {
            smp[rg] = sr.sm + (size_t)min(m0 + 16 * rg + (lane >> 3), M - 1) * K + 16 * (lane & 7) + (size_t)wblk * 128;
            smp8[rg] = sr.sm + (size_t)min(m0 + 16 * rg + 8 + (lane >> 3), M - 1) * K + 16 * (lane & 7) + (size_t)wblk * 128;
            grp[rg] = sr.gr + ((size_t)min(m0 + 16 * rg + (lane >> 2), M - 1) * K >> 1) + 16 * (lane & 3) + (size_t)wblk * 64;
        }
    }
    constexpr int NXP = TURN ? NX * NBT : NBT;
    const uint16_t* xp[NXP];                          // NBT tiles of 16 batch rows share every weight load and decode
#pragma unroll
    for (int t = 0; t < NXP; t++)
        xp[t] = TURN ? act + (size_t)min(4 * t + g, B - 1) * p.act_stride + 8 * n + (size_t)wblk * 128
                     : act + (size_t)min(16 * t + n, B - 1) * p.act_stride + 32 * g + (size_t)wblk * 128;
    // (copied on to LDS as they are, members of uint4 arrays end up in scratch; native vectors stay in registers)
    using Piece = std::conditional_t<TURN, t12_u32x4, uint4>;
    Piece rS[D][RG][2], rG[D][RG], rX[D][NXP][TURN ? 1 : 4];
#define T12_DS_FETCH(slot, j)                                                              \
    {                                                                                      \
        _Pragma("unroll") for (int t = 0; t < NXP; t++)                                    \
            _Pragma("unroll") for (int q = 0; q < (TURN ? 1 : 4); q++)                     \
                rX[slot][t][q] = *(const Piece*)(xp[t] + (size_t)(j) * (NW * 128) + 8 * q); \
        _Pragma("unroll") for (int rg = 0; rg < RG; rg++) {                                \
            rS[slot][rg][0] = *(const Piece*)(smp[rg] + (size_t)(j) * (NW * 128));         \
            rS[slot][rg][1] = *(const Piece*)((TURN ? smp8[rg] : smp[rg] + 16) + (size_t)(j) * (NW * 128)); \
            rG[slot][rg] = *(const Piece*)(grp[rg] + (size_t)(j) * (NW * 64));             \
        }                                                                                  \
    }
#pragma unroll
    for (int d = 0; d < D; d++) {
        T12_DS_FETCH(d, min(d, max(mine - 1, 0)))     // (fewer blocks than slots: the last one again, in bounds)
        __builtin_amdgcn_sched_barrier(0);
    }

    // the first escape entries of the rows: wave w takes entry e_beg + w, requested now and used after the stream
    int pcol[RG], pcorrect[RG], pwrong[RG];
#pragma unroll
    for (int rg = 0; rg < RG; rg++) {
        pcol[rg] = -1;
        pcorrect[rg] = pwrong[rg] = 0;
        if (e_beg[rg] + wave < e_end[rg]) {
            const T12Segment& sr = p.seg[SWI && rg >= RH ? 1 : s];
            pcol[rg] = sr.cols[e_beg[rg] + wave];
            pcorrect[rg] = sr.correct[e_beg[rg] + wave];
            pwrong[rg] = sr.wrong[e_beg[rg] + wave];
        }
    }

    t12_f32x4 acc[NBT][RG];
#pragma unroll
    for (int t = 0; t < NBT; t++)
#pragma unroll
        for (int rg = 0; rg < RG; rg++) acc[t][rg] = t12_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // TURN: a slot's loads -> the wave's buffer -> the operands' lanes (a wave's LDS accesses keep their order: no wait between them)
    uint8_t* const sm_ = TURN ? turn + wave * d16_turn_bytes(NX) : nullptr;
    uint8_t* const gr_ = sm_ + 16 * D16_SM;
    uint8_t* const act_ = gr_ + 16 * D16_GR;
#define T12_DS_TURN(slot)                                                                                    \
    _Pragma("unroll") for (int rg = 0; rg < RG; rg++) {                                                      \
        *(Piece*)(sm_ + (lane >> 3) * D16_SM + (lane & 7) * 16) = rS[slot][rg][0];                           \
        *(Piece*)(sm_ + (8 + (lane >> 3)) * D16_SM + (lane & 7) * 16) = rS[slot][rg][1];                     \
        *(Piece*)(gr_ + (lane >> 2) * D16_GR + (lane & 3) * 16) = rG[slot][rg];                              \
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");                                               \
        _Pragma("unroll") for (int h = 0; h < 2; h++) oS[rg][h] = *(const Piece*)(sm_ + n * D16_SM + g * 32 + h * 16); \
        oG[rg] = *(const Piece*)(gr_ + n * D16_GR + g * 16);                                                 \
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");                                               \
    }                                                                                                        \
    _Pragma("unroll") for (int t = 0; t < NBT; t++) {                                                        \
        _Pragma("unroll") for (int i = 0; i < NXP / NBT; i++)                                                \
            *(Piece*)(act_ + (4 * i + g) * D16_ACT + n * 16) = rX[slot][t * (NXP / NBT) + i][0];             \
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");                                               \
        _Pragma("unroll") for (int q = 0; q < 4; q++)                                                        \
            oX[t][q] = *(const Piece*)(act_ + min(n, 4 * (NXP / NBT) - 1) * D16_ACT + g * 64 + q * 16);      \
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");                                               \
    }
#define T12_DS_CONSUME(slot)                                                                                 \
    Piece oS[RG][2], oG[RG], oX[NBT][4];                                                                     \
    if constexpr (TURN) { T12_DS_TURN(slot) }                                                                \
    _Pragma("unroll") for (int q = 0; q < 4; q++) {                                                          \
        uint4 xa[NBT];                                                                                       \
        _Pragma("unroll") for (int t = 0; t < NBT; t++) xa[t] = t12_pair_acts(__builtin_bit_cast(uint4, TURN ? oX[t][q] : rX[slot][t][TURN ? 0 : q])); \
        _Pragma("unroll") for (int rg = 0; rg < RG; rg++) {                                                  \
            const Piece sv = TURN ? oS[rg][q >> 1] : rS[slot][rg][q >> 1];                                       \
            const Piece gv = TURN ? oG[rg] : rG[slot][rg];                                                       \
            const uint32_t gq = q == 0 ? gv.x : (q == 1 ? gv.y : (q == 2 ? gv.z : gv.w));                    \
            uint32_t w_[4];                                                                                  \
            if (q & 1) t12_decode8(sv.z, sv.w, gq, be2r[rg], w_);                                            \
            else t12_decode8(sv.x, sv.y, gq, be2r[rg], w_);                                                  \
            const uint4 wv = make_uint4(w_[0], w_[1], w_[2], w_[3]);                                         \
            _Pragma("unroll") for (int t = 0; t < NBT; t++)                                                  \
                acc[t][rg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(t12_bf16x8, xa[t]),  \
                                                                     __builtin_bit_cast(t12_bf16x8, wv), acc[t][rg], 0, 0, 0); \
        }                                                                                                    \
    }
    int j = 0;
    for (; j + 2 * D <= mine; j += D) {               // every slot is refilled
#pragma unroll
        for (int d = 0; d < D; d++) {
            T12_DS_CONSUME(d)
            T12_DS_FETCH(d, j + d + D)
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (; j < mine; j += D) {                        // the last (up to 2D - 1) blocks
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (j + d < mine) {
                T12_DS_CONSUME(d)
                if (j + d + D < mine) T12_DS_FETCH(d, j + d + D)
            }
        }
    }
#undef T12_DS_FETCH
#undef T12_DS_CONSUME
#undef T12_DS_TURN

    // ---- escapes.  Accumulator register r of lane (n, g) in batch tile t is D[batch 16t + 4g + r][row n].
    {
        const uint16_t* xrow[NBT][4];
#pragma unroll
        for (int t = 0; t < NBT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) xrow[t][r] = act + (size_t)min(16 * t + 4 * g + r, B - 1) * p.act_stride;
#pragma unroll
        for (int rg = 0; rg < RG; rg++) {
            if (pcol[rg] >= 0) {
                const float delta = t12_bf16_to_f32((uint16_t)pcorrect[rg]) - t12_bf16_to_f32((uint16_t)pwrong[rg]);
#pragma unroll
                for (int t = 0; t < NBT; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[t][rg][r] += delta * t12_bf16_to_f32(xrow[t][r][pcol[rg]]);
            }
            const T12Segment& sr = p.seg[SWI && rg >= RH ? 1 : s];
            for (int e = e_beg[rg] + wave + NW; e < e_end[rg]; e += NW) {        // rows with more than NW escapes
                const int col = sr.cols[e];
                const float delta = t12_bf16_to_f32((uint16_t)sr.correct[e]) - t12_bf16_to_f32((uint16_t)sr.wrong[e]);
#pragma unroll
                for (int t = 0; t < NBT; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[t][rg][r] += delta * t12_bf16_to_f32(xrow[t][r][col]);
            }
        }
    }

    if (TURN) __syncthreads();                        // (the reduction takes the other waves' buffers over)
    // ---- the waves' partial tiles, added in wave order; thread (r, l) = (tid / 64, tid % 64) of the first four waves
    //      finishes element D[batch 16 t + 4 (l / 16) + r][row l % 16] of every batch tile and row group
#pragma unroll
    for (int t = 0; t < NBT; t++)
#pragma unroll
        for (int rg = 0; rg < RG; rg++) red[t * RG + rg][wave][lane] = acc[t][rg];
    __syncthreads();
    if (tid < 256) {
        const int r = tid >> 6, l = tid & 63;
#pragma unroll
        for (int t = 0; t < NBT; t++)
#pragma unroll
            for (int rg = 0; rg < RH; rg++) {
                float v = 0.0f, u = 0.0f;
#pragma unroll
                for (int w = 0; w < NW; w++) v += red[t * RG + rg][w][l][r];
                if (SWI) {
#pragma unroll
                    for (int w = 0; w < NW; w++) u += red[RH + rg][w][l][r];
                }
                const int b = 16 * t + 4 * (l >> 4) + r, row = m0 + 16 * rg + (l & 15);
                if (SWI) {
                    if (b < B && row < M)
                        p.out_bf16[(size_t)b * p.out_bf16_ld + row] = t12_f32_to_bf16(t12_apply_glu(v, u, p.glu));
                } else if (b < B && row < M) outp[(size_t)b * sg.out_stride + row] = v;
            }
    }
    if (DEV && b_first + 16 * NBT < b_all) __syncthreads();  // the next batch rows reuse the reduction buffer
    }
}

template <int NW, int D, int RG, bool DEV = false, int NBT = 1>
__global__ __launch_bounds__(NW * 64) void gemm_dense16_kernel(const GemmParams p)
{
    __shared__ t12_f32x4 red[NBT * RG][NW][64];
    gemm_dense16_body<NW, D, RG, DEV, NBT>(p, red);
}

// The sweep with its loads turned through LDS, B <= 4 NX NBT.
template <int NW, int D, int NX, int RG = 1, int NBT = 1>
__global__ __launch_bounds__(NW * 64) void gemm_dense16_turned_kernel(const GemmParams p)
{
    constexpr int BYTES = d16_turn_bytes(NX) * NW, RED = RG * NBT * NW * 64 * 16;      // (the reduction takes the buffers over)
    __shared__ __align__(16) uint8_t turn[BYTES > RED ? BYTES : RED];
    gemm_dense16_body<NW, D, RG, false, NBT, false, NX>(p, (t12_f32x4(*)[NW][64])turn, turn);
}

// The sweep over one gate / up pair with the SiLU * mul in its last step (blockIdx.x counts sets of 16 RG / 2 rows).
template <int NW, int D, int RG>
__global__ __launch_bounds__(NW * 64) void gemm_dense16_swiglu_kernel(const GemmParams p)
{
    __shared__ t12_f32x4 red[RG][NW][64];
    gemm_dense16_body<NW, D, RG, false, 1, true>(p, red);
}

// The same sweep with two sizes of workgroup in one launch.  With RGA row groups per workgroup (its registers allow one
// workgroup per CU) a launch is a sequence of rounds of one workgroup per CU, each as long as a workgroup lives, and a
// last round that fills a fraction of the chip costs as much as a full one (gate|up at B = 16: 448 workgroups = 256 +
// 192, two rounds of 23 us).  The host therefore cuts every tensor in two: the first n_first segments of the launch
// are the heads of the tensors, swept RGA groups per workgroup in whole rounds, the others their tails, swept RGB < RGA
// groups per workgroup so that the last round covers the chip once with shorter workgroups.
template <int NW, int D, int RGA, int RGB>
__global__ __launch_bounds__(NW * 64) void gemm_dense16_mixed_kernel(const GemmParams p)
{
    __shared__ t12_f32x4 red[RGA][NW][64];
    if (find_segment(p, blockIdx.x) < p.n_first) gemm_dense16_body<NW, D, RGA, false>(p, red);
    else gemm_dense16_body<NW, D, RGB, false>(p, red);
}

// ---------------------------------------------------------------------------
// Two batch rows: the B = 1 kernel's shape with NB accumulators.  A workgroup = 8 waves = 8 consecutive rows;
// a wave reads its whole row front to back in 1024-column tiles (16 bytes of sign/mantissa + 8 bytes of nibbles per
// lane and tile, nontemporal, ring of two tiles) -- the access pattern that streams fastest on this chip -- rebuilds
// 16 weights per tile and multiplies them with the NB activation rows (v_dot2_f32_bf16), which the workgroup staged
// in LDS, paired the way t12_decode8 orders its outputs, laid out per row and 1024-column chunk as [half][lane] x 16 B.
// The decode is shared by the batch rows; per weight the kernel spends 2.25 + NB x 0.5 VALU operations and NB x 2
// bytes of LDS reads: measured with NB = 4 it is level with the MFMA kernel below, which therefore takes over from
// three rows on.  Escapes: (correct - wrong) * x[b, col] after the stream, x from LDS.  Wave sums by DPP.
// Requires K % 1024 == 0, NB * K * 2 bytes of LDS (K <= 8192), 0 <= base_exp <= 240, aligned activation rows.
// blk_start counts 8-row groups per segment.
// ---------------------------------------------------------------------------
template <int NB, int D>
__global__ __launch_bounds__(512) void gemm_rows_kernel(const GemmParams p)
{
    extern __shared__ uint4 lds_x[];                   // [NB][T * 128]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int K = p.K, B = p.B;
    const int T = K >> 10;
    const int blk = blockIdx.x;
    const int s = find_segment(p, blk);
    const T12Segment& sg = p.seg[s];
    const int M = sg.M;
    const int row = (blk - p.blk_start[s]) * 8 + wave;
    const bool live = row < M;                         // wave-uniform
    const uint32_t be2 = t12_opaque(((uint32_t)sg.base_exp << 7) | ((uint32_t)sg.base_exp << 23));

    // activations first (they come out of L2 and must not queue behind the weight tiles): piece = 8 columns,
    // NB * K / 8 pieces over 512 threads
    constexpr int XU = NB * 2;                         // pieces per thread at K = 8192
    const int kp = K >> 3;                             // pieces per batch row
    uint4 xpre[XU];
#pragma unroll
    for (int u = 0; u < XU; u++) {
        const int idx = tid + 512 * u;
        xpre[u] = make_uint4(0, 0, 0, 0);
        if (idx < NB * kp) {
            const int nb = idx / kp, q = idx - nb * kp;
            xpre[u] = *(const uint4*)(p.act + (size_t)min(nb, B - 1) * p.act_stride + q * 8);   // rows past the batch: clamped, never stored
        }
    }
    int e_beg = 0, e_end = 0;
    if (live && sg.row_off) {
        e_beg = sg.row_off[row];
        e_end = sg.row_off[row + 1];
    }
    const size_t e0 = (size_t)min(row, M - 1) * K;     // rows past the end: clamped, never stored
    const uint8_t* smp = sg.sm + e0 + lane * 16;
    const uint8_t* grp = sg.gr + (e0 >> 1) + lane * 8;
    uint4 rS[D];
    uint2 rG[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        const int t = min(d, T - 1);
        rS[d] = t12_ldg_stream16(smp + (size_t)t * 1024);
        rG[d] = t12_ldg_stream8(grp + (size_t)t * 512);
    }
#pragma unroll
    for (int u = 0; u < XU; u++) {
        const int idx = tid + 512 * u;
        if (idx < NB * kp) {
            const int nb = idx / kp, q = idx - nb * kp;
            lds_x[nb * (T * 128) + (q >> 7) * 128 + (q & 1) * 64 + ((q & 127) >> 1)] = t12_pair_acts(xpre[u]);
        }
    }
    __syncthreads();

    float acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) acc[nb] = 0.0f;
    auto consume = [&](int slot, int t) {
        uint32_t w0[4], w1[4];
        t12_decode8(rS[slot].x, rS[slot].y, rG[slot].x, be2, w0);
        t12_decode8(rS[slot].z, rS[slot].w, rG[slot].y, be2, w1);
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            const uint4 a0 = lds_x[nb * (T * 128) + t * 128 + lane];
            const uint4 a1 = lds_x[nb * (T * 128) + t * 128 + 64 + lane];
            float v = acc[nb];
            v = t12_dot2(w0[0], a0.x, v);
            v = t12_dot2(w0[1], a0.y, v);
            v = t12_dot2(w0[2], a0.z, v);
            v = t12_dot2(w0[3], a0.w, v);
            v = t12_dot2(w1[0], a1.x, v);
            v = t12_dot2(w1[1], a1.y, v);
            v = t12_dot2(w1[2], a1.z, v);
            v = t12_dot2(w1[3], a1.w, v);
            acc[nb] = v;
        }
    };
    for (int t = 0; t < T; t += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            if (t + d < T) {
                consume(d, t + d);
                if (t + d + D < T) {
                    rS[d] = t12_ldg_stream16(smp + (size_t)(t + d + D) * 1024);
                    rG[d] = t12_ldg_stream8(grp + (size_t)(t + d + D) * 512);
                }
            }
        }
    }
    // escapes: the streamed value of an escaped weight is its "wrong" value
    for (int e = e_beg + lane; e < e_end; e += 64) {
        const int col = sg.cols[e];
        const float delta = t12_bf16_to_f32((uint16_t)sg.correct[e]) - t12_bf16_to_f32((uint16_t)sg.wrong[e]);
        const int q = col >> 3, i = col & 7;
        const int slot = (q >> 7) * 128 + (q & 1) * 64 + ((q & 127) >> 1);
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            const uint16_t* h = (const uint16_t*)(lds_x + nb * (T * 128) + slot);
            acc[nb] += delta * t12_bf16_to_f32(h[(i & 3) * 2 + (i >> 2)]);
        }
    }
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const float v = t12_wave_sum_lane63(acc[nb]);
        if (lane == 63 && live && nb < B) sg.out[(size_t)nb * sg.out_stride + row] = v;
    }
}

// ---- workspace for the K-split partial sums: one per (device, stream), grown on demand.  Launches on different
//      streams may overlap, so they must not share partial sums; launches on one stream are ordered.
struct Workspace {
    float* ptr = nullptr;
    size_t bytes = 0;
    std::vector<float*> retired;      // outgrown buffers: kernels already in the stream may still write them
};
std::mutex g_ws_mutex;
std::map<std::pair<int, hipStream_t>, Workspace> g_ws;

float* workspace(size_t bytes, hipStream_t st)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    Workspace& w = g_ws[{dev, st}];
    if (w.bytes < bytes) {
        // Grows geometrically, in whole MiB, so a caller whose shapes grow step by step allocates a few times and the
        // outgrown buffers together stay below the live one.  They are kept until release_workspace: hipFree waits
        // for the whole device, which a launch call must not do.
        size_t want = bytes > 2 * w.bytes ? bytes : 2 * w.bytes;
        want = (want + ((size_t)1 << 20) - 1) & ~(((size_t)1 << 20) - 1);
        float* fresh = nullptr;
        if (hipMalloc((void**)&fresh, want) != hipSuccess) {
            (void)hipGetLastError();
            // short of memory: give the outgrown buffers back (this waits for the device) and ask for the exact size
            for (float* r : w.retired) (void)hipFree(r);
            w.retired.clear();
            if (w.ptr) (void)hipFree(w.ptr);
            w.ptr = nullptr;
            w.bytes = 0;
            want = bytes;
            if (hipMalloc((void**)&fresh, want) != hipSuccess) {
                (void)hipGetLastError();
                return nullptr;
            }
        }
        if (w.ptr) w.retired.push_back(w.ptr);
        w.ptr = fresh;
        w.bytes = want;
    }
    return w.ptr;
}

// Frees the K-split workspace of (current device, stream), outgrown buffers included.
void release_workspace(hipStream_t st)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return;
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    auto it = g_ws.find({dev, st});
    if (it == g_ws.end()) return;
    for (float* r : it->second.retired) (void)hipFree(r);
    if (it->second.ptr) (void)hipFree(it->second.ptr);
    g_ws.erase(it);
}

// ---- the same workspace for callers that may not allocate: a fixed array in the code object's own device
//      memory.  Every GPU the library runs on holds its own copy at its own address; the name below is only a
//      host-side handle for hipGetSymbolAddress, never a pointer a kernel could use.
constexpr size_t STATIC_WS_BYTES = (size_t)T12_GEMM_NOALLOC_WS_BYTES;
static __device__ __align__(256) float g_static_ws[STATIC_WS_BYTES / sizeof(float)];
std::mutex g_static_ws_mutex;
float* g_static_ws_ptr[16] = {};                       // per device, filled on the first call on that device

float* static_workspace()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return nullptr;
    std::lock_guard<std::mutex> lock(g_static_ws_mutex);
    if (!g_static_ws_ptr[dev]) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(g_static_ws)) != hipSuccess || !ptr) return nullptr;
        g_static_ws_ptr[dev] = (float*)ptr;
    }
    return g_static_ws_ptr[dev];
}


template <int FB, bool SWI = false, int EPI = T12_ACT_NONE, bool DEV = false>
int launch_tile(GemmParams& p, int tiles, hipStream_t st)
{
    const dim3 grid(tiles, (p.B + 64 * FB - 1) / (64 * FB), p.ksplit);   // batch tiles of one row tile are neighbours in time
    if constexpr (FB == 4) hipLaunchKernelGGL((gemm_tile_kernel<SWI, EPI, DEV>), grid, dim3(512), 0, st, p);
    else hipLaunchKernelGGL((gemm_strip_kernel<FB, SWI, EPI, DEV>), grid, dim3(512), 0, st, p);
    T12_CHECK_LAUNCH("t12_gemm");
    return T12_OK;
}


// Activation rows too far apart for a tile's 32-bit offsets: tiles of 128 batch rows whose lanes hold addresses, for any batch.  14336 x 4096 at 100 / 256
// rows 2^22 + 8 apart 36.0 / 61.6 us, side by side 35.5 / 53.4; the general kernel 3280 / 8130.
template <bool SWI = false, int EPI = T12_ACT_NONE>
int launch_far(GemmParams& p, int tiles, hipStream_t st)
{
    hipLaunchKernelGGL((gemm_strip_kernel<2, SWI, EPI, false, true>), dim3(tiles, (p.B + 127) / 128, p.ksplit), dim3(512), 0, st, p);
    T12_CHECK_LAUNCH("t12_gemm");
    return T12_OK;
}

template <bool SWI = false, int EPI = T12_ACT_NONE>
int launch_wide(GemmParams& p, int tiles, hipStream_t st)
{
    hipLaunchKernelGGL((gemm_wide_kernel<SWI, EPI>), dim3(tiles, (p.B + WIDE - 1) / WIDE, p.ksplit), dim3(512), 0, st, p);
    T12_CHECK_LAUNCH("t12_gemm");
    return T12_OK;
}

template <int RW, int KW, int NBT, bool GLU = false, bool DEV = false>
int launch_ring(GemmParams& p, int tiles, hipStream_t st)
{
    const dim3 grid(tiles, DEV ? 1 : (p.B + 16 * NBT - 1) / (16 * NBT), p.ksplit);
    hipLaunchKernelGGL((gemm_ring_kernel<RW, KW, NBT, GLU, DEV>), grid, dim3(RW * KW * 64), 0, st, p);
    T12_CHECK_LAUNCH("t12_gemm(ring)");
    return T12_OK;
}

// CUs of the current device (a launch of one workgroup per CU is one round of the small-batch kernel).
int device_cus()
{
    static std::mutex mu;
    static int cus[16] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 256;
    std::lock_guard<std::mutex> lock(mu);
    if (!cus[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

// More than 128 rows, unsplit: tiles of 256 x 256 in place of 128 x 256 where their rounds of one workgroup per CU take less time: a round of theirs
// takes 1.75 of the others' (a stage 1.6 us against 0.93, the ends alike).  One round against two: 28672 x 4096 at 512 rows 124 us and 140, 33000 x 256 / 1024 /
// 4096 at 256 17.7 / 36 / 113 and 22.6 / 48 / 129, 20000 x 512 / 2048 at 512 22.8 / 61 and 28.7 / 73; two against four: 128256 x 4096 at 256 300 and 317; one each: 28672 x
// 4096 at 160 / 256 101 / 103 and 77 / 76; two against three: 36000 x 2048 at 512 121 and 112, 28672 x 4096 at 700 219 and 203.
bool prefers_wide(int tiles, int wide, int cus)
{
    const int rounds = (tiles + cus - 1) / cus, rounds_wide = (wide + cus - 1) / cus;
    return rounds_wide * 1.75f < rounds;
}

// The ring kernel's form for a launch of p's segments (0 .. nseg - 1), or none: 3 .. 64 rows, K of whole 128-column
// windows, planes that 16-byte copies may be taken from.
RingPlan ring_plan_of(const GemmParams& p, int nseg)
{
    RingPlan none = {0, 0, 1, 0.0f};
    if (p.B < 3 || p.B > RING_MAX_B || p.K % RING_WC) return none;
    int rows[GMAX];
    for (int i = 0; i < nseg; i++) {
        if ((uintptr_t)p.seg[i].sm % 16 || (uintptr_t)p.seg[i].gr % 16) return none;
        rows[i] = p.seg[i].M;
    }
    return plan_ring(rows, nseg, p.K, p.B, device_cus());
}

template <int NBT, bool GLU>
int launch_ring_nbt(const RingPlan& r, GemmParams& p, int sets, hipStream_t st)
{
    if (r.kw == 1) return launch_ring<8, 1, NBT, GLU>(p, sets, st);
    if (r.kw == 2) return launch_ring<4, 2, NBT, GLU>(p, sets, st);
    if constexpr (NBT <= 2) {
        if (r.kw == 4) return launch_ring<2, 4, NBT, GLU>(p, sets, st);
    }
    if constexpr (NBT == 1) {
        if (r.kw == 8) return launch_ring<1, 8, NBT, GLU>(p, sets, st);
    }
    t12_set_error("t12_gemm: no ring form %d x %d for %d batch tiles", r.rw, r.kw, NBT);
    return T12_EINVAL;
}

template <bool GLU = false>
int launch_ring_form(const RingPlan& r, GemmParams& p, int sets, hipStream_t st)
{
    const int nbt = ring_batch_tiles(p.B);
    if (nbt == 1) return launch_ring_nbt<1, GLU>(r, p, sets, st);
    if (nbt == 2) return launch_ring_nbt<2, GLU>(r, p, sets, st);
    return launch_ring_nbt<4, GLU>(r, p, sets, st);
}

}  // namespace

extern "C" {

int t12_gemm(const T12Segment* segs, int nseg, const void* act_bf16, int act_stride, int out_stride, int K, int B,
             void* stream)
{
    return t12_gemm_deferred(segs, nseg, act_bf16, act_stride, out_stride, K, B, nullptr, stream);
}

// out_bf16[b, m] = bf16( silu(gate[m,:] . X[b,:]) * (up[m,:] . X[b,:]) ): gate|up projection with the SwiGLU
// in the GEMM's epilogue.  Returns T12_OK when launched, 1 when this shape has no fused kernel (the caller
// then runs t12_gemm on the two segments and launch_silu_mul_bf16_batch), negative on bad operands.
int t12_gemm_swiglu(const T12Segment* gate, const T12Segment* up, const void* act_bf16, int act_stride, int K, int B,
                    void* out_bf16, int out_stride, void* stream)
{
    const T12Glu silu = t12_silu_glu();
    return t12_gemm_glu(gate, up, &silu, act_bf16, act_stride, K, B, out_bf16, out_stride, stream);
}

// The same with any gated linear unit.
int t12_gemm_glu(const T12Segment* gate, const T12Segment* up, const T12Glu* glu, const void* act_bf16, int act_stride, int K, int B,
                 void* out_bf16, int out_stride, void* stream)
{
    T12_REQUIRE(gate && up && glu && act_bf16 && out_bf16, "t12_gemm_glu: null operand");
    T12_REQUIRE(K >= 1 && B >= 1 && act_stride >= K, "t12_gemm_glu: K %d, B %d or act_stride %d invalid", K, B, act_stride);
    T12_REQUIRE(gate->M >= 1 && gate->M == up->M, "t12_gemm_glu: gate has %d rows, up has %d", gate->M, up->M);
    T12_REQUIRE(out_stride >= gate->M, "t12_gemm_glu: out_stride %d < M %d", out_stride, gate->M);
    const T12Segment* two[2] = {gate, up};
    const bool aligned = act_stride % 8 == 0 && (uintptr_t)act_bf16 % 16 == 0;
    bool exps = true;
    for (const T12Segment* g : two) {
        T12_REQUIRE(g->sm && g->gr, "t12_gemm_glu: a plane is null");
        T12_REQUIRE(!g->row_off || (g->cols && g->correct && g->wrong), "t12_gemm_glu: row_off without lists");
        T12_REQUIRE(g->base_exp >= -1 && g->base_exp <= 254, "t12_gemm_glu: base_exp %d out of range", g->base_exp);
        if (g->base_exp < 0 || g->base_exp > 240) exps = false;
    }
    hipStream_t st = (hipStream_t)stream;
    GemmParams p;
    p.glu = *glu;
    p.seg[0] = *gate;
    p.seg[1] = *up;
    p.nseg = 2;
    p.K = K;
    p.B = B;
    p.act_stride = act_stride;
    p.act = (const uint16_t*)act_bf16;
    p.ws = nullptr;
    p.ksplit = 1;
    p.m_total = gate->M;
    p.seg_act[0] = p.act;                  // the paired kernels read the fields of segment 0
    p.seg_B[0] = B;
    p.seg_act_stride[0] = act_stride;
    p.seg_row0[0] = p.seg_row0[1] = 0;
    p.out_bf16 = (uint16_t*)out_bf16;
    p.out_bf16_ld = out_stride;
    if (B <= 64) {
        // The form that t12_gemm would take for the two tensors, so that the sums are the same bit for bit; above 8 rows only
        // with one K wave (128-row tiles: the chip is at least half full and nothing is split) from 8192 rows of gate on.  One
        // launch and the fp32 round trip of both projections less; in a loop of its own level at few rows and ahead at more: 14336 x
        // 1024 at B = 9 / 64 15.1 / 18.5 us against 15.5 / 20.0 in two launches, 14336 x 4096 37.4 / 42.6 against 36.7 / 43.4.
        const bool fast = K % 128 == 0 && aligned && exps && B >= 5;
        const RingPlan ring = fast ? ring_plan_of(p, 2) : RingPlan{0, 0, 1, 0.0f};
        if (ring.rw && ring.ks == 1 && (B <= 8 || (ring.kw == 1 && gate->M >= 64 * 128))) {
            const int sets = (gate->M + 8 * ring.rw - 1) / (8 * ring.rw);
            p.kslice = K;
            p.blk_start[0] = 0;
            p.blk_start[1] = p.blk_start[2] = sets;
            return launch_ring_form<true>(ring, p, sets, st);
        }
        if (!fast || B > 8 || ring.rw) return 1;
        // 5 .. 8 batch rows on fewer or shorter rows: the whole-row sweep over 32 rows of gate and the same rows of up per
        // workgroup (no gain at B <= 4, nor above 8, where the unfused launch balances its last round)
        const int sets = (gate->M + 31) / 32;
        p.kslice = K;
        p.blk_start[0] = 0;
        p.blk_start[1] = p.blk_start[2] = sets;
        hipLaunchKernelGGL((gemm_dense16_swiglu_kernel<8, 2, 4>), dim3(sets), dim3(512), 0, st, p);
        T12_CHECK_LAUNCH("t12_gemm_glu(dense16)");
        return T12_OK;
    }
    const bool fast = K % KC == 0 && aligned && exps;
    const int tiles = (gate->M + TM / 2 - 1) / (TM / 2);
    const int btiles = B > 128 ? (B + 255) / 256 : 1;
    if (!fast || tiles * btiles * 4 < 256 * 3) return 1;      // would need a K split: partial sums cannot be gated
    p.kslice = ((K + 2 * KC - 1) / (2 * KC)) * 2 * KC;
    p.blk_start[0] = 0;
    p.blk_start[1] = p.blk_start[2] = tiles;
    if (act_stride > TILE_MAX_STRIDE) return launch_far<true>(p, tiles, st);
    // batch tile of 256 rows, or of 128 for 65 .. 128 rows
    if (B <= 128) return launch_tile<2, true>(p, tiles, st);
    const int wide = (gate->M + WIDE / 2 - 1) / (WIDE / 2);
    if (prefers_wide(tiles * btiles, wide * btiles, device_cus())) {
        p.blk_start[1] = p.blk_start[2] = wide;
        return launch_wide<true>(p, wide, st);
    }
    return launch_tile<4, true>(p, tiles, st);
}

// out_bf16[b, m] = bf16(act(W[m,:] . X[b,:])) with the function in the GEMM's epilogue.  Returns T12_OK when launched, 1
// when this shape has no such kernel (the caller then runs t12_gemm or t12_gemm_deferred and the function on its own).
int t12_gemm_act(const T12Segment* seg, const void* act_bf16, int act_stride, int K, int B, const T12Act* act, void* out_bf16,
                 int out_stride, void* stream)
{
    T12_REQUIRE(seg && act_bf16 && act && out_bf16, "t12_gemm_act: null operand");
    T12_REQUIRE(K >= 1 && B >= 1 && act_stride >= K, "t12_gemm_act: K %d, B %d or act_stride %d invalid", K, B, act_stride);
    T12_REQUIRE(seg->M >= 1 && seg->sm && seg->gr && out_stride >= seg->M, "t12_gemm_act: rows %d, a plane or out_stride %d invalid",
                seg->M, out_stride);
    T12_REQUIRE(!seg->row_off || (seg->cols && seg->correct && seg->wrong), "t12_gemm_act: row_off without lists");
    T12_REQUIRE(seg->base_exp >= -1 && seg->base_exp <= 254, "t12_gemm_act: base_exp %d out of range", seg->base_exp);
    const int tiles = (seg->M + TM - 1) / TM, btiles = B > 128 ? (B + 255) / 256 : 1;
    // more than 64 batch rows, and a shape that is not one of few workgroups, which gemm_impl may split along K
    const bool splits = tiles * btiles * 2 <= 256 + 32 && K / 2 >= 8 * KC;
    if (act->kind != T12_ACT_XIELU || K % KC || act_stride % 8 || (uintptr_t)act_bf16 % 16 || B <= 64 || seg->base_exp < 0 ||
        seg->base_exp > 240 || splits)
        return 1;
    GemmParams p;
    p.seg[0] = *seg;
    p.nseg = 1;
    p.K = K;
    p.B = B;
    p.act_stride = act_stride;
    p.act = (const uint16_t*)act_bf16;
    p.ws = nullptr;
    p.ksplit = 1;
    p.kslice = ((K + 2 * KC - 1) / (2 * KC)) * 2 * KC;
    p.m_total = seg->M;
    p.seg_act[0] = p.act;
    p.seg_B[0] = B;
    p.seg_act_stride[0] = act_stride;
    p.blk_start[0] = 0;
    p.blk_start[1] = tiles;
    p.seg_row0[0] = 0;
    p.out_bf16 = (uint16_t*)out_bf16;
    p.out_bf16_ld = out_stride;
    p.act_a = act->a;
    p.act_b = act->b;
    if (act_stride > TILE_MAX_STRIDE) return launch_far<false, T12_ACT_XIELU>(p, tiles, (hipStream_t)stream);
    if (B <= 128) return launch_tile<2, false, T12_ACT_XIELU>(p, tiles, (hipStream_t)stream);
    const int wide = (seg->M + WIDE - 1) / WIDE;
    if (prefers_wide(tiles * btiles, wide * btiles, device_cus())) {
        p.blk_start[1] = wide;
        return launch_wide<false, T12_ACT_XIELU>(p, wide, (hipStream_t)stream);
    }
    return launch_tile<4, false, T12_ACT_XIELU>(p, tiles, (hipStream_t)stream);
}

}  // extern "C"

namespace {

// The small-batch launch with rg row groups per workgroup whose last round would fill only part of the chip: every
// tensor is cut into a head, swept rg groups per workgroup in whole rounds, and a tail swept in fewer groups per
// workgroup, chosen so that the tails of all tensors together are one round.  p holds the launch as gemm_impl set it up
// (segments, K, B, activations); returns false, with nothing launched, when the plain launch is as good.
bool launch_dense16_mixed(GemmParams p, int nseg, int rg, hipStream_t st)
{
    int rows[GMAX], head_rows[GMAX];
    for (int i = 0; i < nseg; i++) rows[i] = p.seg[i].M;
    const int rgb = t12_plan_dense16_heads(rows, nseg, rg, device_cus(), GMAX, head_rows);
    if (!rgb) return false;
    // heads first, then tails.  A tail is the same tensor from row 16 rg a on: the row pointers of the escape list hold
    // absolute entry numbers, so only the pointer to them moves; 16 rg a rows of K columns are a whole number of bytes of
    // the nibble plane.
    T12Segment src[GMAX];
    for (int i = 0; i < nseg; i++) src[i] = p.seg[i];
    int n = 0, total = 0;
    p.n_first = 0;
    for (int pass = 0; pass < 2; pass++)
        for (int i = 0; i < nseg; i++) {
            const int rows_a = head_rows[i];
            const int m = pass == 0 ? rows_a : src[i].M - rows_a;
            if (m <= 0) continue;
            T12Segment g = src[i];
            if (pass == 1) {
                const size_t e = (size_t)rows_a * p.K;
                g.sm += e;
                g.gr += e / 2;
                if (g.row_off) g.row_off += rows_a;
                g.out += rows_a;
            }
            g.M = m;
            const int per = 16 * (pass == 0 ? rg : rgb);
            p.seg[n] = g;
            p.blk_start[n] = total;
            total += (m + per - 1) / per;
            n++;
            if (pass == 0) p.n_first = n;
        }
    p.blk_start[n] = total;
    p.nseg = n;
    p.ksplit = 1;
    p.kslice = p.K;
    const dim3 grid(total), block(512);
    if (rg == 4 && rgb == 3) hipLaunchKernelGGL((gemm_dense16_mixed_kernel<8, 2, 4, 3>), grid, block, 0, st, p);
    else if (rg == 4 && rgb == 2) hipLaunchKernelGGL((gemm_dense16_mixed_kernel<8, 2, 4, 2>), grid, block, 0, st, p);
    else if (rg == 4 && rgb == 1) hipLaunchKernelGGL((gemm_dense16_mixed_kernel<8, 2, 4, 1>), grid, block, 0, st, p);
    else if (rg == 2 && rgb == 1) hipLaunchKernelGGL((gemm_dense16_mixed_kernel<8, 2, 2, 1>), grid, block, 0, st, p);
    else return false;
    return true;
}

#define NOALLOC_TOO_LARGE                                                                                          \
    "t12_gemm_noalloc: this shape splits K %d ways and needs %zu bytes of partial sums, the fixed "               \
    "workspace holds %zu (B %d x %d rows): use t12_gemm, or a smaller batch"

// Slices that ks slices of whole windows of two stages come to.
int t12_slices(int K, int ks)
{
    const int windows = (K + 2 * KC - 1) / (2 * KC), per = (windows + ks - 1) / ks;
    return (windows + per - 1) / per;
}

// The body of t12_gemm / t12_gemm_deferred / t12_gemm_noalloc.  static_ws: the K-split partial sums go to the
// library's fixed device array instead of a grown hipMalloc buffer, and a launch that needs more is refused.
int gemm_impl(const T12Segment* segs, int nseg, const void* act_bf16, int act_stride, int out_stride, int K,
              int B, T12GemmPartials* part, void* stream, bool static_ws)
{
    if (part) {
        part->ws = nullptr;
        part->nsplit = 1;
        part->ld = 0;
        part->split_stride = 0;
    }
    const char* who = static_ws ? "t12_gemm_noalloc" : "t12_gemm";
    T12_REQUIRE(segs && nseg >= 1 && nseg <= T12_MAX_SEGMENTS, "%s: nseg must be 1..%d (got %d)", who,
                T12_MAX_SEGMENTS, nseg);
    T12_REQUIRE(act_bf16 && K >= 1 && B >= 1, "%s: activations null or K/B < 1 (K=%d B=%d)", who, K, B);
    T12_REQUIRE(act_stride >= K, "%s: act_stride %d < K %d", who, act_stride, K);
    hipStream_t st = (hipStream_t)stream;
    GemmParams p;
    p.nseg = nseg;
    p.K = K;
    p.B = B;
    p.act_stride = act_stride;
    p.act = (const uint16_t*)act_bf16;
    p.ws = nullptr;
    p.out_bf16 = nullptr;
    p.out_bf16_ld = 0;
    bool fast = (K % KC == 0) && (act_stride % 8 == 0) && ((uintptr_t)act_bf16 % 16 == 0);
    int m_total = 0;
    for (int i = 0; i < nseg; i++) {
        const T12Segment& g = segs[i];
        T12_REQUIRE(g.M >= 1 && g.sm && g.gr && g.out, "%s: segment %d has M < 1 or a null pointer", who, i);
        T12_REQUIRE(!g.row_off || (g.cols && g.correct && g.wrong), "%s: segment %d: row_off without lists", who, i);
        T12_REQUIRE(g.base_exp >= -1 && g.base_exp <= 254, "%s: segment %d: base_exp %d out of range", who, i,
                    g.base_exp);
        if (g.base_exp < 0 || g.base_exp > 240) fast = false;
        p.seg[i] = g;
        if (p.seg[i].out_stride == 0) p.seg[i].out_stride = out_stride;
        T12_REQUIRE(p.seg[i].out_stride >= g.M, "%s: out_stride %d < M %d of segment %d", who, p.seg[i].out_stride,
                    g.M, i);
        p.seg_row0[i] = m_total;
        p.seg_act[i] = p.act;
        p.seg_B[i] = B;
        p.seg_act_stride[i] = act_stride;
        m_total += g.M;
    }
    p.m_total = m_total;
    for (int i = 0; i < nseg; i++) {
        p.seg_ws0[i] = (size_t)p.seg_row0[i];
        p.seg_ld[i] = m_total;
    }
    p.split_stride = (size_t)B * m_total;

    if (!fast) {
        int tiles = 0;
        for (int i = 0; i < nseg; i++) {
            p.blk_start[i] = tiles;
            tiles += (segs[i].M + 3) / 4;
        }
        p.blk_start[nseg] = tiles;
        p.ksplit = 1;
        p.kslice = K;
        hipLaunchKernelGGL(gemm_general_kernel, dim3(tiles, (B + 7) / 8), dim3(256), 0, st, p);
        T12_CHECK_LAUNCH("t12_gemm(general)");
        return T12_OK;
    }

    int tiles = 0;
    for (int i = 0; i < nseg; i++) {
        p.blk_start[i] = tiles;
        tiles += (segs[i].M + TM - 1) / TM;
    }
    p.blk_start[nseg] = tiles;
    if (B == 2 && K % 1024 == 0 && K <= 8192) {
        // two batch rows: whole-row waves with two accumulators (gate|up 32 us against 42 for the kernel below; with
        // four accumulators the same kernel is no faster than the kernel below, 43-48 us, so it stops at two)
        int groups = 0;
        for (int i = 0; i < nseg; i++) {
            p.blk_start[i] = groups;
            groups += (segs[i].M + 7) / 8;
        }
        p.blk_start[nseg] = groups;
        p.ksplit = 1;
        p.kslice = K;
        hipLaunchKernelGGL((gemm_rows_kernel<2, 2>), dim3(groups), dim3(512), (size_t)2 * K * 2, st, p);
        T12_CHECK_LAUNCH("t12_gemm(rows)");
        return T12_OK;
    }
    // K split: where the partial sums of p.ksplit slices go, and who adds them up
    auto take_workspace = [&]() {
        const size_t need = (size_t)p.ksplit * B * m_total * sizeof(float);
        if (static_ws) {
            T12_REQUIRE(need <= STATIC_WS_BYTES, NOALLOC_TOO_LARGE, p.ksplit, need, STATIC_WS_BYTES, B, m_total);
            p.ws = static_workspace();
            if (!p.ws) {
                t12_set_error("t12_gemm_noalloc: hipGetSymbolAddress of the fixed workspace failed");
                return T12_ELAUNCH;
            }
            return T12_OK;
        }
        p.ws = workspace(need, st);
        if (!p.ws) {
            t12_set_error("%s: cannot allocate %zu bytes of K-split workspace", who, need);
            return T12_ELAUNCH;
        }
        return T12_OK;
    };
    auto finish = [&]() {
        if (p.ksplit > 1 && part) {
            part->ws = p.ws;
            part->nsplit = p.ksplit;
            part->ld = m_total;
            part->split_stride = (size_t)B * m_total;
        } else if (p.ksplit > 1) {
            launch_reduce(p, B, st);
            T12_CHECK_LAUNCH("t12_gemm(reduce)");
        }
        return T12_OK;
    };
    const RingPlan ring = ring_plan_of(p, nseg);
    if (ring.rw) {
        int sets = 0;
        for (int i = 0; i < nseg; i++) {
            p.blk_start[i] = sets;
            sets += (segs[i].M + 16 * ring.rw - 1) / (16 * ring.rw);
        }
        p.blk_start[nseg] = sets;
        const int per = (K / RING_WC + ring.ks - 1) / ring.ks;
        p.ksplit = ring.ks;
        p.kslice = per * RING_WC;
        if (p.ksplit > 1) {
            const int rc = take_workspace();
            if (rc) return rc;
        }
        const int rc = launch_ring_form(ring, p, sets, st);
        return rc ? rc : finish();
    }
    if (B > 16 && B <= 32 && K % 128 == 0) {
        // 17 .. 32 batch rows on tensors of few rows, which the plan above left to the sweep (or whose planes the ring kernel cannot
        // copy): the sweep of up to 16 rows with two batch tiles per weight load and decode.  One round of workgroups takes the same
        // whatever the row count, because every workgroup reads all B activation rows for its 16 (32) weight rows: at B = 17 / 24 / 32 and
        // 4096 columns 10.4 / 11.0 / 11.3 us (12.0 / 13.1 / 14.4 before the turn through LDS, which the rule was fitted to).
        int groups16 = 0, sets2 = 0;
        for (int i = 0; i < nseg; i++) {
            groups16 += (segs[i].M + 15) / 16;
            sets2 += (segs[i].M + 31) / 32;
        }
        const int rg = sweep_row_groups(groups16, sets2, K, B, device_cus());
        if (rg) {
            int groups = 0;
            for (int i = 0; i < nseg; i++) {
                p.blk_start[i] = groups;
                groups += (segs[i].M + 16 * rg - 1) / (16 * rg);
            }
            p.blk_start[nseg] = groups;
            p.ksplit = 1;
            p.kslice = K;
            if (rg == 2) hipLaunchKernelGGL((gemm_dense16_turned_kernel<8, 2, 4, 2, 2>), dim3(groups), dim3(512), 0, st, p);
            else hipLaunchKernelGGL((gemm_dense16_turned_kernel<8, 2, 4, 1, 2>), dim3(groups), dim3(512), 0, st, p);
            T12_CHECK_LAUNCH("t12_gemm(dense16, two batch tiles)");
            return T12_OK;
        }
    }
    if (B <= 16 && K % 128 == 0) {
        // row groups that share an activation load: as many as leave the launch >= 448 workgroups
        int groups16 = 0;
        for (int i = 0; i < nseg; i++) groups16 += (segs[i].M + 15) / 16;
        // (measured on 28672 x 4096: at B = 16 four groups per load 49 us against 56 with one; at B = 4 45 against 42:
        // rows of a padded batch cost no activation traffic, more rows per wave cost registers)
        const int want = B > 8 ? 4 : (B > 4 ? 2 : 1);
        const int rg = groups16 >= 4 * 448 && want >= 4 ? 4 : (groups16 >= 2 * 448 && want >= 2 ? 2 : 1);
        if (rg > 1 && launch_dense16_mixed(p, nseg, rg, st)) {
            T12_CHECK_LAUNCH("t12_gemm(dense16, two workgroup sizes)");
            return T12_OK;
        }
        int groups = 0;
        for (int i = 0; i < nseg; i++) {
            p.blk_start[i] = groups;
            groups += (segs[i].M + 16 * rg - 1) / (16 * rg);
        }
        p.blk_start[nseg] = groups;
        p.ksplit = 1;
        p.kslice = K;
        if (rg == 4) hipLaunchKernelGGL((gemm_dense16_kernel<8, 2, 4>), dim3(groups), dim3(512), 0, st, p);
        else if (rg == 2) hipLaunchKernelGGL((gemm_dense16_kernel<8, 2, 2>), dim3(groups), dim3(512), 0, st, p);
        else if (B <= 4) hipLaunchKernelGGL((gemm_dense16_turned_kernel<8, 2, 1>), dim3(groups), dim3(512), 0, st, p);
        else if (B <= 8) hipLaunchKernelGGL((gemm_dense16_turned_kernel<8, 2, 2>), dim3(groups), dim3(512), 0, st, p);
        else hipLaunchKernelGGL((gemm_dense16_turned_kernel<8, 2, 4>), dim3(groups), dim3(512), 0, st, p);
        T12_CHECK_LAUNCH("t12_gemm(dense16)");
        return T12_OK;
    }
    // K split: as many workgroups as the chip has CUs, not more (measured on the four Llama-8B layer shapes at B = 32 ..
    // 256: 32 row tiles run best as 8 splits, 48 as 4, 224 unsplit -- every doubling past ~one workgroup per CU costs more
    // in partial sums than it gains), every split at least 8 stages long.
    auto splits_for = [&](int btiles) {
        int ks = 1;
        while (tiles * btiles * ks * 2 <= 256 + 32 && K / (ks * 2) >= 8 * KC && ks < T12_MAX_KSPLIT) ks *= 2;
        return ks;
    };
    const int btiles = B > 128 ? (B + 255) / 256 : 1, btiles128 = (B + 127) / 128, cus = device_cus();
    int ks = splits_for(btiles);
    // A 256-row batch tile whose K slice is under 16 stages (O of the Llama layer: 32 row tiles, 8 splits of 512
    // columns) spends its time filling and draining, and leaves twice the partial sums: such a launch takes 128-row
    // batch tiles and half the splits (with the reduction: O at B = 160 / 256 25.9 / 28.7 -> 23.6 / 25.0 us, 2048 x 8192 at 200 / 256 30 -> 25, 2048 x 2048
    // at 200 20.4 -> 17.6; down, whose slices are long, level at 256 and 77.7 -> 84.3 us at 512 the same way, QKV at 160 / 256, its sums left to
    // the next kernel, 24.8 / 25.7 -> 25.5 / 26.0, so they keep the 256-row tile).
    const bool short_slices = B > 128 && ks > 1 && K / ks < 16 * KC;
    const int ks128 = short_slices ? splits_for(btiles128) : ks;
    if (static_ws) {
        // what t12_gemm_noalloc refuses is said by the full split, whatever is taken below
        p.ksplit = t12_slices(K, ks128);
        const size_t need = (size_t)p.ksplit * B * m_total * sizeof(float);
        T12_REQUIRE(p.ksplit == 1 || need <= STATIC_WS_BYTES, NOALLOC_TOO_LARGE, p.ksplit, need, STATIC_WS_BYTES, B, m_total);
    }
    // (where those are more workgroups than CUs, 256-row tiles are the better ones: 8400 x 1024 at B = 512, 264 workgroups 27.6 us,
    // 132 of the larger ones 22.3)
    const bool tb128 = short_slices && tiles * btiles128 * t12_slices(K, ks128) <= cus;
    if (tb128) ks = ks128;
    // A few workgroups more than CUs are a second round of everything: one round of fewer slices then, or none, by  rounds x (6.5
    // us + stages x c) + what the partial sums cost (2.5 us and 4 TB/s, as for the ring kernel), c = 0.95 us for a stage of 256
    // batch rows, 0.65 for 128 (unsplit 8256 x 2048 / 8704 x 8192 at 512 rows: 0.86 / 0.78).  8256 x 2048 at B = 512: 260 workgroups of 2 slices 42.8 us and a
    // reduction of 12, unsplit 34.0; 8400 x 1024 29.2 and 12, unsplit 22.0; 4224 x 4096: 264 of 4 slices 42.5, 3 slices 28.1; 8704 x 8192: 272 of 2
    // slices 127, unsplit 107.
    if (!tb128 && ks > 1 && tiles * btiles * t12_slices(K, ks) > cus) {
        const int windows = (K + 2 * KC - 1) / (2 * KC);
        float best = 1e30f;
        for (int k = ks; k >= 1; k--) {
            if (k > 1 && tiles * btiles * k > cus) continue;
            const int rounds = (tiles * btiles * k + cus - 1) / cus, per = (windows + k - 1) / k;
            const float us = rounds * (6.5f + 2 * per * (B > 128 ? 0.95f : 0.65f)) + (k > 1 ? 2.5f + (float)k * B * m_total * 1e-6f : 0.0f);
            if (us < best) {
                best = us;
                ks = k;
            }
        }
    }
    int kslice = (((K + 2 * KC - 1) / (2 * KC) + ks - 1) / ks) * 2 * KC;      // whole windows of two stages
    ks = (K + kslice - 1) / kslice;
    p.ksplit = ks;
    p.kslice = kslice;
    if (ks > 1) {
        const int rc_ws = take_workspace();
        if (rc_ws) return rc_ws;
    }
    int rc;
    if (act_stride > TILE_MAX_STRIDE) rc = launch_far(p, tiles, st);
    else if (B <= 64) rc = launch_tile<1>(p, tiles, st);
    else if (B <= 128 || tb128) rc = launch_tile<2>(p, tiles, st);
    else {
        int wide = 0;
        for (int i = 0; i < nseg; i++) wide += (segs[i].M + WIDE - 1) / WIDE;
        if (ks == 1 && prefers_wide(tiles * btiles, wide * btiles, cus)) {
            wide = 0;
            for (int i = 0; i < nseg; i++) {
                p.blk_start[i] = wide;
                wide += (segs[i].M + WIDE - 1) / WIDE;
            }
            p.blk_start[nseg] = wide;
            rc = launch_wide(p, wide, st);
        } else {
            rc = launch_tile<4>(p, tiles, st);
        }
    }
    return rc ? rc : finish();
}

}  // namespace

extern "C" {

// t12_gemm whose K-split partial sums may be left in the workspace for the caller's next kernel to add
// up (part != NULL): part->nsplit == 1 means the outputs are complete in segs[].out.
int t12_gemm_deferred(const T12Segment* segs, int nseg, const void* act_bf16, int act_stride, int out_stride, int K,
                      int B, T12GemmPartials* part, void* stream)
{
    return gemm_impl(segs, nseg, act_bf16, act_stride, out_stride, K, B, part, stream, false);
}

// t12_gemm for callers that may not allocate device memory (HIP graph capture, serving loops, harnesses that forbid
// it): same kernels, same K split, same results bit for bit; the partial sums of a split launch live in a fixed
// T12_GEMM_NOALLOC_WS_BYTES array inside the library's device image instead of a buffer grown with hipMalloc.
// Every launch writes each partial sum it later adds, so the array needs no clearing between calls; all calls on
// one GPU share it, whatever their stream: calls that overlap in time on one GPU race.
int t12_gemm_noalloc(const T12Segment* segs, int nseg, const void* act_bf16, int act_stride, int out_stride, int K,
                     int B, void* stream)
{
    return gemm_impl(segs, nseg, act_bf16, act_stride, out_stride, K, B, nullptr, stream, true);
}

// Several products in one launch, each tensor with its own activations and batch: the experts of a mixture-of-experts
// layer (gate and up of expert e over the rows routed to e), where a launch per expert leaves the chip part empty
// and pays a K-split reduction per expert.  The row tiles of all groups fill one grid; a group with fewer rows than
// the largest simply has fewer batch tiles.  Groups the tile kernel does not take (K % 64, base_exp outside 0..240,
// activations not 16-byte aligned) run as t12_gemm calls, one per group.
int t12_gemm_grouped(const T12Group* groups, int ngroups, int K, void* stream)
{
    T12_REQUIRE(groups && ngroups >= 1 && ngroups <= GMAX, "t12_gemm_grouped: 1..%d groups (got %d)", GMAX, ngroups);
    T12_REQUIRE(K >= 1, "t12_gemm_grouped: K %d", K);
    hipStream_t st = (hipStream_t)stream;
    GemmParams p;
    p.K = K;
    p.act = nullptr;
    p.act_stride = 0;
    p.ws = nullptr;
    p.out_bf16 = nullptr;
    p.out_bf16_ld = 0;
    bool fast = K % KC == 0;
    int n = 0, m_total = 0, max_b = 0, max_stride = 0;
    size_t ws_floats = 0;
    for (int i = 0; i < ngroups; i++) {
        const T12Group& g = groups[i];
        const T12Segment& w = g.seg;
        T12_REQUIRE(g.B >= 0, "t12_gemm_grouped: group %d has B %d", i, g.B);
        if (g.B == 0) continue;                                   // an expert no row was routed to
        T12_REQUIRE(w.M >= 1 && w.sm && w.gr && w.out && g.act_bf16, "t12_gemm_grouped: group %d has M < 1 or a null pointer", i);
        T12_REQUIRE(!w.row_off || (w.cols && w.correct && w.wrong), "t12_gemm_grouped: group %d: row_off without lists", i);
        T12_REQUIRE(w.base_exp >= -1 && w.base_exp <= 254, "t12_gemm_grouped: group %d: base_exp %d out of range", i, w.base_exp);
        T12_REQUIRE(g.act_stride >= K && w.out_stride >= w.M, "t12_gemm_grouped: group %d: act_stride %d < K %d or out_stride %d < M %d",
                    i, g.act_stride, K, w.out_stride, w.M);
        if (w.base_exp < 0 || w.base_exp > 240 || g.act_stride % 8 != 0 || (uintptr_t)g.act_bf16 % 16 != 0) fast = false;
        p.seg[n] = w;
        p.seg_row0[n] = m_total;
        p.seg_act[n] = (const uint16_t*)g.act_bf16;
        p.seg_B[n] = g.B;
        p.seg_act_stride[n] = g.act_stride;
        p.seg_ws0[n] = ws_floats;
        p.seg_ld[n] = w.M;
        ws_floats += (size_t)g.B * w.M;
        m_total += w.M;
        max_b = std::max(max_b, g.B);
        max_stride = std::max(max_stride, g.act_stride);
        n++;
    }
    if (n == 0) return T12_OK;
    if (!fast) {
        for (int i = 0; i < n; i++) {
            const int rc = gemm_impl(&p.seg[i], 1, p.seg_act[i], p.seg_act_stride[i], p.seg[i].out_stride, K, p.seg_B[i],
                                     nullptr, stream, false);
            if (rc) return rc;
        }
        return T12_OK;
    }
    p.nseg = n;
    p.B = max_b;
    p.m_total = m_total;
    p.split_stride = ws_floats;
    // batch tile by the largest group, so that every tensor is streamed once (the two launches of a Mixtral layer of 256 tokens, 48 .. 75
    // rows per expert: 0.58 ms with tiles of 128, 0.69 with tiles of 64 taken twice by the larger groups, 0.80 with 256)
    const int tb = max_b <= 64 ? 64 : (max_b <= 128 ? 128 : 256);
    int tiles = 0;
    long units = 0;                                               // workgroups per K split
    for (int i = 0; i < n; i++) {
        p.blk_start[i] = tiles;
        const int t = (p.seg[i].M + TM - 1) / TM;
        tiles += t;
        units += (long)t * ((p.seg_B[i] + tb - 1) / tb);
    }
    p.blk_start[n] = tiles;
    int ks = 1;
    while (units * ks * 2 <= 256 + 32 && K / (ks * 2) >= 8 * KC && ks < T12_MAX_KSPLIT) ks *= 2;
    const int kslice = (((K + 2 * KC - 1) / (2 * KC) + ks - 1) / ks) * 2 * KC;
    ks = (K + kslice - 1) / kslice;
    p.ksplit = ks;
    p.kslice = kslice;
    if (ks > 1) {
        p.ws = workspace((size_t)ks * ws_floats * sizeof(float), st);
        if (!p.ws) {
            t12_set_error("t12_gemm_grouped: cannot allocate %zu bytes of K-split workspace", (size_t)ks * ws_floats * sizeof(float));
            return T12_ELAUNCH;
        }
    }
    int rc;
    if (max_stride > TILE_MAX_STRIDE) rc = launch_far(p, tiles, st);
    else if (tb == 64) rc = launch_tile<1>(p, tiles, st);
    else if (tb == 128) rc = launch_tile<2>(p, tiles, st);
    else rc = launch_tile<4>(p, tiles, st);
    if (rc) return rc;
    if (ks > 1) {
        launch_reduce(p, max_b, st);
        T12_CHECK_LAUNCH("t12_gemm_grouped(reduce)");
    }
    return T12_OK;
}

// Library-internal (t12_moe_ffn): the experts of a mixture-of-experts layer in one launch, with the rows per expert
// known on the device only.  pairs = 0: segment i belongs to group first_group + i; 1 or 2: the segments are (gate, up)
// pairs, segment i belongs to group first_group + i / 2.  Group g has dev_counts[g] rows, which start dev_base[g] rows
// into act_bf16 and into the outputs: seg.out (fp32), or for pairs = 1 out_bf16 = bf16( silu(gate) * up ), row stride
// out_bf16_ld (asked for with hint_b above 128 only: tiles of 256 batch rows).  hint_b is a count few groups exceed: it
// picks the batch tile (a group above it is streamed once per tile it needs).  K is never split.  Returns 1 when the shape has no such kernel (the caller then sizes launches on the host).
__attribute__((visibility("hidden"))) int t12_gemm_experts(const T12Segment* segs, int nseg, int K, const void* act_bf16,
                                                           int act_stride, const int* dev_counts, const int* dev_base,
                                                           int first_group, int hint_b, int pairs,
                                                           void* out_bf16, int out_bf16_ld, void* stream)
{
    const bool swiglu = pairs == 1;
    if (nseg < 1 || nseg > GMAX || (pairs && nseg % 2)) return 1;
    if (K % KC || act_stride % 8 || (uintptr_t)act_bf16 % 16) return 1;
    for (int i = 0; i < nseg; i++)
        if (segs[i].base_exp < 0 || segs[i].base_exp > 240 || !segs[i].sm || !segs[i].gr) return 1;
    GemmParams p;
    p.K = K;
    p.act = (const uint16_t*)act_bf16;
    p.act_stride = act_stride;
    p.ws = nullptr;
    p.ksplit = 1;
    p.kslice = ((K + 2 * KC - 1) / (2 * KC)) * 2 * KC;
    p.out_bf16 = (uint16_t*)out_bf16;
    p.out_bf16_ld = out_bf16_ld;
    p.dev_counts = dev_counts;
    p.dev_base = dev_base;
    p.nseg = nseg;
    p.B = 1;                               // one workgroup per row tile (it walks the group's batch tiles itself)
    p.split_stride = 0;
    int tiles = 0, m_total = 0;
    for (int i = 0; i < nseg; i++) {
        p.seg[i] = segs[i];
        p.seg_row0[i] = m_total;
        p.seg_act[i] = p.act;
        p.seg_B[i] = 0;
        p.seg_act_stride[i] = act_stride;
        p.seg_ws0[i] = 0;
        p.seg_ld[i] = segs[i].M;
        p.group_of_seg[i] = first_group + (pairs ? i / 2 : i);
        m_total += segs[i].M;
        if (!swiglu) {
            p.blk_start[i] = tiles;
            tiles += (segs[i].M + TM - 1) / TM;
        } else if (i % 2 == 0) {
            if (segs[i].M != segs[i + 1].M) return 1;
            p.blk_start[i / 2] = tiles;
            tiles += (segs[i].M + TM / 2 - 1) / (TM / 2);
        }
    }
    p.m_total = m_total;
    p.npair = swiglu ? nseg / 2 : 1;
    if (!swiglu) p.blk_start[nseg] = tiles;
    hipStream_t st = (hipStream_t)stream;
    // More than a few rows per group: the ring kernel, whose workgroups of 128 rows stream at the memory's rate.  Eight
    // experts of 4096 / 14336, two per token, whole layer: 12 / 40 / 64 / 128 tokens 353 / 365 / 376 / 430 us, 444 / 439 /
    // 448 / 469 through the strip kernel; 8 tokens (hint 8) 285 against 398 by the sweep below.  It stops at a hint of 6: with
    // a few of many small experts named there are too few workgroups (64 experts of 2048 / 1408, six per token: 4 tokens,
    // hint 3, 236 us against the sweep's 177, 16 tokens, hint 7, 245 against 309; 32 of 4096 / 768, hint 5: 186 against 179).
    bool ring = !swiglu && hint_b > 6 && hint_b <= RING_MAX_B && K % RING_WC == 0;
    for (int i = 0; i < nseg; i++) ring = ring && (uintptr_t)segs[i].sm % 16 == 0 && (uintptr_t)segs[i].gr % 16 == 0;
    if (ring) {
        p.kslice = K;
        const int nbt = ring_batch_tiles(hint_b);
        if (nbt == 1) return launch_ring<8, 1, 1, false, true>(p, tiles, st);
        if (nbt == 2) return launch_ring<8, 1, 2, false, true>(p, tiles, st);
        return launch_ring<8, 1, 4, false, true>(p, tiles, st);
    }
    if (!swiglu && hint_b <= 8 && K % 128 == 0) {
        // a few rows per group (a decode step of a mixture-of-experts model): bound by the weight stream, so the kernel
        // that sweeps 16 whole rows per workgroup; groups without rows cost a workgroup's exit
        int groups = 0;
        for (int i = 0; i < nseg; i++) {
            p.blk_start[i] = groups;
            groups += (segs[i].M + 15) / 16;
        }
        p.blk_start[nseg] = groups;
        p.kslice = K;
        hipLaunchKernelGGL((gemm_dense16_kernel<8, 2, 1, true>), dim3(groups), dim3(512), 0, st, p);
        T12_CHECK_LAUNCH("t12_moe_ffn(dense16)");
        return T12_OK;
    }
    if (act_stride > TILE_MAX_STRIDE) return 1;
    if (swiglu) return launch_tile<4, true, T12_ACT_NONE, true>(p, tiles, st);
    if (hint_b <= 64) return launch_tile<1, false, T12_ACT_NONE, true>(p, tiles, st);
    if (hint_b <= 128) return launch_tile<2, false, T12_ACT_NONE, true>(p, tiles, st);
    return launch_tile<4, false, T12_ACT_NONE, true>(p, tiles, st);
}

// The library keeps device buffers per (device, stream): the K-split partial sums of t12_gemm*, the argmax partials and the
// context-split buffers of the glue kernels, the sampler's result ids.  A caller about to destroy a stream hands them back here (waits for the
// stream first); a stream that is used again afterwards simply gets new ones.
int t12_release_stream(void* stream)
{
    hipStream_t st = (hipStream_t)stream;
    if (hipStreamSynchronize(st) != hipSuccess) {
        t12_set_error("t12_release_stream: hipStreamSynchronize failed: %s", hipGetErrorString(hipGetLastError()));
        return T12_ELAUNCH;
    }
    release_workspace(st);
    t12_glue_release_stream(st);
    t12_sampler_release_stream(st);
    return T12_OK;
}

}  // extern "C"
