// What one decode+GEMM launch is told (gemm.hip, gemm_ring.h).
#pragma once
#include "t12_act.h"
#include "t12_device.h"
#include "t12_host.h"

namespace {

constexpr int GMAX = 16;        // segments of one launch (a grouped launch: gate and up of eight experts)
static_assert(GMAX >= T12_MAX_SEGMENTS, "t12_gemm takes T12_MAX_SEGMENTS segments");

// One launch multiplies up to GMAX tensors.  t12_gemm: all of them with the same activations [B, K]; a grouped
// launch (t12_gemm_grouped): segment i with its own seg_act[i] of seg_B[i] rows.  The tile kernel and the K-split
// reduction read the per-segment fields, which t12_gemm fills with the shared values; the other kernels read
// act / B / act_stride.
struct GemmParams {
    T12Segment seg[GMAX];
    int blk_start[GMAX + 1];               // first row-tile of each segment
    int seg_row0[GMAX];                    // first row of each segment among all rows of the launch
    const uint16_t* seg_act[GMAX];
    int seg_B[GMAX];
    int seg_act_stride[GMAX];
    // partial sums of segment i, split z, element (b, m): ws[z * split_stride + seg_ws0[i] + b * seg_ld[i] + m]
    //   t12_gemm: seg_ws0 = seg_row0, seg_ld = m_total (rows of length m_total, what t12_gemm_deferred describes)
    //   grouped:  seg_ws0 = sum of B * M over the segments before, seg_ld = M
    size_t seg_ws0[GMAX];
    int seg_ld[GMAX];
    size_t split_stride;
    int nseg;
    int K, B;                              // B: t12_gemm's batch; grouped: the largest seg_B
    int act_stride;
    int ksplit;                            // workgroups along K
    int kslice;                            // columns per K split (multiple of KC)
    int m_total;                           // sum of M over segments
    const uint16_t* act;
    float* ws;                             // partial sums when ksplit > 1
    uint16_t* out_bf16;                    // SwiGLU mode: bf16 [B, out_bf16_ld], silu(seg 2i) * seg 2i+1 of pair i
    int out_bf16_ld;
    float act_a, act_b;                    // EPI launches: the constants of the unary function
    T12Glu glu = t12_silu_glu();           // SwiGLU mode: the unit
    int npair = 1;                         // SwiGLU mode: (gate, up) pairs of the launch; blk_start[i] = first tile of pair i
    // Rows per group known on the device only (the experts of a mixture-of-experts layer, counted by the routing
    // kernel): group_of_seg[s] picks an entry of dev_counts / dev_base, the segment's batch is dev_counts[.] and its
    // activations, outputs (fp32 and bf16) start dev_base[.] rows into the pointers given.  The grid then has one
    // workgroup per row tile, which walks the group's batch tiles.  nullptr: seg_B as given.
    const int* dev_counts = nullptr;
    const int* dev_base = nullptr;
    int group_of_seg[GMAX];
    int n_first = 0;                       // mixed small-batch launch: segments [0, n_first) take the larger workgroups
};

__device__ __forceinline__ int find_segment(const GemmParams& p, int tile)
{
    int s = 0;
#pragma unroll
    for (int i = 1; i < GMAX; i++)
        if (i < p.nseg && tile >= p.blk_start[i]) s = i;
    return s;
}
__device__ __forceinline__ int find_pair(const GemmParams& p, int tile)
{
    int s = 0;
#pragma unroll
    for (int i = 1; i < GMAX / 2; i++)
        if (i < p.npair && tile >= p.blk_start[i]) s = i;
    return s;
}

}  // namespace
