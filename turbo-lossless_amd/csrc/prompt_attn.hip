// Attention of a prompt pass over an INT8 cache: the rows of the pass are consecutive positions of one sequence whose
// K / V are in the cache already, and row t attends to positions <= its own.  Same function as the decode kernels of
// glue.hip (engine/kernels.hip:499-586) row by row; those read the cache once per row, here 64 (token, query head) pairs
// of a KV group share what is read.
//
// What bounds it is the work per score (about 17 VALU operations, two of three of them for the exponential and for
// splitting the weight), not memory: 512 rows at 1536 .. 2047 positions are 29 M scores per layer and touch 4 MB.
//   * Workgroup = (64 pairs, KV head), eight waves: two of 32 pairs each x four that take 32 of every 128 positions.
//     The four keep maxima, sums and outputs of their own and are put together at the end, so 512 rows of 32 heads are 256
//     workgroups with two waves per SIMD.
//   * Scores transposed, S^T = K Q^T, by v_mfma_i32_32x32x32_i8: K as stored, Q in three INT8 limbs, exact int32 sums.
//     A lane then holds 16 positions of ONE pair: maxima and sums need one exchange with the lane 32 further on.
//   * out^T = V^T P^T by v_mfma_f32_32x32x16_bf16: the lane's 16 weights p * v_scale are its B operand without a
//     move, as two bf16 each (16 bits, relative to the weight itself; the decode kernels: 15 bits relative to the
//     largest).  V is turned into bf16 (exact) and around on its way to LDS.
//   * Outputs are rescaled only when some pair's maximum has grown.
// Measured at 512 rows, 32 / 8 heads of 128: 17.7 / 27.8 / 37.3 / 46.5 us at
// first position 0 / 512 / 1024 / 1536 (the row by row kernels: 51.4 / 109 / 167 / 223), outputs as close to 64 bits
#include <hip/hip_runtime.h>

#include <type_traits>

#include "t12_device.h"
#include "t12_host.h"

namespace {

typedef int pa_i32x4 __attribute__((ext_vector_type(4)));
typedef int pa_i32x16 __attribute__((ext_vector_type(16)));

constexpr int PA_PAIRS = 64;             // (token, head) pairs of a workgroup
constexpr int PA_STEP = 128;             // positions of a step

struct PromptAttn {
    const float* q;                      // [rows][heads * HD], rotated
    const int8_t* ck;
    const int8_t* cv;
    const float* sk;
    const float* sv;
    uint16_t* out;                       // bf16 [rows][heads * HD]
    int rows, first;                     // row r is at position first + r
    int n_head, n_head_kv, log_ratio;
    float scale;
    size_t row_stride, head_off;         // cache: bytes between positions, between KV heads
    int sc_stride;                       // scales: elements between positions
    size_t sc_head;                      //         between KV heads
};

// bytes j of a and b (signed) as a pair of bf16
__device__ __forceinline__ uint32_t pa_pair_bf16(uint32_t a, uint32_t b, int j)
{
    const float x = (float)(int8_t)(a >> (8 * j)), y = (float)(int8_t)(b >> (8 * j));
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, y), __builtin_bit_cast(uint32_t, x), 0x07060302u);   // (exact: the low halves are zero)
}

// two floats rounded to bf16 (nearest even), x in the low half
__device__ __forceinline__ uint32_t pa_round2(float x, float y)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x, y}, t12_bf16x2));
}

template <int HD>
__global__ __launch_bounds__(512, 2) void prompt_attn_kernel(const PromptAttn a)
{
    constexpr int KS = HD / 32;              // score MFMAs per limb
    constexpr int DT = HD / 32;              // tiles of 32 output dims
    constexpr int KROW = HD, VROW = PA_STEP * 2;
    constexpr int KP = HD / 16;              // 16-byte pieces of a K row
    constexpr int KLD = PA_STEP * KP / 512;  // of them, per thread and step
    constexpr int VD = HD / 16;              // dims a thread turns around (4 positions x VD dims)
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * (PA_STEP * KROW + HD * VROW) + 2 * 2 * PA_STEP * 4];
    uint8_t* const lk = lds;                                      // [2][PA_STEP][KROW]
    uint8_t* const lv = lds + 2 * PA_STEP * KROW;                 // [2][HD][VROW]
    float* const lks = (float*)(lds + 2 * (PA_STEP * KROW + HD * VROW));     // [2][PA_STEP] K scales, then V scales
    float* const lvs = lks + 2 * PA_STEP;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, h = lane >> 5;
    const int qw = wave & 1, kg = wave >> 1;                      // which pairs, which positions of a step
    const int kvh = blockIdx.y;
    const int block = gridDim.x - 1 - blockIdx.x;                 // the longest rows first
    const int tokens = PA_PAIRS >> a.log_ratio;
    const int ratio = 1 << a.log_ratio;
    const int row0 = block * tokens;
    const int pair = 32 * qw + n;
    const int row = row0 + (pair >> a.log_ratio);
    const int rrow = min(row, a.rows - 1);                        // rows past the end: computed, not stored
    const int head = kvh * ratio + (pair & (ratio - 1));
    const int pos = a.first + rrow;
    const int last = a.first + min(row0 + tokens, a.rows) - 1;    // last position any pair of the workgroup sees
    const int steps = last / PA_STEP + 1;

    const int8_t* const kb = a.ck + (size_t)kvh * a.head_off;
    const int8_t* const vb = a.cv + (size_t)kvh * a.head_off;
    const float* const skb = a.sk + (size_t)kvh * a.sc_head;
    const float* const svb = a.sv + (size_t)kvh * a.sc_head;

    // ---- staging: K pieces as stored, V turned around as bf16
    t12_u32x4 rk[KLD];
    uint32_t rv[4][VD / 4];
    float rs = 0.0f;
    const int v_d0 = (tid & 15) * VD, v_p4 = tid >> 4;            // 4 positions from 4 v_p4 on, VD dims from v_d0 on
    auto request = [&](int s) __attribute__((always_inline)) {
        const int t0 = s * PA_STEP;
#pragma unroll
        for (int i = 0; i < KLD; i++) {
            const int idx = tid + 512 * i, t = min(t0 + idx / KP, last);
            rk[i] = *(const t12_u32x4*)(kb + (size_t)t * a.row_stride + (idx % KP) * 16);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int t = min(t0 + 4 * v_p4 + j, last);
            const uint32_t* src = (const uint32_t*)(vb + (size_t)t * a.row_stride + v_d0);
#pragma unroll
            for (int w = 0; w < VD / 4; w++) rv[j][w] = src[w];
        }
        if (tid < 2 * PA_STEP) {
            const int t = min(t0 + (tid & (PA_STEP - 1)), last);
            rs = tid < PA_STEP ? skb[(size_t)t * a.sc_stride] : svb[(size_t)t * a.sc_stride];
        }
    };
    // K row t: piece p in slot p ^ swizzle(t); V: dim d's row of 128 positions in 16-byte units, unit 2 (t / 16) + hh holds
    // positions 4 hh .. and 8 + 4 hh .. of its sixteen (what lane half hh multiplies), in slot unit ^ (d ^ d / 8) % 16:
    // neither the reads nor the writes of 16 neighbouring lanes meet in a bank
    auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KLD; i++) {
            const int idx = tid + 512 * i, t = idx / KP, p = idx % KP;
            const int sw = ((t & 7) ^ ((t >> 3) & 1)) & (KP - 1);
            *(t12_u32x4*)(lk + buf * (PA_STEP * KROW) + t * KROW + 16 * (p ^ sw)) = rk[i];
        }
        const int unit = 2 * (v_p4 >> 2) + (v_p4 & 1), half = (v_p4 >> 1) & 1;
#pragma unroll
        for (int w = 0; w < VD / 4; w++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int d = v_d0 + 4 * w + j;
                const uint2 v = make_uint2(pa_pair_bf16(rv[0][w], rv[1][w], j), pa_pair_bf16(rv[2][w], rv[3][w], j));
                *(uint2*)(lv + buf * (HD * VROW) + d * VROW + 16 * (unit ^ ((d ^ (d >> 3)) & 15)) + 8 * half) = v;
            }
        if (tid < 2 * PA_STEP) (tid < PA_STEP ? lks : lvs)[buf * PA_STEP + (tid & (PA_STEP - 1))] = rs;
    };
    request(0);

    // ---- Q: q ~ s (a1 + a2 / 254 + a3 / 254^2), s = max|q| / 127 (error 6e-8 max|q|).  Lane (pair, h) of group kg makes the
    //      limbs of dims h HD / 2 + 16 kg .. (one operand piece); they meet in the buffers of step 1, which are free so far.
    pa_i32x4 Q[3][KS];
    float qf;                                                     // scores in units of log2
    {
        pa_i32x4* const ql = (pa_i32x4*)lds + 2 * PA_STEP;        // [3][KS][2][64 pairs], behind step 0's K rows and ...
        uint32_t* const qmax = (uint32_t*)lds;                    // ... before them (nothing is staged yet): [KS][64 pairs]
        float v[16];
        if (kg < KS) {
            const float* src = a.q + ((size_t)rrow * a.n_head + head) * HD + h * (HD / 2) + 16 * kg;
            uint32_t amax = 0;                                    // (bits of |q|: ordered like the values, NaN last)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const t12_f32x4 x = *(const t12_f32x4*)(src + 4 * i);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    v[4 * i + j] = x[j];
                    amax = max(amax, __float_as_uint(v[4 * i + j]) & 0x7FFFFFFFu);
                }
            }
            amax = max(amax, (uint32_t)__shfl_xor((int)amax, 32, T12_WAVE));
            if (h == 0) qmax[kg * PA_PAIRS + pair] = amax;
        }
        __syncthreads();
        uint32_t abits = qmax[pair];
#pragma unroll
        for (int u = 1; u < KS; u++) abits = max(abits, qmax[u * PA_PAIRS + pair]);
        const float amax = __builtin_bit_cast(float, abits);
        const float inv = amax > 0.0f ? 127.0f / amax : 0.0f;
        // an all-zero query: every score 0, the factor only has to keep masked positions at minus infinity; an infinity or
        // NaN in the query: NaN out
        qf = abits >= 0x7F800000u ? __builtin_nanf("")
                                  : (abits ? amax / 127.0f * a.scale * 1.44269504088896340736f : 1e-30f);
        if (kg < KS) {
            pa_i32x4 limb[3];
#pragma unroll
            for (int w = 0; w < 4; w++) {
                uint32_t l1 = 0, l2 = 0, l3 = 0;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float r0 = v[4 * w + j] * inv;
                    const float a1 = fminf(fmaxf(rintf(r0), -127.0f), 127.0f);
                    const float r1 = (r0 - a1) * 254.0f;
                    const float a2 = fminf(fmaxf(rintf(r1), -127.0f), 127.0f);
                    const float a3 = fminf(fmaxf(rintf((r1 - a2) * 254.0f), -127.0f), 127.0f);
                    l1 |= ((uint32_t)(int)a1 & 0xFFu) << (8 * j);
                    l2 |= ((uint32_t)(int)a2 & 0xFFu) << (8 * j);
                    l3 |= ((uint32_t)(int)a3 & 0xFFu) << (8 * j);
                }
                limb[0][w] = (int)l1;
                limb[1][w] = (int)l2;
                limb[2][w] = (int)l3;
            }
#pragma unroll
            for (int i = 0; i < 3; i++) ql[((i * KS + kg) * 2 + h) * PA_PAIRS + pair] = limb[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int u = 0; u < KS; u++) Q[i][u] = ql[((i * KS + u) * 2 + h) * PA_PAIRS + pair];
        __syncthreads();
    }

    float m = -1e30f, l = 0.0f;                                   // running maximum (before qf), sum of this lane's half
    t12_f32x16 acc[DT];
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[d][r] = 0.0f;

    store(0);
    __syncthreads();
    for (int s = 0; s < steps; s++) {
        const int buf = s & 1;
        if (s + 1 < steps) request(s + 1);
        const int t0 = s * PA_STEP + 32 * kg;                     // this wave's 32 positions
        if (t0 <= last) {
            // scores of positions 8 (r / 4) + 4 h + r % 4
            const uint8_t* krow = lk + buf * (PA_STEP * KROW) + (32 * kg + n) * KROW;
            const int sw = ((n & 7) ^ ((n >> 3) & 1)) & (KP - 1);
            pa_i32x16 s1, s2, s3;
#pragma unroll
            for (int r = 0; r < 16; r++) s1[r] = s2[r] = s3[r] = 0;
#pragma unroll
            for (int u = 0; u < KS; u++) {
                const pa_i32x4 K = *(const pa_i32x4*)(krow + 16 * ((h * KS + u) ^ sw));
                s1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(K, Q[0][u], s1, 0, 0, 0);
                s2 = __builtin_amdgcn_mfma_i32_32x32x32_i8(K, Q[1][u], s2, 0, 0, 0);
                s3 = __builtin_amdgcn_mfma_i32_32x32x32_i8(K, Q[2][u], s3, 0, 0, 0);
            }
            float x[16];
            const float* ks = lks + buf * PA_STEP + 32 * kg + 4 * h;
            const float* vs = lvs + buf * PA_STEP + 32 * kg + 4 * h;
#pragma unroll
            for (int r = 0; r < 16; r++)
                x[r] = ((float)s1[r] + (float)(__mul24(s2[r], 254) + s3[r]) * (1.0f / 64516.0f)) * ks[8 * (r >> 2) + (r & 3)];   // (|s2| < 2^22)
            const bool edge = t0 + 31 > a.first + row0;           // some pair does not see all of them
            if (edge) {
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (t0 + 8 * (r >> 2) + 4 * h + (r & 3) > pos) x[r] = -__builtin_inff();
            }
            float mx = x[0];
#pragma unroll
            for (int r = 1; r < 16; r++) mx = fmaxf(mx, x[r]);
            mx = fmaxf(mx, __shfl_xor(mx, 32, T12_WAVE));
            if (__any(mx > m)) {
                const float mn = fmaxf(m, mx);
                const float c = __builtin_amdgcn_exp2f((m - mn) * qf);
                m = mn;
                l *= c;
#pragma unroll
                for (int d = 0; d < DT; d++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[d][r] *= c;
            }
            // weights: p in the sum, p * v_scale as two bf16 in the products
            const float mq = fmaxf(m * qf, -3e38f);
            uint32_t hi[8], lo[8];
            auto weights = [&](auto edge) __attribute__((always_inline)) {
#pragma unroll
                for (int r = 0; r < 16; r += 2) {
                    float w[2];
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const int o = 8 * ((r + j) >> 2) + ((r + j) & 3);
                        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(x[r + j], qf, -mq));
                        l += p;
                        w[j] = p * vs[o];
                        if (edge.value && t0 + 4 * h + o > pos) w[j] = 0.0f;   // (a scale out of sight may be an infinity)
                    }
                    hi[r >> 1] = pa_round2(w[0], w[1]);
                    lo[r >> 1] = pa_round2(w[0] - __builtin_bit_cast(float, hi[r >> 1] << 16),
                                           w[1] - __builtin_bit_cast(float, hi[r >> 1] & 0xFFFF0000u));
                }
            };
            if (edge) weights(std::true_type{});
            else weights(std::false_type{});
            const uint8_t* vt = lv + buf * (HD * VROW);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const t12_bf16x8 ph = __builtin_bit_cast(t12_bf16x8, make_uint4(hi[4 * j], hi[4 * j + 1], hi[4 * j + 2], hi[4 * j + 3]));
                const t12_bf16x8 pl = __builtin_bit_cast(t12_bf16x8, make_uint4(lo[4 * j], lo[4 * j + 1], lo[4 * j + 2], lo[4 * j + 3]));
#pragma unroll
                for (int d = 0; d < DT; d++) {
                    const int dim = 32 * d + n, unit = 2 * (2 * kg + j) + h;
                    const t12_bf16x8 v = *(const t12_bf16x8*)(vt + dim * VROW + 16 * (unit ^ ((dim ^ (dim >> 3)) & 15)));
                    acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, ph, acc[d], 0, 0, 0);
                    acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, pl, acc[d], 0, 0, 0);
                }
            }
        }
        if (s + 1 < steps) store(buf ^ 1);                        // (last read two barriers ago)
        __syncthreads();
    }
    l += __shfl_xor(l, 32, T12_WAVE);

    // ---- the four position groups of a pair put together: out = sum_g e^(m_g - M) acc_g / sum_g e^(m_g - M) l_g.  Through
    //      LDS in two halves of the dims (the staging buffers hold one).
    float* const fm = (float*)lds;                                // [4][64 pairs] m, then l
    float* const fl = fm + 4 * PA_PAIRS;
    float* const fa = fl + 4 * PA_PAIRS;                          // [3][2][DT / 2 * 16][64 lanes]
    if (h == 0) {
        fm[kg * PA_PAIRS + pair] = m;
        fl[kg * PA_PAIRS + pair] = l;
    }
    __syncthreads();
    float M = fm[pair], L = 0.0f, own = 0.0f;
#pragma unroll
    for (int g = 1; g < 4; g++) M = fmaxf(M, fm[g * PA_PAIRS + pair]);
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const float e = __builtin_amdgcn_exp2f((fm[g * PA_PAIRS + pair] - M) * qf);
        L += e * fl[g * PA_PAIRS + pair];
        if (g == kg) own = e;
    }
    const float inv = L > 0.0f ? own / L : 0.0f;
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[d][r] *= inv;
    constexpr int HT = DT / 2;                                    // dim tiles per half
#pragma unroll
    for (int half = 0; half < 2; half++) {
        if (kg > 0) {
#pragma unroll
            for (int d = 0; d < HT; d++)
#pragma unroll
                for (int r = 0; r < 16; r++) fa[(((kg - 1) * 2 + qw) * (HT * 16) + d * 16 + r) * 64 + lane] = acc[half * HT + d][r];
        }
        __syncthreads();
        if (kg == 0 && row < a.rows) {
            uint16_t* o = a.out + ((size_t)row * a.n_head + head) * HD + half * (HD / 2);
#pragma unroll
            for (int d = 0; d < HT; d++)
#pragma unroll
                for (int r4 = 0; r4 < 4; r4++) {
                    uint16_t b[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        float v = acc[half * HT + d][4 * r4 + j];
#pragma unroll
                        for (int g = 0; g < 3; g++) v += fa[((g * 2 + qw) * (HT * 16) + d * 16 + 4 * r4 + j) * 64 + lane];
                        b[j] = t12_f32_to_bf16(v);
                    }
                    *(uint2*)(o + 32 * d + 8 * r4 + 4 * h) = make_uint2(b[0] | ((uint32_t)b[1] << 16), b[2] | ((uint32_t)b[3] << 16));
                }
        }
        __syncthreads();
    }
}

}  // namespace

// Library-internal (glue.hip): shapes and addresses the kernel takes.
extern "C" __attribute__((visibility("hidden"))) bool t12_prompt_attention_takes(
    const float* q, const int8_t* ck, const int8_t* cv, const int16_t* out, int rows, int first, int n_head, int n_head_kv,
    int head_dim, float scale)
{
    if (n_head_kv < 1 || n_head % n_head_kv || (head_dim != 64 && head_dim != 128)) return false;
    const int ratio = n_head / n_head_kv;
    if (ratio < 1 || ratio > 8 || (ratio & (ratio - 1)) || rows < 1 || first < 0 || !(scale > 0.0f)) return false;
    return (uintptr_t)q % 16 == 0 && (uintptr_t)ck % 16 == 0 && (uintptr_t)cv % 16 == 0 && (uintptr_t)out % 8 == 0;
}

// Library-internal (glue.hip): out[r] = attention of row r at position first + r over positions 0 .. first + r of one
// cache region, all of them stored, for what the rule above takes.  hm as in glue.hip: 0 = [position][kv head][dim], > 0 =
// [kv head][hm][dim].
extern "C" __attribute__((visibility("hidden"))) void t12_prompt_attention(
    const float* q, const int8_t* ck, const int8_t* cv, const float* sk, const float* sv, int16_t* out, int rows, int first,
    int n_head, int n_head_kv, int head_dim, float scale, int hm, hipStream_t st)
{
    const int ratio = n_head / n_head_kv;
    PromptAttn a;
    a.q = q;
    a.ck = ck;
    a.cv = cv;
    a.sk = sk;
    a.sv = sv;
    a.out = (uint16_t*)out;
    a.rows = rows;
    a.first = first;
    a.n_head = n_head;
    a.n_head_kv = n_head_kv;
    a.log_ratio = ratio == 1 ? 0 : (ratio == 2 ? 1 : (ratio == 4 ? 2 : 3));
    a.scale = scale;
    a.row_stride = hm ? (size_t)head_dim : (size_t)n_head_kv * head_dim;
    a.head_off = hm ? (size_t)hm * head_dim : (size_t)head_dim;
    a.sc_stride = hm ? 1 : n_head_kv;
    a.sc_head = hm ? (size_t)hm : 1;
    const int tokens = PA_PAIRS / ratio;
    const dim3 grid((rows + tokens - 1) / tokens, n_head_kv);
    if (head_dim == 128) hipLaunchKernelGGL((prompt_attn_kernel<128>), grid, dim3(512), 0, st, a);
    else hipLaunchKernelGGL((prompt_attn_kernel<64>), grid, dim3(512), 0, st, a);
}
