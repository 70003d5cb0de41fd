// Generalized delta rule (T12DeltaRule, t12_mixers.h): per head a [dim, dim] fp32 state, per token
//     S <- diag(w) S - (a u) (u^T S) + k v^T,   o = S^T r.
//
// A value channel's column of S never meets another one, so columns are spread over waves and the time axis is walked
// inside a wave: sixteen lanes (one DPP row) own one column, lane l the key channels RL l .. RL l + RL - 1, so a reduction
// over the key channels is RL multiply-adds and four DPP additions.  States are stored [value channel][key channel] to
// match: a wave reads and writes whole lines.
//
// Everything a token contributes is the same for all columns of a head but for its one value; a preparation kernel forms it
// once per token and head and leaves it in a workspace.  The output is taken from the OLD state as well,
// S_new^T r = S^T (w r) - (r . a u) (u^T S) + (r . k) v, so that of a token's two reductions only u^T S is in the way of
// the next token; the other one is put off and taken for sixteen tokens at once.

#include <mutex>

#include "delta_rule.h"
#include "t12_act.h"
#include "t12_device.h"
#include "t12_host.h"

using namespace delta_rule;

namespace {

// Workgroup = 16 tokens of one head.  Dynamic LDS: tanh(w1) [rank][16].
constexpr int PREP_TOK = 16;
template <int DP>
__global__ __launch_bounds__(256) void delta_prep_kernel(const DeltaParams p)
{
    extern __shared__ float4 th4[];
    float* th = (float*)th4;
    __shared__ float inv[PREP_TOK], dots[PREP_TOK][DP / 64][2];   // r . (a u), r . k of every token by stretches of 64 channels
    const T12DeltaRule& d = p.d;
    const int head = blockIdx.y, t0 = blockIdx.x * PREP_TOK, nt = min(PREP_TOK, p.n - t0);
    const int tid = threadIdx.x, D = d.dim, rank = d.rank, HD = d.heads * D;
    for (int i = tid; i < PREP_TOK * rank; i += 256) {
        const int c = d.w1_off + i % rank, t = min(i / rank, nt - 1);
        th[(i % rank) * PREP_TOK + i / rank] = tanhf(p.in[(size_t)(t0 + t) * p.ld + c] + p.bias[c]);
    }
    {
        const int t = tid >> 4, l = tid & 15;              // sixteen lanes per token
        float ss = 0.0f;
        if (t < nt)
            for (int i = l; i < D; i += 16) {
                const int c = d.k_off + head * D + i;
                const float k = p.in[(size_t)(t0 + t) * p.ld + c] + p.bias[c];
                ss += k * k;
            }
        ss = row_sum16(ss);
        if (l == 0) inv[t] = 1.0f / sqrtf(ss + d.unit_eps);
    }
    __syncthreads();
    constexpr int GRP = DP >= 256 ? 1 : 256 / DP;          // token groups side by side
    constexpr int PER = PREP_TOK / GRP;
    const int grp = DP >= 256 ? 0 : tid / DP;
    for (int i = DP >= 256 ? tid : tid % DP; i < DP; i += 256) {
        const int hc = head * D + min(i, D - 1);
        // everything the channel takes from its tokens is requested ahead of the sum over the rank
        float k[PER], a[PER], rr[PER], v[PER];
        const float* x = p.in + (size_t)(t0 + grp * PER) * p.ld;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const float* y = x + (size_t)min(j, max(nt - 1 - grp * PER, -grp * PER)) * p.ld;     // (clamped to the tokens there are)
            k[j] = y[d.k_off + hc];
            a[j] = y[d.a_off + hc];
            rr[j] = y[d.r_off + hc];
            v[j] = y[d.v_off + hc];
        }
        float z[PER];
        const float w0 = d.w0[hc];
#pragma unroll
        for (int j = 0; j < PER; j++) z[j] = 0.0f;
#pragma unroll 16
        for (int r = 0; r < rank; r++) {
            const float w = d.w2t[(size_t)r * HD + hc];
#pragma unroll
            for (int j = 0; j < PER; j++) z[j] += w * th[r * PREP_TOK + grp * PER + j];
        }
        const float bk = p.bias[d.k_off + hc], ba = p.bias[d.a_off + hc], br = p.bias[d.r_off + hc], bv = p.bias[d.v_off + hc];
        const float one = i < D ? 1.0f : 0.0f;             // channels past the head's size: zero records
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int t = grp * PER + j;
            const float kk = (k[j] + bk) * one, u = kk * inv[t], au = t12_sigmoid(a[j] + ba) * u;
            const float w = expf(-d.decay_rate * t12_sigmoid(z[j] + w0)) * one, ri = (rr[j] + br) * one;
            if (t < nt) {
                float* rec = p.rec + ((size_t)(t0 + t) * d.heads + head) * rec_floats(DP) + i;
                rec[0] = u;
                rec[DP] = au;
                rec[2 * DP] = w;
                rec[3 * DP] = kk;
                rec[4 * DP] = ri * w;
                rec[5 * DP] = (v[j] + bv) * one;
            }
            // (whole waves share a token: DP is a multiple of 64)
            const float ra = t12_wave_sum_lane63(ri * au), rk = t12_wave_sum_lane63(ri * kk);
            if ((tid & 63) == 63) {
                dots[t][i / 64][0] = ra;
                dots[t][i / 64][1] = rk;
            }
        }
    }
    __syncthreads();
    if (tid < nt * 2) {
        float v = 0.0f;
#pragma unroll
        for (int q = 0; q < DP / 64; q++) v += dots[tid / 2][q][tid % 2];
        p.rec[((size_t)(t0 + tid / 2) * d.heads + head) * rec_floats(DP) + (NREC + 1) * DP + tid % 2] = v * 0.0625f;
    }
}

// Rows that are sequences of their own: one token each.  Workgroup = 256 threads = sixteen columns of one head of one row.
template <int RL>
__global__ __launch_bounds__(256) void delta_token_kernel(const DeltaParams p)
{
    const T12DeltaRule& d = p.d;
    const int row = blockIdx.x, head = blockIdx.y, group = blockIdx.z * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (group * 4 >= d.dim) return;
    Columns<RL> C;
    C.load(d, p.rows[row], head, group);
    Token<RL> t;
    t.read(p.rec + ((size_t)row * d.heads + head) * rec_floats(RL * 16), C.l, C.jc);
    const float y = row_sum16(t.advance(C));
    if (C.live && C.l == 0) p.o[((size_t)row * d.heads + head) * d.dim + C.j] = y;
    C.store();
}

// A run of tokens of one sequence.  Workgroup = two waves = eight columns of one head, so that the heads of a model spread
// over the chip.  The records of CH tokens are brought into LDS together, the next CH are on their way meanwhile; the
// outputs of sixteen tokens are added up across the lanes at once.  Dynamic LDS: run_lds_bytes().
template <int RL, int CH>
constexpr size_t run_lds_bytes()
{
    return (size_t)2 * ((CH * rec_floats(RL * 16) / 4 + 127) / 128) * 128 * 16;
}
template <int RL, int CH>
__global__ __launch_bounds__(128) void delta_run_kernel(const DeltaParams p)
{
    constexpr int DP = RL * 16, RF = rec_floats(DP), PIECES = CH * RF / 4, NP = (PIECES + 127) / 128;
    static_assert(CH % 16 == 0, "outputs are added up sixteen tokens at a time");
    extern __shared__ float4 lds4[];
    float* lds = (float*)lds4;
    const T12DeltaRule& d = p.d;
    const int head = blockIdx.x, tid = threadIdx.x, len = p.n;
    const int group = blockIdx.y * 2 + __builtin_amdgcn_readfirstlane(tid >> 6);
    Columns<RL> C;
    C.load(d, p.rows[0], head, min(group, (d.dim - 1) / 4));
    C.live = C.live && group * 4 < d.dim;                  // (a wave past the end works on the last columns and stores nothing)
    const float* rec = p.rec + (size_t)head * RF;
    const size_t rec_step = (size_t)d.heads * RF;
    float* o = p.o + (size_t)head * d.dim + C.j;
    const size_t o_step = (size_t)d.heads * d.dim;
    const int chunks = len / CH;
    // piece q of a chunk = 16 bytes of token q / (RF / 4); a thread's pieces lie at fixed offsets from the chunk's first record
    uint32_t from[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int q = min(tid + i * 128, PIECES - 1);
        from[i] = (uint32_t)((q / (RF / 4)) * rec_step + (q % (RF / 4)) * 4);
    }
    t12_f32x4 ahead[NP];
#define T12_REQUEST(c)                                                                        \
    {                                                                                         \
        const float* base_ = rec + (size_t)(c) * CH * rec_step;                               \
        _Pragma("unroll") for (int i = 0; i < NP; i++) ahead[i] = *(const t12_f32x4*)(base_ + from[i]); \
    }
    if (chunks > 0) T12_REQUEST(0)
    for (int c = 0; c < chunks; c++) {
        t12_f32x4* buf = (t12_f32x4*)lds4 + (c & 1) * (NP * 128);
#pragma unroll
        for (int i = 0; i < NP; i++) buf[tid + i * 128] = ahead[i];
        __syncthreads();                                   // (the other buffer was last read before the previous barrier)
        if (c + 1 < chunks) T12_REQUEST(c + 1)
        const float* x = lds + (size_t)(c & 1) * (NP * 128 * 4);
        Token<RL> t[2];
        t[0].read(x, C.l, C.jc);
#pragma unroll
        for (int s = 0; s < CH; s += 16) {
            float y[16];
#pragma unroll
            for (int f = 0; f < 16; f++) {
                const int at = s + f;
                if (at + 1 < CH) t[(at + 1) & 1].read(x + (at + 1) * RF, C.l, C.jc);
                y[f] = t[at & 1].advance(C);
                __builtin_amdgcn_sched_barrier(0);         // (a token's reads stay one token ahead)
            }
            const float v = transpose_sum16(y, C.l);
            if (C.live) o[(size_t)(c * CH + s + C.l) * o_step] = v;
        }
    }
#undef T12_REQUEST
    for (int t = chunks * CH; t < len; t++) {              // the last tokens straight from memory
        Token<RL> tok;
        tok.read(rec + (size_t)t * rec_step, C.l, C.jc);
        const float y = row_sum16(tok.advance(C));
        if (C.live && C.l == 0) o[(size_t)t * o_step] = y;
    }
    C.store();
}

// The same without LDS, for heads whose records are too large for it.
template <int RL>
__global__ __launch_bounds__(64) void delta_run_direct_kernel(const DeltaParams p)
{
    const T12DeltaRule& d = p.d;
    const int head = blockIdx.x;
    Columns<RL> C;
    C.load(d, p.rows[0], head, blockIdx.y);
    for (int t = 0; t < p.n; t++) {
        Token<RL> tok;
        tok.read(p.rec + ((size_t)t * d.heads + head) * rec_floats(RL * 16), C.l, C.jc);
        const float y = row_sum16(tok.advance(C));
        if (C.live && C.l == 0) p.o[((size_t)t * d.heads + head) * d.dim + C.j] = y;
    }
    C.store();
}

// One wave per (row, head): o over its RMS, times the plain weight and the sigmoid gate.
template <bool F32>
__global__ __launch_bounds__(256) void delta_out_kernel(const DeltaParams p)
{
    const T12DeltaRule& d = p.d;
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (item >= p.n * d.heads) return;
    const int row = item / d.heads, head = item % d.heads, D = d.dim;
    const float* o = p.o + (size_t)item * D;
    float ss = 0.0f;
    for (int i = lane; i < D; i += 64) ss += o[i] * o[i];
    const float rn = 1.0f / sqrtf(t12_wave_sum(ss) / (float)D + d.out_eps);
    for (int i = lane; i < D; i += 64) {
        const int hc = head * D + i;
        const float g = p.in[(size_t)row * p.ld + d.g_off + hc] + p.bias[d.g_off + hc];
        const float v = o[i] * rn * d.norm_w[hc] * t12_sigmoid(g) * p.out_scale;
        if (F32) ((float*)p.out)[(size_t)row * p.out_ld + hc] = v;
        else ((uint16_t*)p.out)[(size_t)row * p.out_ld + hc] = t12_f32_to_bf16(v);
    }
}

template <int RL, int CH>
int launch_rule(const DeltaParams& p, hipStream_t st)
{
    hipLaunchKernelGGL((delta_prep_kernel<RL * 16>), dim3((p.n + PREP_TOK - 1) / PREP_TOK, p.d.heads), dim3(256),
                       (size_t)PREP_TOK * p.d.rank * sizeof(float), st, p);
    if (!p.run) {
        hipLaunchKernelGGL(delta_token_kernel<RL>, dim3(p.n, p.d.heads, (p.d.dim + 15) / 16), dim3(256), 0, st, p);
    } else if constexpr (CH > 0) {
        constexpr size_t lds = run_lds_bytes<RL, CH>();
        if (lds > 64 * 1024) {
            static std::once_flag once[16];                // the attribute is per device
            int dev = 0;
            if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) dev = 0;
            hipError_t e = hipSuccess;
            std::call_once(once[dev], [&] { e = hipFuncSetAttribute((const void*)delta_run_kernel<RL, CH>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
            if (e != hipSuccess) {
                t12_set_error("t12_delta_rule: cannot reserve %zu bytes of LDS", lds);
                return T12_ELAUNCH;
            }
        }
        hipLaunchKernelGGL((delta_run_kernel<RL, CH>), dim3(p.d.heads, (p.d.dim + 7) / 8), dim3(128), lds, st, p);
    } else {
        hipLaunchKernelGGL(delta_run_direct_kernel<RL>, dim3(p.d.heads, (p.d.dim + 3) / 4), dim3(64), 0, st, p);
    }
    T12_CHECK_LAUNCH("t12_delta_rule");
    return T12_OK;
}

}  // namespace

extern "C" {

int t12_delta_plan(T12DeltaRule* d)
{
    T12_REQUIRE(d && d->heads >= 1 && d->dim >= 1 && d->dim <= 512 && d->rank >= 1 && d->rank <= 512,
                "t12_delta_plan: heads %d, dim %d (1..512) or rank %d (1..512) out of range", d ? d->heads : 0, d ? d->dim : 0,
                d ? d->rank : 0);
    d->dim_p = 64;
    while (d->dim_p < d->dim) d->dim_p *= 2;
    d->state_elems = (size_t)d->heads * d->dim * d->dim_p;
    d->work_elems = (size_t)d->heads * (rec_floats(d->dim_p) + d->dim);
    return T12_OK;
}

int t12_delta_rule(const T12DeltaRule* d, const float* in, const float* bias, int ld, const T12Row* rows, int n, int run,
                   float out_scale, float* work, void* out, int out_f32, int out_ld, void* stream)
{
    T12_REQUIRE(d && in && bias && rows && work && out && d->state && d->w2t && d->w0 && d->norm_w && n >= 1,
                "t12_delta_rule: null operand or no rows");
    T12_REQUIRE(d->dim_p >= d->dim && d->dim_p % 64 == 0 && d->state_elems == (size_t)d->heads * d->dim * d->dim_p,
                "t12_delta_rule: t12_delta_plan has not been called");
    const int HD = d->heads * d->dim;
    for (int off : {d->r_off, d->k_off, d->v_off, d->a_off, d->g_off})
        T12_REQUIRE(off >= 0 && off + HD <= ld, "t12_delta_rule: columns %d + %d outside a row of %d", off, HD, ld);
    T12_REQUIRE(d->w1_off >= 0 && d->w1_off + d->rank <= ld && out_ld >= HD, "t12_delta_rule: row strides too small");
    hipStream_t st = (hipStream_t)stream;
    DeltaParams p;
    p.d = *d;
    p.in = in;
    p.bias = bias;
    p.ld = ld;
    p.rows = rows;
    p.n = n;
    p.run = run;
    p.out_scale = out_scale;
    p.rec = work;
    p.o = work + (size_t)n * d->heads * rec_floats(d->dim_p);
    p.out = out;
    p.out_ld = out_ld;
    int rc;
    switch (d->dim_p) {
        // (tokens between two barriers: handing a chunk over costs a wave that is alone on its SIMD about 1 us.  512 tokens, 16
        // heads of 64: 81 us with 16, 66 us with 32, 100 KB of LDS; heads of 128 have room for 16)
        case 64: rc = launch_rule<4, 32>(p, st); break;
        case 128: rc = launch_rule<8, 16>(p, st); break;
        case 256: rc = launch_rule<16, 0>(p, st); break;
        default: rc = launch_rule<32, 0>(p, st); break;
    }
    if (rc) return rc;
    const int items = n * d->heads;
    if (out_f32) hipLaunchKernelGGL(delta_out_kernel<true>, dim3((items + 3) / 4), dim3(256), 0, st, p);
    else hipLaunchKernelGGL(delta_out_kernel<false>, dim3((items + 3) / 4), dim3(256), 0, st, p);
    T12_CHECK_LAUNCH("t12_delta_rule(out)");
    return T12_OK;
}

}  // extern "C"
