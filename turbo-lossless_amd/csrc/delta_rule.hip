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
//
// Runs of heads of 32 to 64 channels take sixteen tokens at a time instead (delta_plan.h), on the matrix cores.

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "delta_plan.h"
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
// over the chip.  The records of sixteen tokens are brought into LDS together, the next sixteen (or the last few tokens) are on their way
// meanwhile; the outputs of the sixteen are added up across the lanes at once.  Dynamic LDS: run_lds_bytes().
constexpr int RUN_TOK = 16;
template <int RL>
constexpr size_t run_lds_bytes()
{
    return (size_t)2 * ((RUN_TOK * rec_floats(RL * 16) / 4 + 127) / 128) * 128 * 16;
}
// Tokens past the last whole chunk that are worth bringing through LDS: straight from memory each costs 0.68 us, in a chunk 0.12 and
// all together 1.5 us more (16 heads of 64, whole call: 1 / 4 / 15 tokens 10.5 / 13.4 / 18.4 us straight, 11.5 / 13.4 / 14.5 staged).
constexpr int RUN_STAGED_TAIL = 5;
template <int RL>
__global__ __launch_bounds__(128) void delta_run_kernel(const DeltaParams p)
{
    constexpr int CH = RUN_TOK, DP = RL * 16, RF = rec_floats(DP), PIECES = CH * RF / 4, NP = (PIECES + 127) / 128;
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
    const int chunks = len / CH, tail = len % CH;
    // piece q of a chunk = 16 bytes of token q / (RF / 4); a thread's pieces lie at fixed offsets from the chunk's first record.
    // A run that ends inside a chunk brings its last CH tokens again, or all it has.
    const int pieces = min(CH, len) * (RF / 4);
    uint32_t from[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int q = min(tid + i * 128, pieces - 1);
        from[i] = (uint32_t)((q / (RF / 4)) * rec_step + (q % (RF / 4)) * 4);
    }
    t12_f32x4 ahead[NP];
#define T12_REQUEST(c)                                                                       \
    {                                                                                        \
        const float* base_ = rec + (size_t)max(min((c) * CH, len - CH), 0) * rec_step;       \
        _Pragma("unroll") for (int i = 0; i < NP; i++) ahead[i] = *(const t12_f32x4*)(base_ + from[i]); \
    }
    T12_REQUEST(0)
    for (int c = 0; c < chunks; c++) {
        t12_f32x4* buf = (t12_f32x4*)lds4 + (c & 1) * (NP * 128);
#pragma unroll
        for (int i = 0; i < NP; i++) buf[tid + i * 128] = ahead[i];
        __syncthreads();                                   // (the other buffer was last read before the previous barrier)
        T12_REQUEST(c + 1)
        const float* x = lds + (size_t)(c & 1) * (NP * 128 * 4);
        Token<RL> t[2];
        t[0].read(x, C.l, C.jc);
        float y[CH];
#pragma unroll
        for (int f = 0; f < CH; f++) {
            if (f + 1 < CH) t[(f + 1) & 1].read(x + (f + 1) * RF, C.l, C.jc);
            y[f] = t[f & 1].advance(C);
            __builtin_amdgcn_sched_barrier(0);             // (a token's reads stay one token ahead)
        }
        const float v = transpose_sum16(y, C.l);
        if (C.live) o[(size_t)(c * CH + C.l) * o_step] = v;
    }
#undef T12_REQUEST
    if (tail < RUN_STAGED_TAIL) {                          // a few last tokens straight from memory
        for (int t = chunks * CH; t < len; t++) {
            Token<RL> tok;
            tok.read(rec + (size_t)t * rec_step, C.l, C.jc);
            const float y = row_sum16(tok.advance(C));
            if (C.live && C.l == 0) o[(size_t)t * o_step] = y;
        }
    } else {                                               // more of them: the same as a chunk on what there is
        t12_f32x4* buf = (t12_f32x4*)lds4 + (chunks & 1) * (NP * 128);
#pragma unroll
        for (int i = 0; i < NP; i++) buf[tid + i * 128] = ahead[i];
        __syncthreads();
        const float* x = lds + (size_t)(chunks & 1) * (NP * 128 * 4) + (chunks ? CH - tail : 0) * RF;
        Token<RL> t[2];
        t[0].read(x, C.l, C.jc);
        float y[CH];
#pragma unroll
        for (int f = 0; f < CH; f++) {
            y[f] = 0.0f;
            if (f < tail) {
                t[(f + 1) & 1].read(x + min(f + 1, tail - 1) * RF, C.l, C.jc);
                y[f] = t[f & 1].advance(C);
            }
        }
        const float v = transpose_sum16(y, C.l);
        if (C.live && C.l < tail) o[(size_t)(chunks * CH + C.l) * o_step] = v;
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

// ---------------------------------------------------------------------------------------------------------------------
// A run of tokens, sixteen at a time, for heads of 32 to 64 channels.
//
// Inside a chunk let P_t be the product of the decays of its tokens up to t (per key channel) and S0 the state before it.  With
//   u~_t = u_t P_(t-1),  r~_t = r_t P_t,   z_t = u_t^T S_(t-1) (what the rule takes away),
// the recurrence written out is
//   z_t = u~_t S0 + sum over s < t of [ (u~_t . k_s / P_s) v_s - (u~_t . a_s / P_s) z_s ],          a_s = (a u)_s
//   o_t = r~_t S0 + sum over s <= t of [ (r~_t . k_s / P_s) v_s - (r~_t . a_s / P_s) z_s ],
//   S   = P S0 + sum over s of (P / P_s) (k_s v_s - a_s z_s)                                         P: the whole chunk's decay.
// The first line is a unit lower triangular system: solved once per chunk for the columns of u~ and for those of the v term, it is
//   z = TU S0 + Y,   o = RU S0 + Q,   S = P S0 + K~^T v - A~^T z,
// and everything but S0 is known beforehand: delta_chunk_kernel forms it for all chunks side by side, and what is left of the chain
// is two dependent products of 16 x 16 x 64 per sixteen tokens (delta_scan_kernel) in place of sixteen reductions.
//
// 1 / P_s stays below e^(16 decay_rate): the path is for decay rates up to one (9e6 at most; 1.6e4 at e^-0.5).
//
// Where keys resemble each other, a token takes away most of what the one before it put in: K~^T v and A~^T z, sums over sixteen tokens, are much
// larger than their difference, and Y comes out of such differences too.  In 32 bits that was 1.3 to 4 times the error of the rule token by
// token, which rounds after every difference.  So a chunk is formed in 64 bits (each operand rounded once, when it is stored), and the scan takes the
// two products into S on the 64-bit matrix instruction and keeps S itself in 64 bits over the run; z and o, sums of like size, stay on
// the 32-bit one.  Products that 32 bits cannot hold then do no harm to the tokens before them either.  Error against 64 bits, outputs and state,
// chunks / token by token (4 heads of 64, 304 tokens, decay rate e^-0.5; the inputs' rounding is in both): independent keys 2.05e-7 / 2.37e-7 and
// 2.57e-7 / 2.89e-7, cosine 0.9 2.81e-7 / 3.21e-7 and 4.53e-7 / 4.82e-7, 0.999 and removal near one 4.94e-7 / 6.07e-7 and 3.08e-7 / 3.47e-7.
//
// Times (16 heads of 64, 512 tokens): delta_chunk_kernel 18.6 us (17.6 in 32 bits), two workgroups per CU, each a serial chain of its own (memory,
// sums over 64 channels, the triangular solution); delta_scan_kernel 25 (18.6), 0.78 us per chunk: two products of four dependent matrix
// instructions, 64 cycles each in the second, and one exchange through LDS.  Token by token they were 12 and 67.
//
// A token that is not finite must not reach the tokens before it, which a product with a zero would do.  In k, a or w: the chunk is formed
// without the tokens from it on; their outputs and the state behind the chunk are NaN.  In a channel of v: the channel is formed without it, and from that
// token on its z and its outputs are NaN, which makes its column of the state NaN and no other.  (An r that is not finite stays in its
// own token's row.)
// ---------------------------------------------------------------------------------------------------------------------
// LDS rows of 66 and 18 doubles: sixteen rows read 16 bytes each over all banks.
constexpr int CDP = CD + 2, CP = CHUNK + 2, CV = CD + 4;
// A chunk in the workspace, [head][chunk][CHUNK_FLOATS]: TU, RU, -A~, K~, v, Y of 16 x 64 floats each, in the order in which the scan's waves take
// them (a wave's load is one stretch of 1 KB; row by row they were 4 to 16 pieces, and the scan waited for its cache), then P [64].
//   token order (-A~, K~, v, Y): [channel / 16][token / 4][channel % 16][token % 4]
//   key order   (TU, RU):        [channel / 16][channel % 4][token][channel / 4 % 4];  P: [channel / 16][channel % 4][channel / 4 % 4]
// (Register e of lane 16 g + m is row 4 g + e of a 32-bit product's result and row 4 e + g of a 64-bit one's: z is 32-bit, S 64-bit.)
enum { C_TU, C_RU, C_NA, C_K, C_V, C_Y, C_P };
constexpr int C_ARRAY = CHUNK * CD;

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ f64x4 mfma64(double a, double b, f64x4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ t12_f32x4 mfma32(float a, float b, t12_f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// four neighbouring doubles of LDS
__device__ __forceinline__ f64x4 four_doubles(const double* x)
{
    const f64x2 lo = *(const f64x2*)x, hi = *(const f64x2*)(x + 2);
    return f64x4{lo[0], lo[1], hi[0], hi[1]};
}

// Workgroup = one chunk of one head.  Wave w has the channels 16 w .. 16 w + 15, lane group g of it the tokens 4 g .. 4 g + 3: where the
// matrix product with W2 leaves them.
__global__ __launch_bounds__(256) void delta_chunk_kernel(const DeltaParams p)
{
    __shared__ __align__(16) double token[4][CHUNK * CDP], pair[4][CHUNK * CP];
    __shared__ float vs[CHUNK * CV], norm[4][CHUNK];
    __shared__ int bad, bad_v[CD];
    double *const us = token[0], *const as = token[1], *const ks = token[2], *const rs = token[3];
    float* const th = (float*)token;                       // tanh(w1) [16][rank rounded up to 64, + 4], before the tokens' vectors
    static_assert(CHUNK * (CHUNK_MAX_RANK + 4) * sizeof(float) <= sizeof(token) && CHUNK_MAX_RANK % 64 == 0, "tanh(w1) in the place of the vectors");
    const T12DeltaRule& d = p.d;
    const int head = blockIdx.y, t0 = blockIdx.x * CHUNK, nt = min(CHUNK, p.n - t0);
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, m = lane & 15, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int D = d.dim, rank = d.rank, HD = d.heads * D, rank_p = (rank + 63) & ~63, th_row = rank_p + 4;
    const int ch = wave * 16 + m, hc = head * D + min(ch, D - 1);
    float k[4], a[4], r[4], v[4], w[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float* y = p.in + (size_t)(t0 + min(g * 4 + j, nt - 1)) * p.ld + hc;
        k[j] = y[d.k_off];
        a[j] = y[d.a_off];
        r[j] = y[d.r_off];
        v[j] = y[d.v_off];
    }
    const float bk = p.bias[d.k_off + hc], ba = p.bias[d.a_off + hc], br = p.bias[d.r_off + hc], bv = p.bias[d.v_off + hc], w0 = d.w0[hc];
    // W2, sixty-four rows at a time (the first of them ahead of all that waits): step e of sixteen rows contracts its rows 4 g + e
    auto w2_at = [&](int q0, int e) __attribute__((always_inline)) { return d.w2t[(size_t)(uint32_t)(min(q0 + (e & 12) * 4 + g * 4 + (e & 3), rank - 1) * HD) + hc]; };
    float w2[16];
#pragma unroll
    for (int e = 0; e < 16; e++) w2[e] = w2_at(0, e);
    if (tid == 0) bad = CHUNK;
    if (tid < CD) bad_v[tid] = CHUNK;
    for (int q = tid; q < CHUNK * rank_p; q += 256) {      // (past the rank: zeros)
        const int t = q / rank_p, c = q % rank_p, from = d.w1_off + min(c, rank - 1);
        const float x = tanhf(p.in[(size_t)(t0 + min(t, nt - 1)) * p.ld + from] + p.bias[from]);
        th[t * th_row + c] = c < rank ? x : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        k[j] = ch < D ? k[j] + bk : 0.0f;
        const float ss = row_sum16(k[j] * k[j]);
        if (m == 0) norm[wave][g * 4 + j] = ss;
    }
    __syncthreads();
    t12_f32x4 z = (t12_f32x4)(0.0f);
    {
        const float* x = th + m * th_row + g * 4;
        for (int q0 = 0; q0 < rank_p; q0 += 64) {
            if (q0)
#pragma unroll
                for (int e = 0; e < 16; e++) w2[e] = w2_at(q0, e);
#pragma unroll
            for (int e = 0; e < 16; e++) z = mfma32(x[q0 + (e & 12) * 4 + (e & 3)], w2[e], z);
        }
    }
    double own = 1.0;                                      // decay of the thread's four tokens
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int t = g * 4 + j;
        const bool in = t < nt && ch < D;
        const float u = k[j] * (1.0f / sqrtf((norm[0][t] + norm[1][t]) + (norm[2][t] + norm[3][t]) + d.unit_eps));
        a[j] = t12_sigmoid(a[j] + ba) * u;
        w[j] = expf(-d.decay_rate * t12_sigmoid(z[j] + w0));
        v[j] += bv;
        if (in && !(__builtin_isfinite(k[j]) && __builtin_isfinite(a[j]) && __builtin_isfinite(w[j]))) atomicMin(&bad, t);
        if (in && !__builtin_isfinite(v[j])) atomicMin(&bad_v[ch], t);
        if (!in || !__builtin_isfinite(w[j])) w[j] = 1.0f; // (tokens and channels that are not there leave the state alone)
        if (!in || !__builtin_isfinite(v[j])) v[j] = 0.0f;
        r[j] = in ? r[j] + br : 0.0f;
        z[j] = in ? u : 0.0f;                              // from here on: u
        if (!in) k[j] = a[j] = 0.0f;
        own *= w[j];
    }
    double before = 1.0, after = 1.0, all = 1.0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const double x = __shfl(own, q * 16 + m);
        if (q < g) before *= x;
        if (q > g) after *= x;
        all *= x;
    }
    __syncthreads();
    const int first_bad = bad;
    float* chunk = p.rec + ((size_t)head * gridDim.x + blockIdx.x) * CHUNK_FLOATS;
    float* out = chunk + tid * 4;
    {
        t12_f32x4 na, kt, vt;
#pragma unroll
        for (int j = 3; j >= 0; j--) {
            if (g * 4 + j >= first_bad) k[j] = a[j] = v[j] = z[j] = 0.0f;
            na[j] = (float)(-after * (double)a[j]);        // (after: decay of the tokens behind this one)
            kt[j] = (float)(after * (double)k[j]);
            vt[j] = v[j];
            after *= w[j];
        }
        *(t12_f32x4*)(out + C_NA * C_ARRAY) = na;
        *(t12_f32x4*)(out + C_K * C_ARRAY) = kt;
        *(t12_f32x4*)(out + C_V * C_ARRAY) = vt;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int at = (g * 4 + j) * CDP + ch;
        us[at] = before * (double)z[j];
        before *= w[j];
        const double guess = (double)(1.0f / (float)before);   // 1 / before to 24 bits, and to 48 with what is left of one step from there
        const double back = fma(guess, fma(-before, guess, 1.0), guess);
        as[at] = back * (double)a[j];
        ks[at] = back * (double)k[j];
        rs[at] = before * (double)r[j];
        vs[(g * 4 + j) * CV + ch] = v[j];
    }
    if (g == 0) chunk[C_P * C_ARRAY + wave * 16 + (m & 3) * 4 + (m >> 2)] = first_bad < CHUNK ? __builtin_nanf("") : (float)all;
    __syncthreads();
    {
        // wave 0: u~ . a / P (token, earlier token; the other way round in LDS), 1: u~ . k / P, 2: - r~ . a / P, 3: r~ . k / P
        const double *x = (wave < 2 ? us : rs) + m * CDP + g * 4, *y = (wave & 1 ? ks : as) + m * CDP + g * 4;
        f64x4 c[2] = {(f64x4)(0.0), (f64x4)(0.0)};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const f64x4 xa = four_doubles(x + q * 16), yb = four_doubles(y + q * 16);
#pragma unroll
            for (int e = 0; e < 4; e++) c[e & 1] = mfma64(xa[e], yb[e], c[e & 1]);
        }
        c[0] += c[1];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int t = e * 4 + g;
            const double x_ = m < t + (wave >> 1) ? c[0][e] : 0.0;
            pair[wave][wave ? t * CP + m : m * CP + t] = wave == 2 ? -x_ : x_;
        }
    }
    __syncthreads();
    // the v terms, sixteen value channels per wave; that of z goes where k was
    f64x4 bv4 = (f64x4)(0.0), lv = (f64x4)(0.0);
    {
        const f64x4 cb = four_doubles(pair[1] + m * CP + g * 4), cl = four_doubles(pair[3] + m * CP + g * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const double x = (double)vs[(g * 4 + e) * CV + ch];
            bv4 = mfma64(cb[e], x, bv4);
            lv = mfma64(cl[e], x, lv);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) ks[(e * 4 + g) * CDP + ch] = bv4[e];
    }
    __syncthreads();
    if (wave < 2) {                                        // wave 0: the columns of u~, wave 1: those of the v term; solved in place
        double* col = (wave ? ks : us) + lane;
        double x[CHUNK];
#pragma unroll
        for (int t = 0; t < CHUNK; t++) x[t] = col[t * CDP];
#pragma unroll
        for (int t = 0; t < CHUNK; t++) {
#pragma unroll
            for (int q = 0; q < CHUNK / 2; q++)
                if (q * 2 + 1 > t) {
                    const f64x2 c = *(const f64x2*)(pair[0] + t * CP + q * 2);
#pragma unroll
                    for (int e = 0; e < 2; e++)
                        if (q * 2 + e > t) x[q * 2 + e] = fma(-c[e], x[t], x[q * 2 + e]);
                }
            col[t * CDP] = x[t];
        }
    }
    __syncthreads();
    // what a token takes off its own output and off that of those behind it: sixteen columns each of RU and of Q per wave
    f64x4 ru = (f64x4)(0.0);
    t12_f32x4 y, tu;
    const int first_bad_v = bad_v[ch];
    {
        const f64x4 cm = four_doubles(pair[2] + m * CP + g * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int t = g * 4 + e;
            const double x = ks[t * CDP + ch];
            ru = mfma64(cm[e], us[t * CDP + ch], ru);
            lv = mfma64(cm[e], x, lv);
            y[e] = t < first_bad_v ? (float)x : __builtin_nanf("");
        }
    }
    *(t12_f32x4*)(out + C_Y * C_ARRAY) = y;
#pragma unroll
    for (int e = 0; e < 4; e++) tu[e] = (float)us[m * CDP + wave * 16 + e * 4 + g];
    *(t12_f32x4*)(out + C_TU * C_ARRAY) = tu;
#pragma unroll
    for (int e = 0; e < 4; e++) rs[(e * 4 + g) * CDP + ch] += ru[e];     // (turned round inside the wave's own sixteen columns)
    float* o = p.o + ((size_t)t0 * d.heads + head) * D + ch;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int t = e * 4 + g;
        if (t < nt && ch < D) o[(size_t)t * HD] = t < first_bad && t < first_bad_v ? (float)lv[e] : __builtin_nanf("");
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int e = 0; e < 4; e++) tu[e] = (float)rs[m * CDP + wave * 16 + e * 4 + g];
    *(t12_f32x4*)(out + C_RU * C_ARRAY) = tu;
}

// What a wave takes of one chunk: operands of its sixteen key channels and sixteen value channels.  The four registers of an operand are
// the four steps of a product: step e contracts what register e of a result holds, the tokens 4 g + e of z and the keys 4 e + g of S.
struct ChunkOperands {
    t12_f32x4 tu, ru, na, k, v, y, decay;
    float q;
};
// Buffer loads: their 32-bit offsets (bytes from the head's first chunk) are all the address arithmetic, which as 64-bit pointers takes longer
// than a chunk's products, and what is requested past the last chunk or token is past the buffer's end and reads as zero.
typedef __amdgpu_buffer_rsrc_t Buffer;
__device__ __forceinline__ Buffer buffer_of(const float* x, size_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, (int)bytes, 0x00027000);     // raw, 32-bit elements
}
__device__ __forceinline__ float load1(Buffer b, uint32_t at)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, at, 0, 0));
}
__device__ __forceinline__ t12_f32x4 load4(Buffer b, uint32_t at)
{
    return __builtin_bit_cast(t12_f32x4, __builtin_amdgcn_raw_buffer_load_b128(b, at, 0, 0));
}
__device__ __forceinline__ void store1(float x, Buffer b, uint32_t at)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, x), b, at, 0, 0);
}
// a quarter of a chunk's requests; keys, values: where in the chunk the wave's key channels and its value channels start for this lane
__device__ __forceinline__ void request_step(ChunkOperands& x, int e, Buffer b, uint32_t keys, uint32_t values, uint32_t decay)
{
    if (e == 0) x.tu = load4(b, keys + C_TU * C_ARRAY * 4);
    if (e == 0) x.k = load4(b, keys + C_K * C_ARRAY * 4);
    if (e == 1) x.v = load4(b, values + C_V * C_ARRAY * 4);
    if (e == 1) x.ru = load4(b, keys + C_RU * C_ARRAY * 4);
    if (e == 2) x.y = load4(b, values + C_Y * C_ARRAY * 4);
    if (e == 2) x.na = load4(b, keys + C_NA * C_ARRAY * 4);
    if (e == 3) x.decay = load4(b, decay + C_P * C_ARRAY * 4);
}

// Workgroup = sixteen value channels of one head; wave w holds S of the key channels 16 w .. 16 w + 15.  z and o are sums over the key
// channels, so over the waves: they cross through LDS, one barrier per chunk (two buffers).  Operands are requested three chunks ahead.
__global__ __launch_bounds__(256) void delta_scan_kernel(const DeltaParams p)
{
    __shared__ t12_f32x4 zs[2][4][64], os[2][4][64];
    const T12DeltaRule& d = p.d;
    const int head = blockIdx.x, j0 = blockIdx.y * 16, lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const T12Row first = p.rows[0];
    const size_t region = (size_t)(first.slot >> 1) * 2 * d.state_elems;
    const size_t cell = ((size_t)head * d.dim + min(j0 + m, d.dim - 1)) * CD + wave * 16 + g;
    t12_f32x4 Sf = (t12_f32x4)(0.0f);
    if (first.position != 0)
#pragma unroll
        for (int e = 0; e < 4; e++) Sf[e] = d.state[region + (size_t)(first.slot & 1) * d.state_elems + cell + e * 4];
    const int chunks = (p.n + CHUNK - 1) / CHUNK, o_step = d.heads * d.dim;
    float* o_head = p.o + (size_t)head * d.dim + j0;
    constexpr uint32_t STEP = CHUNK_FLOATS * 4;            // bytes from chunk to chunk
    const Buffer operands = buffer_of(p.rec + (size_t)head * chunks * CHUNK_FLOATS, (size_t)chunks * STEP);
    const Buffer outs = buffer_of(o_head, ((size_t)(p.n - 1) * o_step + d.dim - j0) * 4);
    const uint32_t keys = (uint32_t)(wave * 64 + lane) * 16, values = (uint32_t)(blockIdx.y * 64 + lane) * 16, decay = (uint32_t)(wave * 4 + g) * 16;
    const uint32_t o_at = (uint32_t)((g * 4 + wave) * o_step + m) * 4;
    ChunkOperands op[4];
#pragma unroll
    for (int f = 0; f < 3; f++) {
#pragma unroll
        for (int e = 0; e < 4; e++) request_step(op[f], e, operands, f * STEP + keys, f * STEP + values, f * STEP + decay);
        op[f].q = load1(outs, (uint32_t)(f * CHUNK * o_step) * 4 + o_at);
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("" : "+v"(Sf));                           // (waited for here, not by a wait at the loop's head that would hold for the others too)
    f64x4 S = {Sf[0], Sf[1], Sf[2], Sf[3]};
    const float* ow = (const float*)&os[0][0][lane] + wave;
    // Each wave finishes the outputs of the tokens 4 g + wave of a chunk, one chunk later (and in the end).
    uint32_t store_at = 0xFFFFFFFFu;                       // (outside the buffer: not stored)
    float q = 0.0f;
    int c = 0;
    // chunk c + F of the run, F = (c + F) % 4: the registers its operands are in
    auto step = [&](auto F) __attribute__((always_inline)) {
        constexpr int f = decltype(F)::value;
        ChunkOperands &x = op[f], &y = op[(f + 3) & 3];
        const int buf = f & 1;
        const uint32_t ahead = (uint32_t)(c + f + 3) * STEP;
        t12_f32x4 z = (t12_f32x4)(0.0f), o = (t12_f32x4)(0.0f);
        f64x4 to_s = (f64x4)(0.0);
#pragma unroll
        for (int e = 0; e < 4; e++) z = mfma32(x.tu[e], Sf[e], z);
        __builtin_amdgcn_sched_barrier(0);                 // (the matrix cores have work while z crosses)
        to_s = mfma64((double)x.k[0], (double)x.v[0], to_s);
        __builtin_amdgcn_sched_barrier(0);
        zs[buf][wave][lane] = z;
        __builtin_amdgcn_sched_barrier(0);
        to_s = mfma64((double)x.k[1], (double)x.v[1], to_s);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();                                   // (a buffer is written again two chunks on, behind the next barrier)
        t12_f32x4 part[4];
        float done[4];
#pragma unroll
        for (int w = 0; w < 4; w++) part[w] = zs[buf][w][lane];
#pragma unroll
        for (int w = 0; w < 4; w++) done[w] = ow[(buf ^ 1) * 1024 + w * 256];
        // what the chain does not need runs while these are on their way
#pragma unroll
        for (int e = 0; e < 4; e++) {
            __builtin_amdgcn_sched_barrier(0);
            if (e < 2) to_s = mfma64((double)x.k[e + 2], (double)x.v[e + 2], to_s);
            request_step(y, e, operands, ahead + keys, ahead + values, ahead + decay);
            o = mfma32(x.ru[e], Sf[e], o);
        }
        double na[4], own_y[4], all[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            na[e] = (double)x.na[e];
            own_y[e] = (double)x.y[e];
            all[e] = (double)x.decay[e];
        }
        __builtin_amdgcn_sched_barrier(0);
        z = (part[0] + part[1]) + (part[2] + part[3]);
#pragma unroll
        for (int e = 0; e < 4; e++) to_s = mfma64(na[e], (double)z[e] + own_y[e], to_s);
        os[buf][wave][lane] = o;
        store1((done[0] + done[1]) + (done[2] + done[3]) + q, outs, store_at);
        q = x.q;
        y.q = load1(outs, (uint32_t)((c + f + 3) * CHUNK * o_step) * 4 + o_at);
        store_at = j0 + m < d.dim ? (uint32_t)((c + f) * CHUNK * o_step) * 4 + o_at : 0xFFFFFFFFu;
#pragma unroll
        for (int e = 0; e < 4; e++) {                      // (in 64 bits over the whole run)
            S[e] = fma(all[e], S[e], to_s[e]);
            Sf[e] = (float)S[e];
        }
    };
    // (the last one to three behind the loop: with ways out inside it the compiler moves the operands' registers about and waits for all of them)
    for (; c + 4 <= chunks; c += 4) {
        step(std::integral_constant<int, 0>());
        step(std::integral_constant<int, 1>());
        step(std::integral_constant<int, 2>());
        step(std::integral_constant<int, 3>());
    }
    if (c < chunks) step(std::integral_constant<int, 0>());
    if (c + 1 < chunks) step(std::integral_constant<int, 1>());
    if (c + 2 < chunks) step(std::integral_constant<int, 2>());
    ow += ((chunks - 1) & 1) * 1024;
    __syncthreads();
    store1((ow[0] + ow[256]) + (ow[512] + ow[768]) + q, outs, store_at);
    if (j0 + m < d.dim)
#pragma unroll
        for (int e = 0; e < 4; e++) d.state[region + (size_t)((first.slot & 1) ^ 1) * d.state_elems + cell + e * 4] = Sf[e];
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

// STAGED: records through LDS, which has room for those of heads of up to 128 channels.
template <int RL, bool STAGED>
int launch_rule(const DeltaParams& p, hipStream_t st)
{
    hipLaunchKernelGGL((delta_prep_kernel<RL * 16>), dim3((p.n + PREP_TOK - 1) / PREP_TOK, p.d.heads), dim3(256),
                       (size_t)PREP_TOK * p.d.rank * sizeof(float), st, p);
    if (!p.run) {
        hipLaunchKernelGGL(delta_token_kernel<RL>, dim3(p.n, p.d.heads, (p.d.dim + 15) / 16), dim3(256), 0, st, p);
    } else if constexpr (STAGED) {
        constexpr size_t lds = run_lds_bytes<RL>();
        if (lds > 64 * 1024) {
            static std::once_flag once[16];                // the attribute is per device
            int dev = 0;
            if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) dev = 0;
            hipError_t e = hipSuccess;
            std::call_once(once[dev], [&] { e = hipFuncSetAttribute((const void*)delta_run_kernel<RL>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); });
            if (e != hipSuccess) {
                t12_set_error("t12_delta_rule: cannot reserve %zu bytes of LDS", lds);
                return T12_ELAUNCH;
            }
        }
        hipLaunchKernelGGL(delta_run_kernel<RL>, dim3(p.d.heads, (p.d.dim + 7) / 8), dim3(128), lds, st, p);
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
    d->work_elems = (size_t)d->heads * ((d->dim_p == 64 ? std::max(CHUNK_ROW, rec_floats(64)) : rec_floats(d->dim_p)) + d->dim);
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
    const bool chunked = run && d->dim_p == CD && takes_chunks(d->heads, d->dim, d->rank, n, d->decay_rate);
    p.o = work + (size_t)n * d->heads * (chunked ? CHUNK_ROW : rec_floats(d->dim_p));
    p.out = out;
    p.out_ld = out_ld;
    int rc;
    if (chunked) {
        hipLaunchKernelGGL(delta_chunk_kernel, dim3((n + CHUNK - 1) / CHUNK, d->heads), dim3(256), 0, st, p);
        hipLaunchKernelGGL(delta_scan_kernel, dim3(d->heads, (d->dim + 15) / 16), dim3(256), 0, st, p);
        T12_CHECK_LAUNCH("t12_delta_rule(chunks)");
        rc = T12_OK;
    } else
    switch (d->dim_p) {
        case 64: rc = launch_rule<4, true>(p, st); break;  // (short runs, and decay rates the chunks are not for)
        case 128: rc = launch_rule<8, true>(p, st); break;
        case 256: rc = launch_rule<16, false>(p, st); break;
        default: rc = launch_rule<32, false>(p, st); break;
    }
    if (rc) return rc;
    const int items = n * d->heads;
    if (out_f32) hipLaunchKernelGGL(delta_out_kernel<true>, dim3((items + 3) / 4), dim3(256), 0, st, p);
    else hipLaunchKernelGGL(delta_out_kernel<false>, dim3((items + 3) / 4), dim3(256), 0, st, p);
    T12_CHECK_LAUNCH("t12_delta_rule(out)");
    return T12_OK;
}

}  // extern "C"
