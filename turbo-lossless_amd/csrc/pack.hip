// GPU-side split-12 packer (gfx950): bf16 matrix in HBM -> planes + CSR escape
// list, byte-identical to what the reference's CPU packer emits.
//
//   t12_pack_histogram + t12_pack_base_exp   = split12_find_base_exp (split12_pack.c:18-37)
//   t12_pack_planes / _row_offsets / _escapes = pack_split12          (split12_pack.c:47-128)
//
// The reference makes two O(M*K) passes on one CPU thread; here the first pass
// is a streaming kernel (16 weights per lane, 32 B in, 24 B out), the CSR pointers
// come from a single-workgroup scan of the per-row escape counts, and the
// second pass compacts each row's escapes in ascending column order with one
// wave per row (ballot + prefix popcount), so the order inside a row is the
// reference's.

#include "t12_device.h"
#include "t12_host.h"

namespace {

__device__ __forceinline__ uint32_t group_of(uint32_t v, int base_exp)
{
    const int g = (int)((v >> 7) & 0xFFu) - base_exp;
    return (g >= 1 && g <= 15) ? (uint32_t)g : 0u;
}

// Exponent histogram.  The exponents of a weight matrix fall into a handful of bins, so 64 lanes adding into one
// 256-bin table serialise on those bins (LDS atomics to one address execute one lane at a time: measured 0.8 TB/s).
// Every lane of a wave has a copy of the table, laid out [bin][copy]: no two lanes on one counter, nor on one bank.  One workgroup per CU, of
// sixteen waves: each adds a sum per bin to the same few words of memory at the end.  14336 x 4096: 20.6 us, 25.4 with sixteen copies
// and 512 workgroups of four waves; the read alone takes 19.
constexpr int HIST_COPIES = 64;
__global__ __launch_bounds__(1024) void histogram_kernel(const uint16_t* __restrict__ w, size_t n,
                                                        unsigned long long* __restrict__ hist)
{
    __shared__ unsigned int h[256 * HIST_COPIES];
    for (int i = threadIdx.x; i < 256 * HIST_COPIES; i += 1024) h[i] = 0;
    __syncthreads();
    const int copy = threadIdx.x & (HIST_COPIES - 1);
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t n8 = n / 8;
    // four 16-byte pieces per lane in flight (the grid is small, see the launcher)
    for (size_t q0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q0 < n8; q0 += 4 * stride) {
        uint4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const size_t q = q0 + u * stride;
            v[u] = q < n8 ? *(const uint4*)(w + q * 8) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (q0 + u * stride >= n8) break;
            const uint32_t d[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                atomicAdd(&h[(((d[i] >> 7) & 0xFFu) * HIST_COPIES) | copy], 1u);
                atomicAdd(&h[(((d[i] >> 23) & 0xFFu) * HIST_COPIES) | copy], 1u);
            }
        }
    }
    if (blockIdx.x == 0)
        for (size_t i = n8 * 8 + threadIdx.x; i < n; i += blockDim.x) atomicAdd(&h[(((uint32_t)w[i] >> 7) & 0xFFu) * HIST_COPIES], 1u);
    __syncthreads();
    // four lanes per bin, sixteen copies each
    const int bin = threadIdx.x >> 2, part = threadIdx.x & 3;
    unsigned int sum = 0;
#pragma unroll
    for (int c = 0; c < HIST_COPIES / 4; c++) sum += h[bin * HIST_COPIES + 16 * part + ((c + bin) & 15)];
    sum += __shfl_xor(sum, 1, T12_WAVE);
    sum += __shfl_xor(sum, 2, T12_WAVE);
    if (part == 0 && sum) atomicAdd(&hist[bin], (unsigned long long)sum);
}

// Planes for the whole 16-element pieces of the flat array.
// (base_dev: the base exponent in device memory, in the place of base_exp)
__global__ __launch_bounds__(256) void planes_kernel(const uint16_t* __restrict__ w, size_t n16, int K,
                                                     int base_exp, const int32_t* __restrict__ base_dev, uint8_t* __restrict__ sm,
                                                     uint8_t* __restrict__ gr, int32_t* __restrict__ row_cnt)
{
    if (base_dev) base_exp = *base_dev;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n16; q += stride) {
        const uint4 lo = *(const uint4*)(w + q * 16);
        const uint4 hi = *(const uint4*)(w + q * 16 + 8);
        const uint32_t d[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        uint32_t s[4] = {0, 0, 0, 0};
        uint32_t g[2] = {0, 0};
        uint32_t esc = 0;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t v = (d[i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
            const uint32_t gi = group_of(v, base_exp);
            s[i >> 2] |= (((v >> 15) << 7) | (v & 0x7Fu)) << (8 * (i & 3));
            g[i >> 3] |= gi << (4 * (i & 7));
            esc |= (gi == 0u) << i;
        }
        *(uint4*)(sm + q * 16) = make_uint4(s[0], s[1], s[2], s[3]);
        *(uint2*)(gr + q * 8) = make_uint2(g[0], g[1]);
        while (esc) {                                   // rare: ~0.05 % of the weights
            const int i = __builtin_ctz(esc);
            esc &= esc - 1;
            atomicAdd(&row_cnt[(q * 16 + i) / (size_t)K], 1);
        }
    }
}

// The last n % 16 elements, by one lane (an odd count leaves the high nibble 0).
__global__ void planes_tail_kernel(const uint16_t* __restrict__ w, size_t first, size_t n, int K, int base_exp,
                                   const int32_t* __restrict__ base_dev, uint8_t* __restrict__ sm, uint8_t* __restrict__ gr,
                                   int32_t* __restrict__ row_cnt)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    if (base_dev) base_exp = *base_dev;
    for (size_t i = first; i < n; i++) {
        const uint32_t v = w[i];
        const uint32_t gi = group_of(v, base_exp);
        sm[i] = (uint8_t)(((v >> 15) << 7) | (v & 0x7Fu));
        if (i & 1) gr[i >> 1] = (uint8_t)(gr[i >> 1] | (gi << 4));
        else gr[i >> 1] = (uint8_t)gi;
        if (gi == 0u) atomicAdd(&row_cnt[i / (size_t)K], 1);
    }
}

// The window rule of t12_pack_base_exp on the histogram in device memory; 256 lanes.  Also clears the rows' counts, which the next
// kernel adds to.
__global__ __launch_bounds__(256) void base_exp_kernel(const unsigned long long* __restrict__ hist, int32_t* __restrict__ base,
                                                       int32_t* __restrict__ row_cnt, int M)
{
    if (blockIdx.x == 0) {
        __shared__ unsigned long long h[256], best[256];
        __shared__ int at[256];
        const int t = threadIdx.x;
        h[t] = hist[t];
        __syncthreads();
        unsigned long long run = 0;
        if (t <= 241)
            for (int j = 0; j < 15; j++) run += h[t + j];
        best[t] = run;
        at[t] = t;
        __syncthreads();
        for (int half = 128; half; half >>= 1) {              // the first of the largest windows
            if (t < half && (best[t + half] > best[t] || (best[t + half] == best[t] && at[t + half] < at[t]))) {
                best[t] = best[t + half];
                at[t] = at[t + half];
            }
            __syncthreads();
        }
        if (t == 0) *base = at[0] - 1;
    }
    for (uint32_t r = blockIdx.x * 256 + threadIdx.x; r < (uint32_t)M; r += gridDim.x * 256) row_cnt[r] = 0;
}

// row_off[0] = 0, row_off[r+1] = sum of cnt[0..r]; one workgroup of 1024 lanes, eight neighbouring counts per lane and step, the next
// step's requested ahead (14336 rows: 15.2 us with a stretch of the rows per lane, 8.7).
// (Row numbers unsigned: a step past the last of up to 2^31 - 1 rows.)
__global__ __launch_bounds__(1024) void scan_kernel(const int32_t* __restrict__ cnt, uint32_t M,
                                                    int32_t* __restrict__ row_off)
{
    __shared__ int part[2][16];
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    constexpr uint32_t OWN = 8, STEP = 1024 * OWN;
    const bool vec = (uintptr_t)cnt % 16 == 0;
    auto fetch = [&](uint32_t r0, int (&c)[OWN]) __attribute__((always_inline)) {
        const uint32_t r = r0 + OWN * t;
        if (vec && r + OWN <= M) {
#pragma unroll
            for (uint32_t i = 0; i < OWN; i += 4) {
                const int4 v = *(const int4*)(cnt + r + i);
                c[i] = v.x;
                c[i + 1] = v.y;
                c[i + 2] = v.z;
                c[i + 3] = v.w;
            }
        } else {
#pragma unroll
            for (uint32_t i = 0; i < OWN; i++) c[i] = r + i < M ? cnt[r + i] : 0;
        }
    };
    int c[OWN], next[OWN] = {}, carry = 0;
    fetch(0, c);
    if (t == 0) row_off[0] = 0;
    for (uint32_t r0 = 0, k = 0; r0 < M; r0 += STEP, k ^= 1) {
        if (r0 + STEP < M) fetch(r0 + STEP, next);
        int own = 0;
#pragma unroll
        for (uint32_t i = 0; i < OWN; i++) own += c[i];
        int sum = own;                                      // inclusive over the wave
#pragma unroll
        for (uint32_t o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(sum, o, T12_WAVE);
            if (lane >= o) sum += v;
        }
        if (lane == 63) part[k][wave] = sum;
        __syncthreads();                                    // (two tables: one barrier per step)
        int run = carry + sum - own;
#pragma unroll
        for (uint32_t w = 0; w < 16; w++) {
            const int v = part[k][w];
            run += w < wave ? v : 0;
            carry += v;
        }
#pragma unroll
        for (uint32_t i = 0; i < OWN; i++) {
            run += c[i];
            if (r0 + OWN * t + i < M) row_off[r0 + OWN * t + i + 1] = run;
            c[i] = next[i];
        }
    }
}

// The same list from the nibble plane, where a zero is an escape: a quarter of the bytes, and a weight itself is read only where there is
// one.  K % 32 == 0 and a plane that 16-byte loads may be taken from.  A lane takes 32 neighbouring columns per step, the wave 2048;
// two steps are requested together (14336 x 4096: 8.7 us, 18.2 from the weights).
__global__ __launch_bounds__(256) void escapes_plane_kernel(const uint16_t* __restrict__ w, const uint8_t* __restrict__ gr, int M, int K,
                                                            int base_exp, const int32_t* __restrict__ row_off,
                                                            int32_t* __restrict__ cols, int16_t* __restrict__ correct,
                                                            int16_t* __restrict__ wrong)
{
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= M) return;
    const int lane = threadIdx.x & 63;
    const uint16_t* wr = w + (size_t)row * K;
    const uint8_t* gp = gr + (size_t)row * K / 2;
    const unsigned long long below = (1ull << lane) - 1ull;
    int base = row_off[row];
    const int end = row_off[row + 1];
    for (int k0 = 0; k0 < K && base < end; k0 += 4096) {
        uint4 v[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int k = k0 + 2048 * u + 32 * lane;
            v[u] = k < K ? *(const uint4*)(gp + k / 2) : make_uint4(~0u, ~0u, ~0u, ~0u);
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const uint32_t x[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
            uint32_t zero[4];                                // bit 4 j: nibble j is zero
            int n = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t any = x[i] | x[i] >> 1;
                any |= any >> 2;
                zero[i] = ~any & 0x11111111u;
                n += __popc(zero[i]);
            }
            if (__ballot(n != 0) == 0ull) continue;
            int before = 0, total = 0;                       // a prefix sum of the lanes' counts (at most 32), a ballot per bit
#pragma unroll
            for (int bit = 0; bit < 6; bit++) {
                const unsigned long long m = __ballot((n >> bit) & 1);
                before += __popcll(m & below) << bit;
                total += __popcll(m) << bit;
            }
            int pos = base + before;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                while (zero[i]) {
                    const int k = k0 + 2048 * u + 32 * lane + 8 * i + (__builtin_ctz(zero[i]) >> 2);
                    zero[i] &= zero[i] - 1;
                    const uint32_t e = wr[k];
                    cols[pos] = k;
                    correct[pos] = (int16_t)e;
                    wrong[pos] = (int16_t)t12_decode_scalar(((e >> 15) << 7) | (e & 0x7Fu), 0u, base_exp);
                    pos++;
                }
            }
            base += total;
        }
    }
}

// One wave per row: ordered compaction of the row's escapes.  K % 8 == 0 (rows start 16-byte aligned): a lane takes
// eight consecutive columns per step with one 128-bit load and the wave skips a step without escapes after one
// ballot; the order of the list (ascending column) is lane-major within a step, so an entry's place is the count of
// escapes in lower lanes plus the lane's own earlier ones.  Other K: one column per lane and step.
__global__ __launch_bounds__(256) void escapes_kernel(const uint16_t* __restrict__ w, int M, int K, int base_exp,
                                                      const int32_t* __restrict__ row_off,
                                                      int32_t* __restrict__ cols, int16_t* __restrict__ correct,
                                                      int16_t* __restrict__ wrong)
{
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= M) return;
    const int lane = threadIdx.x & 63;
    int base = row_off[row];
    if (row_off[row + 1] == base) return;               // nothing to write in this row
    const uint16_t* wr = w + (size_t)row * K;
    if ((K & 7) == 0 && ((uintptr_t)w & 15) == 0) {
        const unsigned long long below = (1ull << lane) - 1ull;
        for (int k0 = 0; k0 < K; k0 += T12_WAVE * 8) {
            const int k = k0 + lane * 8;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (k < K) v = *(const uint4*)(wr + k);
            const uint32_t d[4] = {v.x, v.y, v.z, v.w};
            uint32_t mine = 0;                           // bit j: column k + j is an escape
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t e = (d[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
                if (k < K && group_of(e, base_exp) == 0u) mine |= 1u << j;
            }
            if (__ballot(mine != 0u) == 0ull) continue;
            // escapes in lower lanes: a wave prefix sum of the lanes' counts, by one ballot per bit of the count (<= 8)
            const int cnt = __popc(mine);
            int before = 0;
#pragma unroll
            for (int bit = 0; bit < 4; bit++)
                before += __popcll(__ballot((cnt >> bit) & 1) & below) << bit;
            int total = 0;
#pragma unroll
            for (int bit = 0; bit < 4; bit++) total += __popcll(__ballot((cnt >> bit) & 1)) << bit;
            int pos = base + before;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if (mine & (1u << j)) {
                    const uint32_t e = (d[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
                    cols[pos] = k + j;
                    correct[pos] = (int16_t)e;
                    wrong[pos] = (int16_t)t12_decode_scalar(((e >> 15) << 7) | (e & 0x7Fu), 0u, base_exp);
                    pos++;
                }
            }
            base += total;
        }
        return;
    }
    for (int k0 = 0; k0 < K; k0 += T12_WAVE) {
        const int k = k0 + lane;
        const uint32_t v = k < K ? wr[k] : 0u;
        const bool esc = k < K && group_of(v, base_exp) == 0u;
        const unsigned long long m = __ballot(esc);
        if (esc) {
            const int pos = base + __popcll(m & ((1ull << lane) - 1ull));
            cols[pos] = k;
            correct[pos] = (int16_t)v;
            wrong[pos] = (int16_t)t12_decode_scalar(((v >> 15) << 7) | (v & 0x7Fu), 0u, base_exp);
        }
        base += __popcll(m);
    }
}

int blocks_for(size_t items)
{
    const size_t want = (items + 255) / 256;
    return (int)(want < 1 ? 1 : (want < 256 * 32 ? want : 256 * 32));
}

int launch_planes(const void* w_bf16, int M, int K, int base_exp, const int32_t* base_dev, void* sm, void* gr, void* row_cnt, hipStream_t st)
{
    const size_t n = (size_t)M * K, n16 = n / 16;
    if (n16) {
        hipLaunchKernelGGL(planes_kernel, dim3(blocks_for(n16)), dim3(256), 0, st, (const uint16_t*)w_bf16, n16, K,
                           base_exp, base_dev, (uint8_t*)sm, (uint8_t*)gr, (int32_t*)row_cnt);
        T12_CHECK_LAUNCH("t12_pack_planes");
    }
    if (n16 * 16 < n) {
        hipLaunchKernelGGL(planes_tail_kernel, dim3(1), dim3(64), 0, st, (const uint16_t*)w_bf16, n16 * 16, n, K,
                           base_exp, base_dev, (uint8_t*)sm, (uint8_t*)gr, (int32_t*)row_cnt);
        T12_CHECK_LAUNCH("t12_pack_planes(tail)");
    }
    return T12_OK;
}

}  // namespace

extern "C" {

int t12_pack_histogram(const void* w_bf16, size_t n, void* hist_u64x256, void* stream)
{
    T12_REQUIRE(hist_u64x256 && (w_bf16 || n == 0), "t12_pack_histogram: null operand");
    T12_REQUIRE((uintptr_t)w_bf16 % 16 == 0, "t12_pack_histogram: input must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    if (hipMemsetAsync(hist_u64x256, 0, 256 * sizeof(unsigned long long), st) != hipSuccess) return T12_ELAUNCH;
    if (n == 0) return T12_OK;
    // few workgroups, long strides: every workgroup ends with one 64-bit atomic per bin it met, and those all land on
    // the same dozen addresses (8192 workgroups spent 130 us there, whatever the size of the matrix)
    const size_t want = (n / 8 + 1023) / 1024;
    const int blocks = want < 1 ? 1 : (want < 256 ? (int)want : 256);
    hipLaunchKernelGGL(histogram_kernel, dim3(blocks), dim3(1024), 0, st, (const uint16_t*)w_bf16, n,
                       (unsigned long long*)hist_u64x256);
    T12_CHECK_LAUNCH("t12_pack_histogram");
    return T12_OK;
}

// Host: the window rule of split12_find_base_exp on a 256-bin histogram.
int t12_pack_base_exp(const uint64_t* hist_host)
{
    uint64_t best = 0, run = 0;
    int best_start = 0;
    for (int j = 0; j < 15; j++) run += hist_host[j];
    for (int s = 0; s <= 241; s++) {
        if (s > 0) run += hist_host[s + 14] - hist_host[s - 1];
        if (run > best) { best = run; best_start = s; }
    }
    return best_start - 1;
}

int t12_pack_planes(const void* w_bf16, int M, int K, int base_exp, void* sm, void* gr, void* row_cnt,
                    void* stream)
{
    T12_REQUIRE(M >= 1 && K >= 1 && w_bf16 && sm && gr && row_cnt, "t12_pack_planes: bad operands");
    T12_REQUIRE(base_exp >= -1 && base_exp <= 240, "t12_pack_planes: base_exp %d out of range", base_exp);
    T12_REQUIRE((uintptr_t)w_bf16 % 16 == 0 && (uintptr_t)sm % 16 == 0 && (uintptr_t)gr % 8 == 0,
                "t12_pack_planes: buffers must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    if (hipMemsetAsync(row_cnt, 0, (size_t)M * sizeof(int32_t), st) != hipSuccess) return T12_ELAUNCH;
    return launch_planes(w_bf16, M, K, base_exp, nullptr, sm, gr, row_cnt, st);
}

// Histogram, base exponent, planes and row offsets in one go, without the host in between.
int t12_pack_begin(const void* w_bf16, int M, int K, void* hist_u64x256, void* base_exp, void* sm, void* gr, void* row_cnt, void* row_off,
                   void* stream)
{
    T12_REQUIRE(M >= 1 && K >= 1 && w_bf16 && hist_u64x256 && base_exp && sm && gr && row_cnt && row_off, "t12_pack_begin: bad operands");
    T12_REQUIRE((uintptr_t)w_bf16 % 16 == 0 && (uintptr_t)sm % 16 == 0 && (uintptr_t)gr % 8 == 0,
                "t12_pack_begin: buffers must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    int rc = t12_pack_histogram(w_bf16, (size_t)M * K, hist_u64x256, stream);
    if (rc) return rc;
    const int blocks = M < 64 * 4096 ? (M + 4095) / 4096 : 64;
    hipLaunchKernelGGL(base_exp_kernel, dim3(blocks), dim3(256), 0, st, (const unsigned long long*)hist_u64x256, (int32_t*)base_exp,
                       (int32_t*)row_cnt, M);
    T12_CHECK_LAUNCH("t12_pack_begin(base)");
    rc = launch_planes(w_bf16, M, K, 0, (const int32_t*)base_exp, sm, gr, row_cnt, st);
    return rc ? rc : t12_pack_row_offsets(row_cnt, M, row_off, stream);
}

int t12_pack_row_offsets(const void* row_cnt, int M, void* row_off, void* stream)
{
    T12_REQUIRE(M >= 1 && row_cnt && row_off, "t12_pack_row_offsets: bad operands");
    hipLaunchKernelGGL(scan_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, (const int32_t*)row_cnt, M,
                       (int32_t*)row_off);
    T12_CHECK_LAUNCH("t12_pack_row_offsets");
    return T12_OK;
}

int t12_pack_escapes(const void* w_bf16, int M, int K, int base_exp, const void* row_off, void* cols,
                     void* correct, void* wrong, void* stream)
{
    T12_REQUIRE(M >= 1 && K >= 1 && w_bf16 && row_off, "t12_pack_escapes: bad operands");
    if (!cols || !correct || !wrong) return T12_OK;     // P == 0: nothing to fill
    hipLaunchKernelGGL(escapes_kernel, dim3((M + 3) / 4), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t*)w_bf16, M, K, base_exp, (const int32_t*)row_off, (int32_t*)cols,
                       (int16_t*)correct, (int16_t*)wrong);
    T12_CHECK_LAUNCH("t12_pack_escapes");
    return T12_OK;
}

// t12_pack_escapes with the nibble plane at hand.
int t12_pack_escapes_plane(const void* w_bf16, const void* gr, int M, int K, int base_exp, const void* row_off, void* cols,
                           void* correct, void* wrong, void* stream)
{
    T12_REQUIRE(M >= 1 && K >= 1 && w_bf16 && gr && row_off, "t12_pack_escapes_plane: bad operands");
    if (!cols || !correct || !wrong) return T12_OK;     // P == 0: nothing to fill
    if (K % 32 || (uintptr_t)gr % 16) return t12_pack_escapes(w_bf16, M, K, base_exp, row_off, cols, correct, wrong, stream);
    hipLaunchKernelGGL(escapes_plane_kernel, dim3((M + 3) / 4), dim3(256), 0, (hipStream_t)stream, (const uint16_t*)w_bf16,
                       (const uint8_t*)gr, M, K, base_exp, (const int32_t*)row_off, (int32_t*)cols, (int16_t*)correct,
                       (int16_t*)wrong);
    T12_CHECK_LAUNCH("t12_pack_escapes_plane");
    return T12_OK;
}

}  // extern "C"
