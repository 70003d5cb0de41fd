// Standalone split-12 decompress: planes -> bf16 matrix, bit-exact (gfx950).
//
// out[i] = sign<<15 | (base_exp + group)<<7 | mantissa  for every flat element i,
// the function of the reference's nv_decode_split12_to_bf16
// (nvidia_kernels.cu:533-548); in patched mode the escapes (group 0) are then
// overwritten with their exact bf16 from the CSR list, which makes the result
// equal to the tensor that was packed (inverse of pack_split12,
// split12_pack.c:47-128).
// The decode is elementwise on the flat index, so the kernel ignores the row
// structure: a lane turns 16 B of sm + 8 B of gr into 32 B of bf16.
// HBM bound: 1.5 B read + 2 B written per weight.

#include "t12_device.h"
#include "t12_host.h"

namespace {

// Eight elements per lane and step (whole lines of loads and stores per wave), two steps in flight; n16 = number of whole 16-element pieces.
__global__ __launch_bounds__(256) void decompress_vec_kernel(const uint8_t* __restrict__ sm,
                                                             const uint8_t* __restrict__ gr,
                                                             uint32_t be2, uint16_t* __restrict__ out,
                                                             size_t n16)
{
    const size_t n8 = n16 * 2, stride = (size_t)gridDim.x * 512;
    be2 = t12_opaque(be2);
    for (size_t q0 = (size_t)blockIdx.x * 512 + threadIdx.x; q0 < n8; q0 += stride) {
        const size_t q1 = q0 + 256;
        const bool two = q1 < n8;
        uint2 S[2] = {t12_ldg_stream8(sm + q0 * 8), make_uint2(0, 0)};
        uint32_t G[2] = {__builtin_nontemporal_load((const uint32_t*)(gr + q0 * 4)), 0};
        if (two) {
            S[1] = t12_ldg_stream8(sm + q1 * 8);
            G[1] = __builtin_nontemporal_load((const uint32_t*)(gr + q1 * 4));
        }
        uint32_t a[4];
        t12_decode8_seq(S[0].x, S[0].y, G[0], be2, a);
        t12_stg_stream16(out + q0 * 8, make_uint4(a[0], a[1], a[2], a[3]));
        if (two) {
            t12_decode8_seq(S[1].x, S[1].y, G[1], be2, a);
            t12_stg_stream16(out + q1 * 8, make_uint4(a[0], a[1], a[2], a[3]));
        }
    }
}

// The same with the escapes written in the same launch (patched mode, n % 16 == 0): a workgroup owns PIECES x 4096
// consecutive elements; the rows it touches are consecutive, so their CSR entries are one slice [e0, e1) of the list, and the
// workgroup overwrites those of them that fall into its own elements once its decoded values are stored (a barrier and
// a workgroup-scope fence in between; no other workgroup writes these addresses).
template <int PIECES>
__global__ __launch_bounds__(256) void decompress_patched_kernel(const uint8_t* __restrict__ sm,
                                                                 const uint8_t* __restrict__ gr, uint32_t be2,
                                                                 const int32_t* __restrict__ row_off,
                                                                 const int32_t* __restrict__ cols,
                                                                 const int16_t* __restrict__ correct,
                                                                 uint16_t* __restrict__ out, size_t n16, int M, int K)
{
    constexpr size_t CHUNK = (size_t)PIECES * 4096;
    const size_t c0 = (size_t)blockIdx.x * CHUNK;
    const size_t c1 = min(c0 + CHUNK, n16 * 16);
    const int r_lo = (int)(c0 / (size_t)K), r_hi = (int)((c1 - 1) / (size_t)K);
    // the slice of the list is requested before the planes: it is used last
    const int e0 = row_off[r_lo], e1 = row_off[r_hi + 1];
    be2 = t12_opaque(be2);
    // Units of eight elements, unit u * 256 + thread: both loads and the 16-byte store of a unit are whole lines of a wave.  (Pieces of 16
    // per lane store 16 bytes in every 32: 14336 x 4096, buffers changing, 40.1 us, this 36.4; into one that the cache holds 41.1, 31.1.)
    constexpr int UNITS = PIECES * 2;
    const size_t n8 = n16 * 2, first = (size_t)blockIdx.x * (256 * UNITS) + threadIdx.x;
    uint2 S[UNITS];
    uint32_t G[UNITS];
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        const size_t q = first + u * 256;
        if (q < n8) {
            S[u] = t12_ldg_stream8(sm + q * 8);
            G[u] = __builtin_nontemporal_load((const uint32_t*)(gr + q * 4));
        }
    }
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        const size_t q = first + u * 256;
        if (q < n8) {
            uint32_t a[4];
            t12_decode8_seq(S[u].x, S[u].y, G[u], be2, a);
            t12_stg_stream16(out + q * 8, make_uint4(a[0], a[1], a[2], a[3]));
        }
    }
    if (e0 == e1) return;                                // (workgroup-uniform)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    int r = r_lo;
    for (int p = e0 + (int)threadIdx.x; p < e1; p += 256) {
        while (r < r_hi && row_off[r + 1] <= p) r++;     // entries ascend with the rows: the cursor only moves forward
        const size_t flat = (size_t)r * K + cols[p];
        if (flat >= c0 && flat < c1) out[flat] = (uint16_t)correct[p];
    }
}

// Scalar rule for what the vector kernel cannot take: the tail (n % 16), a
// base_exp outside 0..240, unaligned outputs.  Elements [first, n).
__global__ __launch_bounds__(256) void decompress_scalar_kernel(const uint8_t* __restrict__ sm,
                                                                const uint8_t* __restrict__ gr,
                                                                int base_exp, uint16_t* __restrict__ out,
                                                                size_t first, size_t n)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = first + (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint32_t g = (gr[i >> 1] >> (4 * (i & 1))) & 0xFu;
        out[i] = t12_decode_scalar(sm[i], g, base_exp);
    }
}

// One wave per row writes that row's exact values.
__global__ __launch_bounds__(256) void scatter_escapes_kernel(const int32_t* __restrict__ row_off,
                                                              const int32_t* __restrict__ cols,
                                                              const int16_t* __restrict__ correct,
                                                              uint16_t* __restrict__ out, int M, int K)
{
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= M) return;
    const int beg = row_off[row], end = row_off[row + 1];
    for (int p = beg + (threadIdx.x & 63); p < end; p += T12_WAVE)
        out[(size_t)row * K + cols[p]] = (uint16_t)correct[p];
}

}  // namespace

extern "C" int t12_decompress(const void* sm, const void* gr, int base_exp, const void* row_off,
                              const void* cols, const void* correct, void* out_bf16,
                              int M, int K, int patched, void* stream)
{
    T12_REQUIRE(M >= 0 && K >= 0, "t12_decompress: negative shape %d x %d", M, K);
    if (M == 0 || K == 0) return T12_OK;
    T12_REQUIRE(sm && gr && out_bf16, "t12_decompress: null plane or output");
    T12_REQUIRE(base_exp >= -1 && base_exp <= 254, "t12_decompress: base_exp %d out of range", base_exp);
    T12_REQUIRE(!patched || !row_off || (cols && correct), "t12_decompress: row_off given without cols/correct");
    hipStream_t st = (hipStream_t)stream;
    const size_t n = (size_t)M * K;
    const bool vec_ok = base_exp >= 0 && base_exp <= 240 && ((uintptr_t)sm % 16 == 0) &&
                        ((uintptr_t)gr % 8 == 0) && ((uintptr_t)out_bf16 % 16 == 0);
    const size_t n16 = vec_ok ? n / 16 : 0;
    if (n16 && n16 * 16 == n && patched && row_off && (n + 4095) / 4096 <= 0x7FFFFFFFull) {
        const uint32_t be2 = ((uint32_t)base_exp << 7) | ((uint32_t)base_exp << 23);
        // (two units per lane and 4096 elements per workgroup; with pieces of 16, two and four times as many were 5-8 % slower)
        hipLaunchKernelGGL(decompress_patched_kernel<1>, dim3((unsigned)((n + 4095) / 4096)), dim3(256), 0, st, (const uint8_t*)sm,
                           (const uint8_t*)gr, be2, (const int32_t*)row_off, (const int32_t*)cols, (const int16_t*)correct,
                           (uint16_t*)out_bf16, n16, M, K);
        T12_CHECK_LAUNCH("t12_decompress(patched)");
        return T12_OK;
    }
    if (n16) {
        const uint32_t be2 = ((uint32_t)base_exp << 7) | ((uint32_t)base_exp << 23);
        const size_t want = (n16 + 255) / 256;
        const int blocks = (int)(want < 256 * 64 ? want : 256 * 64);
        hipLaunchKernelGGL(decompress_vec_kernel, dim3(blocks), dim3(256), 0, st, (const uint8_t*)sm,
                           (const uint8_t*)gr, be2, (uint16_t*)out_bf16, n16);
        T12_CHECK_LAUNCH("t12_decompress(vec)");
    }
    if (n16 * 16 < n) {
        const size_t rest = n - n16 * 16;
        const size_t want = (rest + 255) / 256;
        const int blocks = (int)(want < 256 * 64 ? want : 256 * 64);
        hipLaunchKernelGGL(decompress_scalar_kernel, dim3(blocks), dim3(256), 0, st, (const uint8_t*)sm,
                           (const uint8_t*)gr, base_exp, (uint16_t*)out_bf16, n16 * 16, n);
        T12_CHECK_LAUNCH("t12_decompress(scalar)");
    }
    if (patched && row_off) {
        hipLaunchKernelGGL(scatter_escapes_kernel, dim3((M + 3) / 4), dim3(256), 0, st, (const int32_t*)row_off,
                           (const int32_t*)cols, (const int16_t*)correct, (uint16_t*)out_bf16, M, K);
        T12_CHECK_LAUNCH("t12_decompress(escapes)");
    }
    return T12_OK;
}
