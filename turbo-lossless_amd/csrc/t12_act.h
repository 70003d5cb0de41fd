// Unary functions of a projection's fp32 sums, shared by the kernels that apply them (T12Act, t12_mixers.h).
#pragma once
#include <hip/hip_runtime.h>
#include "t12_mixers.h"

template <int KIND>
__device__ __forceinline__ float t12_apply_act(float z, float a, float b)
{
    if (KIND == T12_ACT_XIELU) return z > 0.0f ? a * z * z + 0.5f * z : b * (expm1f(z) - z) + 0.5f * z;
    if (KIND == T12_ACT_SOFTCAP) return a * tanhf(z / a);
    return z;
}

__device__ __forceinline__ float t12_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

// g / (1 + e^-x): the exponential as a power of two, corrected by what y = -x log2(e) lost in rounding, and a reciprocal with one Newton
// step: 16 operations where expf and a division are 45 (64 pairs per lane in the tile kernel's epilogue: 28672 x 512 at 256 rows 21.9 ->
// 20.5 us, a prompt of 2048 tokens through four layers 6.397 -> 6.367 ms).  Within 4 x 2^-23 of the exact value; zero below x = -88, where 32 bits hold next to nothing.
__device__ __forceinline__ float t12_gate(float g, float x)
{
    const float t = __builtin_amdgcn_fmed3f(-x, -104.0f, 88.0f);
    const float y = t * 0x1.715476p+0f;
    const float lost = __builtin_fmaf(t, 0x1.4ae0bep-26f, __builtin_fmaf(t, 0x1.715476p+0f, -y));
    float e = __builtin_amdgcn_exp2f(y);
    e = __builtin_fmaf(e, lost * 0x1.62e43p-1f, e);
    const float d = 1.0f + e;
    float r = __builtin_amdgcn_rcpf(d);
    r = __builtin_fmaf(r, __builtin_fmaf(-d, r, 1.0f), r);
    return g * (x < -88.0f ? 0.0f : r);
}

// Gated linear unit of a (gate, up) pair of sums.
__device__ __forceinline__ float t12_apply_glu(float g, float u, const T12Glu& p)
{
    g = fminf(g, p.limit);
    u = __builtin_amdgcn_fmed3f(u, -p.limit, p.limit);
    return t12_gate(g, p.slope * g) * (u + p.offset);
}

// What SiLU(gate) * up is in these terms.
inline T12Glu t12_silu_glu() { return {__builtin_inff(), 1.0f, 0.0f}; }
