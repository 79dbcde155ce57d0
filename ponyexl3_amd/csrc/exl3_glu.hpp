// Gated activations of the routed experts (ponyexl3/mlx/exl3_moe.py:62-75).
#pragma once

#include <hip/hip_runtime.h>

namespace exl3 {

// g / (1 + exp(-g)). The exponential by reduction to a power of two, the product with log2(e) in two parts as in Cody and
// Waite's: exp(-g) = 2^n 2^f with n + f = -g log2(e), n whole and f at most 1/2, where the second part of log2(e)
// keeps the bits below the first product; 2^f by v_exp_f32. The quotient by v_rcp_f32 and one Newton correction with the
// remainder; it needs no scaling, as its divisor is 1 and more. Rounded to a half the result is that of
// g / (1.0f + expf(-g)) for all 65536 halfs g, and over 2^22 normal g of deviation 4 the fp32 errors are the same (2.02 ulp at most,
// 0.472 rms). So are zeros, infinities and NaNs: -g goes in between -100, where 1 + exp(-g) is 1, and 200, where
// exp(-g) is infinite, and v_div_fixup gives what an infinite g or divisor makes of a quotient.
__device__ __forceinline__ float silu(float g) {
#pragma clang fp contract(off)
    const float t = __builtin_amdgcn_fmed3f(-g, -100.f, 200.f);
    const float h = t * 1.44269504f, n = __builtin_rintf(h);
    const float f = (h - n) + __builtin_fmaf(t, 1.92596299e-8f, __builtin_fmaf(t, 1.44269504f, -h));
    const float d = __builtin_ldexpf(__builtin_amdgcn_exp2f(f), (int)n) + 1.f;
    const float r = __builtin_amdgcn_rcpf(d);
    const float q = g * r;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, g), r, q), d, g);
}

// activation 0: SiLU, 1: tanh-GELU
__device__ __forceinline__ float glu_act(float g, float u, int activation) {
#pragma clang fp contract(off)
    if (activation == 1) {
        const float t = 0.797884560803f * (g + 0.044715f * g * g * g);
        return 0.5f * g * (1.0f + tanhf(t)) * u;
    }
    return silu(g) * u;
}

}  // namespace exl3
