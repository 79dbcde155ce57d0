// Gated activations of the routed experts (ponyexl3/mlx/exl3_moe.py:62-75).
#pragma once

#include <hip/hip_runtime.h>

namespace exl3 {

// activation 0: SiLU, 1: tanh-GELU
__device__ __forceinline__ float glu_act(float g, float u, int activation) {
#pragma clang fp contract(off)
    if (activation == 1) {
        const float t = 0.797884560803f * (g + 0.044715f * g * g * g);
        return 0.5f * g * (1.0f + tanhf(t)) * u;
    }
    return (g / (1.0f + expf(-g))) * u;
}

}  // namespace exl3
