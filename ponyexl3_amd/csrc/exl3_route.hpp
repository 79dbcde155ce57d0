// Router arithmetic of EXL3MoEBlock (ponyexl3/mlx/exl3_moe.py:817-836), one wave per token: used by the
// router's own kernel and by the expert kernel of a few slots, which finds its experts itself.
#pragma once

#include "exl3_device.hpp"

namespace exl3 {

constexpr int kRouteMaxExperts = 1024;  // 16 per lane
constexpr int kRouteMaxTopK = 64;       // one per lane

template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ void swap16_i32(int& a, int& b) {
    float x = __builtin_bit_cast(float, a), y = __builtin_bit_cast(float, b);
    swap_rows16(x, y);
    a = __builtin_bit_cast(int, x);
    b = __builtin_bit_cast(int, y);
}
__device__ __forceinline__ void swap32_i32(int& a, int& b) {
    float x = __builtin_bit_cast(float, a), y = __builtin_bit_cast(float, b);
    swap_halves32(x, y);
    a = __builtin_bit_cast(int, x);
    b = __builtin_bit_cast(int, y);
}
// op over the wave, the result in every lane: lanes 1, 2, 4, 8 apart through DPP operands
// (quad permutations, mirrors), 16 and 32 apart by swapping registers
template <typename Op>
__device__ __forceinline__ int wave_all(int v, Op op) {
    v = op(v, dpp_i32<0xB1>(v));
    v = op(v, dpp_i32<0x4E>(v));
    v = op(v, dpp_i32<0x141>(v));
    v = op(v, dpp_i32<0x140>(v));
    int a = v, b = v;
    swap16_i32(a, b);
    v = op(a, b);
    a = v, b = v;
    swap32_i32(a, b);
    return op(a, b);
}
__device__ __forceinline__ int wave_max_i32(int v) {
    return wave_all(v, [](int a, int b) { return a > b ? a : b; });
}
__device__ __forceinline__ float wave_max_f32(float v) {
    return __builtin_bit_cast(float, wave_all(__builtin_bit_cast(int, v), [](int a, int b) {
                                  return __builtin_bit_cast(int, __builtin_fmaxf(__builtin_bit_cast(float, a),
                                                                                 __builtin_bit_cast(float, b)));
                              }));
}
__device__ __forceinline__ float wave_sum_f32(float v) {
    return __builtin_bit_cast(float, wave_all(__builtin_bit_cast(int, v), [](int a, int b) {
                                  return __builtin_bit_cast(int, __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b));
                              }));
}

// Lane l holds experts l, l + 64, ..: softmax in fp32, as keys whose order is that of the
// probabilities (they are non-negative, so their bits order like they do; an absent expert is -1).
template <typename T, int EPL>
__device__ __forceinline__ void route_probabilities(const T* __restrict__ row, int n_experts, int lane, int (&key)[EPL]) {
    float v[EPL], m = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < EPL; i++) {
        v[i] = i * 64 + lane < n_experts ? (float)row[i * 64 + lane] : -__builtin_inff();
        m = __builtin_fmaxf(m, v[i]);
    }
    m = wave_max_f32(m);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < EPL; i++) {
        v[i] = expf(v[i] - m);  // 0 where there is no expert
        sum += v[i];
    }
    sum = wave_sum_f32(sum);
#pragma unroll
    for (int i = 0; i < EPL; i++)
        key[i] = i * 64 + lane < n_experts ? __builtin_bit_cast(int, v[i] / sum) & 0x7FFFFFFF : -1;
}

struct RouteChoice {
    float p;  // lane j: probability and expert of choice j
    int e;
};

// Choice j: largest probability, lowest expert among equals; returns the expert (uniform).
template <int EPL>
__device__ __forceinline__ int route_next(int (&key)[EPL], int lane, int j, RouteChoice& c) {
    int best = key[0];
#pragma unroll
    for (int i = 1; i < EPL; i++) best = key[i] > best ? key[i] : best;
    best = __builtin_amdgcn_readfirstlane(wave_max_i32(best));
    int e = 0;
#pragma unroll
    for (int i = EPL - 1; i >= 0; i--) {
        const unsigned long long hit = __ballot(key[i] == best);
        if (hit) e = i * 64 + (int)__builtin_ctzll(hit);
    }
#pragma unroll
    for (int i = 0; i < EPL; i++)
        if (e == i * 64 + lane) key[i] = -1;
    if (lane == j) {
        c.p = __builtin_bit_cast(float, best);
        c.e = e;
    }
    return e;
}

// Row t of the routing table after top_k choices, with a shared expert behind them whose gate's logit
// is given. PUBLISH: indices through the level that the XCDs share, for a workgroup of the same launch.
template <typename T, bool PUBLISH = false>
__device__ __forceinline__ void route_write(RouteChoice c, int lane, int t, int n_experts, int top_k, int norm,
                                            bool shared, T shared_logit, int* __restrict__ indices,
                                            half_t* __restrict__ scores) {
    if (norm) c.p = c.p / wave_sum_f32(c.p);
    const int slots = top_k + shared;
    auto put = [&](int j, int e) {
        int* at = indices + (size_t)t * slots + j;
        if constexpr (PUBLISH) __hip_atomic_store(at, e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *at = e;
    };
    if (lane < top_k) {
        put(lane, c.e);
        scores[(size_t)t * slots + lane] = (half_t)c.p;
    }
    if (shared && lane == 0) {
        const float s = (float)shared_logit;
        put(top_k, n_experts);
        scores[(size_t)t * slots + top_k] = (half_t)(float)(T)(1.0f / (1.0f + expf(-s)));
    }
}

}  // namespace exl3
