// Router and weighted sum around the routed experts: what EXL3MoEBlock does between the
// router's matrix product and its output (ponyexl3/mlx/exl3_moe.py:817-839).
//
// Both are bound by latency at decode sizes: as tensor operations they were twelve launches
// of 1.5-12 us each (57 us of GPU time and 120 us of host time per decoded token), here they
// are one launch before the experts and one behind them.
#include "exl3_device.hpp"
#include "exl3_host.hpp"
#include "exl3_groups.hpp"
#include "exl3_route.hpp"

namespace exl3 {

// fp16(x . w) over a wave, fp32 sums; n % 8 == 0
__device__ __forceinline__ half_t wave_dot(const half_t* __restrict__ x, const half_t* __restrict__ w, int n, int lane) {
    float acc[8] = {};
    for (int c0 = lane * 8; c0 < n; c0 += 4 * 512) {
        uint4_t a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int c = min(c0 + i * 512, n - 8);
            a[i] = *reinterpret_cast<const uint4_t*>(x + c);
            b[i] = *reinterpret_cast<const uint4_t*>(w + c);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float u[8], v[8];
            halfs_to_floats(a[i], u);
            halfs_to_floats(b[i], v);
            if (c0 + i * 512 < n) {
#pragma unroll
                for (int k = 0; k < 8; k++) acc[k] = __builtin_fmaf(u[k], v[k], acc[k]);
            }
        }
    }
    const float s = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
    return (half_t)wave_sum_f32(s);
}

// One wave per token, see route_probabilities() and route_next(). With a shared expert its index n_experts
// and sigmoid(shared logit) follow the top_k. The logit is given, or x and the weight of its gate are: as a
// library product of its own it takes 7 us at 1537 tokens of 2048 and 5 at 100, here nothing that shows
// next to the 6 us of the ranking, and 1 MB to 6 MB more to read.
template <typename T, int EPL>
__global__ __launch_bounds__(256) void moe_route_kernel(const T* __restrict__ logits,
                                                        const T* __restrict__ shared_logits,
                                                        const half_t* __restrict__ x, const half_t* __restrict__ w_shared,
                                                        int D, int tokens, int n_experts, int top_k, int norm,
                                                        int* __restrict__ indices, half_t* __restrict__ scores) {
    const int lane = threadIdx.x & 63;
    const long long t = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= tokens) return;
    T shared{};
    if (w_shared) shared = (T)wave_dot(x + t * D, w_shared, D, lane);
    else if (shared_logits) shared = shared_logits[t];
    int key[EPL];
    route_probabilities<T, EPL>(logits + t * n_experts, n_experts, lane, key);
    RouteChoice c{0.f, 0};
    for (int j = 0; j < top_k; j++) route_next<EPL>(key, lane, j, c);
    route_write<T>(c, lane, (int)t, n_experts, top_k, norm, w_shared || shared_logits, shared, indices, scores);
}

// The same (logits given) with the list of slot groups for the expert kernels behind it, made by the
// workgroup that comes last: 24 tokens of 9 slots 5.1 -> 7.0 us, where a launch of its
// own for the list takes 2.8 to 4.7 and a gap.
template <int EPL>
__global__ __launch_bounds__(kGroupThreads) void moe_route_groups_kernel(
    const half_t* __restrict__ logits, const half_t* __restrict__ shared_logits, int tokens, int n_experts, int top_k,
    int norm, int* indices, half_t* __restrict__ scores, int num_experts, int4* groups, int* arrived) {
    __shared__ GroupScratch scratch;
    __shared__ int last_flag;
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * (kGroupThreads / kWave) + (threadIdx.x >> 6);
    if (t < tokens) {
        const half_t shared = shared_logits ? shared_logits[t] : half_t{};
        int key[EPL];
        route_probabilities<half_t, EPL>(logits + (size_t)t * n_experts, n_experts, lane, key);
        RouteChoice c{0.f, 0};
        for (int j = 0; j < top_k; j++) route_next<EPL>(key, lane, j, c);
        route_write<half_t, true>(c, lane, t, n_experts, top_k, norm, shared_logits, shared, indices, scores);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every wave's own indices have reached the shared level
    __syncthreads();
    if (threadIdx.x == 0)
        last_flag = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
    __syncthreads();
    if (!last_flag) return;
    if (threadIdx.x == 0) __hip_atomic_store(arrived, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    make_slot_groups([&](int s) { return __hip_atomic_load(indices + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); },
                     tokens * (top_k + (shared_logits != nullptr)), num_experts, groups, scratch);
}

// Router logits of a few tokens: logits[t][e] = fp16(x[t] . w[e]), the shared gate's row (if
// any) behind the experts', fp32 sums. A workgroup takes 16 experts and up to 16 tokens on
// v_mfma_f32_16x16x32_f16; its eight waves share the reduction (32-deep steps dealt round
// robin), so that 16 rows of 4 KiB are in flight at once, and meet in LDS. Bound by one
// round trip to memory: 1 MB of weights over 17 CUs. The library's product takes 6.7 us of
// GPU and 20 us of host time for 1 x 2048 x 256.
constexpr int kGateWaves = 8;

__global__ __launch_bounds__(kGateWaves * 64) void moe_gate_kernel(
    const half_t* __restrict__ x, const half_t* __restrict__ w, const half_t* __restrict__ w_shared, int tokens,
    int n_experts, int D, half_t* __restrict__ logits, half_t* __restrict__ shared_logits) {
    __shared__ float4_t red[kGateWaves][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int fr = lane & 15, q = lane >> 4;
    const int rows = n_experts + (w_shared != nullptr);
    const int e = min((int)blockIdx.x * 16 + fr, rows - 1), t = min((int)blockIdx.y * 16 + fr, tokens - 1);
    const half_t* wr = (e < n_experts ? w + (size_t)e * D : w_shared) + q * 8;
    const half_t* xr = x + (size_t)t * D + q * 8;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    const int steps = D >> 5;
    for (int s0 = wave; s0 < steps; s0 += 8 * kGateWaves) {
        half8_t a[8], b[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int s = min(s0 + i * kGateWaves, steps - 1);
            a[i] = *reinterpret_cast<const half8_t*>(wr + s * 32);
            b[i] = *reinterpret_cast<const half8_t*>(xr + s * 32);
        }
#pragma unroll
        for (int i = 0; i < 8; i++)
            if (s0 + i * kGateWaves < steps) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[i], acc, 0, 0, 0);
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave != 0) return;
    float4_t sum = red[0][lane];
#pragma unroll
    for (int i = 1; i < kGateWaves; i++) sum = sum + red[i][lane];
    // the lane holds experts 4 q .. 4 q + 3 of token fr
    const int tt = blockIdx.y * 16 + fr;
    if (tt >= tokens) return;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int ee = blockIdx.x * 16 + q * 4 + c;
        if (ee < n_experts) logits[(size_t)tt * n_experts + ee] = (half_t)sum[c];
        else if (ee < rows) shared_logits[tt] = (half_t)sum[c];
    }
}

// out[t][:] = fp16(sum_j y[t][j][:] * scores[t][j]), fp32 products and sum in slot order;
// eight columns per lane, four slots' rows in flight.
__global__ __launch_bounds__(256) void moe_combine_kernel(const half_t* __restrict__ y,
                                                          const half_t* __restrict__ scores, long long n_chunks,
                                                          int slots, int D, half_t* __restrict__ out) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n_chunks) return;
    const int chunks = D >> 3;
    const long long t = i / chunks;
    const int c = (int)(i % chunks) * 8;
    const half_t* yt = y + t * slots * D + c;
    const half_t* st = scores + t * slots;
    float acc[8] = {};
    for (int j0 = 0; j0 < slots; j0 += 4) {
        uint4_t q[4];
        float s[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int jj = j0 + j < slots ? j0 + j : slots - 1;
            q[j] = *reinterpret_cast<const uint4_t*>(yt + (size_t)jj * D);
            s[j] = (float)st[jj];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j0 + j < slots) {
                float v[8];
                halfs_to_floats(q[j], v);
#pragma unroll
                for (int k = 0; k < 8; k++) acc[k] = __builtin_fmaf(v[k], s[j], acc[k]);
            }
        }
    }
    half8_t o;
#pragma unroll
    for (int k = 0; k < 8; k++) o[k] = (half_t)acc[k];
    *reinterpret_cast<half8_t*>(out + t * D + c) = o;
}

template <typename T>
static int launch_route(const void* logits, const void* shared_logits, const uint16_t* x, const uint16_t* w_shared,
                        int D, int tokens, int n_experts, int top_k, int norm, int32_t* indices, uint16_t* scores, hipStream_t stream) {
    auto go = [&](auto epl) {
        moe_route_kernel<T, epl.value><<<dim3((unsigned)((tokens + 3) / 4)), dim3(256), 0, stream>>>(
            static_cast<const T*>(logits), static_cast<const T*>(shared_logits), reinterpret_cast<const half_t*>(x),
            reinterpret_cast<const half_t*>(w_shared), D, tokens, n_experts, top_k, norm, indices, reinterpret_cast<half_t*>(scores));
        return launch_status();
    };
    if (n_experts <= 64) return go(std::integral_constant<int, 1>{});
    if (n_experts <= 128) return go(std::integral_constant<int, 2>{});
    if (n_experts <= 256) return go(std::integral_constant<int, 4>{});
    if (n_experts <= 512) return go(std::integral_constant<int, 8>{});
    return go(std::integral_constant<int, 16>{});
}

int launch_moe_route_groups(const uint16_t* logits, const uint16_t* shared_logits, int tokens, int n_experts, int top_k,
                            int norm, int32_t* indices, uint16_t* scores, int num_experts, int4* groups, int* arrived,
                            hipStream_t stream) {
    if (!logits || !indices || !scores || !groups || !arrived) return EXL3_E_NULL_POINTER;
    if (tokens < 1 || n_experts < 1 || top_k < 1 || top_k > n_experts ||
        n_experts + (shared_logits != nullptr) > num_experts || num_experts > kGroupMaxExperts ||
        tokens * (top_k + (shared_logits != nullptr)) > kGroupMaxSlots)
        return EXL3_E_BAD_SHAPE;
    if (n_experts > kRouteMaxExperts || top_k > kRouteMaxTopK) return EXL3_E_UNSUPPORTED;
    constexpr int kTokens = kGroupThreads / kWave;
    auto go = [&](auto epl) {
        moe_route_groups_kernel<epl.value><<<dim3((unsigned)((tokens + kTokens - 1) / kTokens)), dim3(kGroupThreads), 0, stream>>>(
            reinterpret_cast<const half_t*>(logits), reinterpret_cast<const half_t*>(shared_logits), tokens, n_experts,
            top_k, norm, indices, reinterpret_cast<half_t*>(scores), num_experts, groups, arrived);
        return launch_status();
    };
    if (n_experts <= 64) return go(std::integral_constant<int, 1>{});
    if (n_experts <= 128) return go(std::integral_constant<int, 2>{});
    if (n_experts <= 256) return go(std::integral_constant<int, 4>{});
    if (n_experts <= 512) return go(std::integral_constant<int, 8>{});
    return go(std::integral_constant<int, 16>{});
}

}  // namespace exl3

EXL3_EXPORT int exl3_moe_route(const void* logits, int logits_fp32, const void* shared_logits, int tokens,
                               int n_experts, int top_k, int norm, int32_t* indices, uint16_t* scores,
                               void* stream) {
    using namespace exl3;
    if (!logits || !indices || !scores) return EXL3_E_NULL_POINTER;
    if (tokens < 0 || n_experts < 1 || top_k < 1 || top_k > n_experts) return EXL3_E_BAD_SHAPE;
    if (n_experts > kRouteMaxExperts || top_k > kRouteMaxTopK) return EXL3_E_UNSUPPORTED;
    if (tokens == 0) return EXL3_OK;
    return logits_fp32 ? launch_route<float>(logits, shared_logits, nullptr, nullptr, 0, tokens, n_experts, top_k,
                                             norm, indices, scores, as_stream(stream))
                       : launch_route<half_t>(logits, shared_logits, nullptr, nullptr, 0, tokens, n_experts, top_k,
                                              norm, indices, scores, as_stream(stream));
}

EXL3_EXPORT int exl3_moe_route_shared(const uint16_t* logits, const uint16_t* x, int D, const uint16_t* w_shared,
                                      int tokens, int n_experts, int top_k, int norm, int32_t* indices,
                                      uint16_t* scores, void* stream) {
    using namespace exl3;
    if (!logits || !x || !w_shared || !indices || !scores) return EXL3_E_NULL_POINTER;
    if (tokens < 0 || n_experts < 1 || top_k < 1 || top_k > n_experts || D < 8 || D % 8) return EXL3_E_BAD_SHAPE;
    for (const void* p : {(const void*)x, (const void*)w_shared})
        if (reinterpret_cast<uintptr_t>(p) & 15) return EXL3_E_BAD_SHAPE;
    if (n_experts > kRouteMaxExperts || top_k > kRouteMaxTopK) return EXL3_E_UNSUPPORTED;
    if (tokens == 0) return EXL3_OK;
    return launch_route<half_t>(logits, nullptr, x, w_shared, D, tokens, n_experts, top_k, norm, indices, scores,
                                as_stream(stream));
}

EXL3_EXPORT int exl3_moe_gate(const uint16_t* x, int tokens, int D, const uint16_t* w, int n_experts,
                              const uint16_t* w_shared, uint16_t* logits, uint16_t* shared_logits, void* stream) {
    using namespace exl3;
    if (!x || !w || !logits || (w_shared && !shared_logits)) return EXL3_E_NULL_POINTER;
    if (tokens < 0 || tokens > 16 * 65535 || n_experts < 1 || D < 32 || D % 32) return EXL3_E_BAD_SHAPE;
    for (const void* p : {(const void*)x, (const void*)w, (const void*)w_shared})
        if (reinterpret_cast<uintptr_t>(p) & 15) return EXL3_E_BAD_SHAPE;
    if (tokens == 0) return EXL3_OK;
    const int rows = n_experts + (w_shared != nullptr);
    moe_gate_kernel<<<dim3((unsigned)((rows + 15) / 16), (unsigned)((tokens + 15) / 16)), dim3(kGateWaves * 64), 0,
                      as_stream(stream)>>>(
        reinterpret_cast<const half_t*>(x), reinterpret_cast<const half_t*>(w),
        reinterpret_cast<const half_t*>(w_shared), tokens, n_experts, D, reinterpret_cast<half_t*>(logits),
        reinterpret_cast<half_t*>(shared_logits));
    return launch_status();
}

EXL3_EXPORT int exl3_moe_combine(const uint16_t* y, const uint16_t* scores, int tokens, int slots, int D,
                                 uint16_t* out, void* stream) {
    using namespace exl3;
    if (!y || !scores || !out) return EXL3_E_NULL_POINTER;
    if (tokens < 0 || slots < 1 || D < 8 || D % 8) return EXL3_E_BAD_SHAPE;
    if ((reinterpret_cast<uintptr_t>(y) & 15) || (reinterpret_cast<uintptr_t>(out) & 15)) return EXL3_E_BAD_SHAPE;
    if (tokens == 0) return EXL3_OK;
    const long long n = (long long)tokens * (D / 8);
    const long long grid = (n + 255) / 256;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    moe_combine_kernel<<<dim3((unsigned)grid), dim3(256), 0, as_stream(stream)>>>(
        reinterpret_cast<const half_t*>(y), reinterpret_cast<const half_t*>(scores), n, slots, D,
        reinterpret_cast<half_t*>(out));
    return launch_status();
}
