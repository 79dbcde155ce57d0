// Routed MoE expert chain for a handful of tokens (decode / speculative verify):
// per slot (token t, expert e) gate and up GEMVs, GLU, down GEMV, each an EXL3
// linear with its own suh/svh. Only the selected experts' tile columns of the
// stacked trellises are read: the GEMV kernel is pointed at them through
// per-group tables built on the device from the routing indices.
//
// Two launches when the caller provides zeroed counters:
//   A. moe_gateup_kernel    per (slot, gate|up, 128 columns of H): input rotation
//                           in the wave, decode GEMV over D, workgroup sum; the
//                           last workgroup of a (slot, column block) adds the
//                           partial rows of gate and up, applies post-Hadamard,
//                           svh and the GLU and rotates the block for the down
//                           projection (a Hadamard block of H is exactly one
//                           128-column group of gate/up)
//   B. moe_down_kernel      per (slot, 128 columns of D): decode GEMV over H on
//                           the rotated block, sum, post-Hadamard, svh
//   (four waves per workgroup, one Hadamard block of the reduction each; with few
//   slots eight waves on half a block each, which doubles the loads in flight)
//   With several tokens and enough slots per expert (moe_*_grouped_kernel) the slots
//   that route to one expert share a pass over its weights, four batch rows at a time.
// Without counters the same result comes from a chain of five launches:
//   1. moe_prep_kernel      rotated activations per (slot, proj) + group tables
//   2. gemv_kernel          gate/up partial sums, fp32
//   3. moe_glu_kernel       split reduction, post-Hadamard, svh, GLU, then the
//                           down projection's input rotation
//   4. gemv_kernel          down partial sums
//   5. moe_finish_kernel    split reduction, post-Hadamard, per-expert svh
//
// Semantics follow the unfused chain of ponyexl3/mlx/exl3_moe.py:648-682 with
// the casts of ponyexl3/ref/forward.py:34,41,42; the Metal A2/B2 kernels
// (ponyexl3/mlx/exl3_moe.py:345-422) are what this replaces.
#include "exl3_device.hpp"
#include "exl3_host.hpp"
#include "exl3_glu.hpp"
#include "exl3_sort.hpp"
#include "exl3_groups.hpp"
#include "exl3_route.hpp"
#include "exl3_small.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

#pragma clang fp contract(off)

namespace exl3 {

// xh_gu[s][p][:] = fp16(had(x[t] * gu_suh[e][p])); also fills the group tables:
//   gate/up GEMV group (s, p, hg): sub = 2s+p, tile = (p*E + e)*(H/16) + 8*hg
//   down GEMV group (s, og):       sub = s,    tile = e*(D/16) + 8*og
__global__ __launch_bounds__(256) void moe_prep_kernel(
    const half_t* __restrict__ x, const int* __restrict__ indices,
    const half_t* __restrict__ gu_suh, half_t* __restrict__ xh_gu, int* __restrict__ gu_sub,
    int* __restrict__ gu_tile, int* __restrict__ dn_sub, int* __restrict__ dn_tile, int slots,
    int top_k, int E, int D, int H) {
    const int lane = threadIdx.x & 63;
    const int dblocks = D >> 7, hblocks = H >> 7;
    const int wave_id = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int gtid = blockIdx.x * 256 + threadIdx.x;
    if (gtid < slots * 2 * hblocks) {
        const int hg = gtid % hblocks, sp = gtid / hblocks;
        const int e = clamp_expert(indices[sp >> 1], E);
        gu_sub[gtid] = sp;
        gu_tile[gtid] = ((sp & 1) * E + e) * (H >> 4) + 8 * hg;
    }
    if (gtid < slots * dblocks) {
        const int og = gtid % dblocks, s = gtid / dblocks;
        dn_sub[gtid] = s;
        dn_tile[gtid] = clamp_expert(indices[s], E) * (D >> 4) + 8 * og;
    }
    if (wave_id >= slots * 2 * dblocks) return;
    const int blk = wave_id % dblocks;
    const int sp = wave_id / dblocks;
    const int s = sp >> 1, p = sp & 1;
    const int t = s / top_k;
    const int e = clamp_expert(indices[s], E);
    const half2_t xv = *reinterpret_cast<const half2_t*>(x + (size_t)t * D + blk * 128 + 2 * lane);
    const half2_t sv = *reinterpret_cast<const half2_t*>(gu_suh + ((size_t)e * 2 + p) * D +
                                                         blk * 128 + 2 * lane);
    float a = (float)xv.x * (float)sv.x, b = (float)xv.y * (float)sv.y;
    wht128_lanes(a, b, lane);
    half2_t o;
    o.x = (half_t)(a * kHadScaleF);
    o.y = (half_t)(b * kHadScaleF);
    *reinterpret_cast<half2_t*>(xh_gu + (size_t)sp * D + blk * 128 + 2 * lane) = o;
}

// One wave per (slot, 128-block of H): finishes gate and up, applies the GLU and
// rotates the result for the down projection.
__global__ __launch_bounds__(256) void moe_glu_kernel(
    const float* __restrict__ partial, int n_splits, size_t split_stride,
    const int* __restrict__ indices, const half_t* __restrict__ gu_svh,
    const half_t* __restrict__ dn_suh, half_t* __restrict__ xh_dn, int slots, int H, int E,
    int activation) {
    const int lane = threadIdx.x & 63;
    const int hblocks = H >> 7;
    const int wave_id = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wave_id >= slots * hblocks) return;
    const int blk = wave_id % hblocks, s = wave_id / hblocks;
    const int e = clamp_expert(indices[s], E);
    float v[2][2];
#pragma unroll
    for (int p = 0; p < 2; p++) {
        // partial layout: [split][(s*2+p)*H + h]
        const size_t off = ((size_t)s * 2 + p) * H + blk * 128 + 2 * lane;
        float2_t acc = *reinterpret_cast<const float2_t*>(partial + off);
        for (int i = 1; i < n_splits; i++) {
            const float2_t q = *reinterpret_cast<const float2_t*>(partial + i * split_stride + off);
            acc.x = acc.x + q.x;
            acc.y = acc.y + q.y;
        }
        float a = (float)(half_t)acc.x, b = (float)(half_t)acc.y;
        wht128_lanes(a, b, lane);
        const half2_t sv = *reinterpret_cast<const half2_t*>(gu_svh + (size_t)e * 2 * H + p * H +
                                                             blk * 128 + 2 * lane);
        v[p][0] = (float)(half_t)(a * kHadScaleF * (float)sv.x);
        v[p][1] = (float)(half_t)(b * kHadScaleF * (float)sv.y);
    }
    const float h0 = (float)(half_t)glu_act(v[0][0], v[1][0], activation);
    const float h1 = (float)(half_t)glu_act(v[0][1], v[1][1], activation);
    const half2_t ds =
        *reinterpret_cast<const half2_t*>(dn_suh + (size_t)e * H + blk * 128 + 2 * lane);
    float a = h0 * (float)ds.x, b = h1 * (float)ds.y;
    wht128_lanes(a, b, lane);
    half2_t o;
    o.x = (half_t)(a * kHadScaleF);
    o.y = (half_t)(b * kHadScaleF);
    *reinterpret_cast<half2_t*>(xh_dn + (size_t)s * H + blk * 128 + 2 * lane) = o;
}

__global__ __launch_bounds__(256) void moe_finish_kernel(
    const float* __restrict__ partial, int n_splits, size_t split_stride,
    const int* __restrict__ indices, const half_t* __restrict__ dn_svh, half_t* __restrict__ y,
    int slots, int D, int E) {
    const int lane = threadIdx.x & 63;
    const int dblocks = D >> 7;
    const int wave_id = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wave_id >= slots * dblocks) return;
    const int blk = wave_id % dblocks, s = wave_id / dblocks;
    const int e = clamp_expert(indices[s], E);
    const size_t off = (size_t)s * D + blk * 128 + 2 * lane;
    float2_t acc = *reinterpret_cast<const float2_t*>(partial + off);
    for (int i = 1; i < n_splits; i++) {
        const float2_t q = *reinterpret_cast<const float2_t*>(partial + i * split_stride + off);
        acc.x = acc.x + q.x;
        acc.y = acc.y + q.y;
    }
    float a = (float)(half_t)acc.x, b = (float)(half_t)acc.y;
    wht128_lanes(a, b, lane);
    const half2_t sv =
        *reinterpret_cast<const half2_t*>(dn_svh + (size_t)e * D + blk * 128 + 2 * lane);
    half2_t o;
    o.x = (half_t)(a * kHadScaleF * (float)sv.x);
    o.y = (half_t)(b * kHadScaleF * (float)sv.y);
    *reinterpret_cast<half2_t*>(y + off) = o;
}


// ---------------------------------------------------------------------------
// Fused chain: shared tail of both kernels. The NW waves of a workgroup are
// added through LDS in wave order; returns the two sums of this lane's columns
// (2*lane, 2*lane+1) to wave 0.
template <int NW>
__device__ __forceinline__ float2_t moe_wg_sum(float (*red)[128], const float (&acc)[1][2],
                                               int lane, int wave) {
    const int c0 = (lane >> 3) * 16 + (lane & 7);
    red[wave][c0] = acc[0][0];
    red[wave][c0 + 8] = acc[0][1];
    __syncthreads();
    float2_t v{red[0][2 * lane], red[0][2 * lane + 1]};
#pragma unroll
    for (int w = 1; w < NW; w++) {
        v.x = __fadd_rn(v.x, red[w][2 * lane]);
        v.y = __fadd_rn(v.y, red[w][2 * lane + 1]);
    }
    return v;
}

// Partial rows cross workgroups through device-scope accesses only (the XCDs'
// L2 caches are not coherent with each other): store, wait, bump the counter;
// the workgroup that sees `expected - 1` is the last one and reads them back.
__device__ __forceinline__ bool moe_publish(float* row, float2_t v, int* counter, int expected,
                                            int lane) {
    __hip_atomic_store(reinterpret_cast<uint64_t*>(row + 2 * lane),
                       __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int seen = 0;
    if (lane == 0)
        seen = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __shfl(seen, 0, kWave) == expected - 1;
}

// Eight partial rows in flight (a batch that runs past the last row re-reads that row and
// drops it, so that every batch is one round trip); added in index order.
__device__ __forceinline__ float2_t moe_sum_rows(const float* rows, int n, int lane) {
    float a = 0.f, b = 0.f;
    for (int s = 0; s < n; s += 8) {
        uint64_t v[8];
#pragma unroll
        for (int i = 0; i < 8; i++)
            v[i] = __hip_atomic_load(
                reinterpret_cast<const uint64_t*>(rows + (size_t)min(s + i, n - 1) * 128 + 2 * lane),
                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if (s + i < n) {
                const float2_t f = __builtin_bit_cast(float2_t, v[i]);
                a = __fadd_rn(a, f.x);
                b = __fadd_rn(b, f.y);
            }
        }
    }
    return float2_t{a, b};
}

// fp16(had128(fp16(sum)) / sqrt(128) * sv): the finish of one EXL3 linear on one
// 128-column block (ponyexl3/ref/forward.py:41-42).
__device__ __forceinline__ void moe_finish_block(float2_t sum, half2_t sv, int lane, float& o0,
                                                 float& o1) {
    float a = (float)(half_t)sum.x, b = (float)(half_t)sum.y;
    wht128_lanes(a, b, lane);
    o0 = (float)(half_t)(a * kHadScaleF * (float)sv.x);
    o1 = (float)(half_t)(b * kHadScaleF * (float)sv.y);
}

// Routing by the expert kernel itself, from the router's logits: 3.4 us in front of the first weights
// (8.0 -> 11.4 us) where a launch of its own in between takes 4.0 us and a gap of about 1, and 3.5 us of host time. Every wave finds the expert of its slot;
// one workgroup a token writes the token's row of the routing table for the launch behind.
// logits == nullptr: the table is there.
constexpr int kInlineRouteExperts = 256;  // four per lane
struct MoeRoute {
    const half_t* logits;  // fp16 [tokens][n_experts]
    const half_t* shared_logits;
    int n_experts, norm;
    half_t* scores;  // fp16 [tokens][top_k], top_k with the shared expert
};

// writes: by the first workgroup of a token's last slot, which chooses them all anyway.
__device__ __forceinline__ int moe_route_slot(const MoeRoute& r, int s, int top_k, int* indices, bool writes, int lane) {
    const int t = s / top_k, j = s - t * top_k, ranked = top_k - (r.shared_logits != nullptr);
    if (j == ranked && !writes) return r.n_experts;  // the shared expert
    int key[kInlineRouteExperts / 64];
    route_probabilities<half_t>(r.logits + (size_t)t * r.n_experts, r.n_experts, lane, key);
    RouteChoice c{0.f, 0};
    int e = r.n_experts;
    const int rounds = writes ? ranked : j + 1;
    for (int i = 0; i < rounds; i++) {
        const int chosen = route_next(key, lane, i, c);
        if (i == j) e = chosen;
    }
    if (writes) route_write<half_t>(c, lane, t, r.n_experts, ranked, r.norm, r.shared_logits != nullptr,
                                     r.shared_logits ? r.shared_logits[t] : (half_t)0.f, indices, r.scores);
    return e;
}

// Weighted sum over the slots of a token by the wave that stores the last of them: one 128-column block o of
// slot s goes to y[s] through the level that the XCDs share, the wave that completes
// (token, block) adds the token's slots in slot order (the arithmetic of moe_combine_kernel). A launch
// of its own behind the experts takes 2.4 us and a gap, this 1.6. scores == nullptr: rows only. The
// block at one token (2048 x 512, 8 of 256 experts): five launches 28.0 us, three 21.2.
struct MoeCombine {
    const half_t* scores;  // fp16 [tokens][top_k]
    half_t* out;           // fp16 [tokens][D]
    int* counters;         // int32 [tokens][D/128], zero on entry and exit
    int top_k;
};

__device__ __forceinline__ void moe_store_row(const MoeCombine& c, half_t* y, int s, int og, int D, half2_t o, int lane) {
    half_t* at = y + (size_t)s * D + og * 128 + 2 * lane;
    if (!c.scores) {
        *reinterpret_cast<half2_t*>(at) = o;
        return;
    }
    __hip_atomic_store(reinterpret_cast<uint32_t*>(at), half2_to_bits(o), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int t = s / c.top_k;
    int* counter = c.counters + (size_t)t * (D >> 7) + og;
    int seen = 0;
    if (lane == 0) seen = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__shfl(seen, 0, kWave) != c.top_k - 1) return;
    asm volatile("" ::: "memory");
    const half_t* row = y + (size_t)t * c.top_k * D + og * 128 + 2 * lane;
    const half_t* score = c.scores + (size_t)t * c.top_k;
    float a = 0.f, b = 0.f;
    for (int j0 = 0; j0 < c.top_k; j0 += 8) {
        uint32_t v[8];
        float w[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int jj = min(j0 + j, c.top_k - 1);
            v[j] = __hip_atomic_load(reinterpret_cast<const uint32_t*>(row + (size_t)jj * D), __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
            w[j] = (float)score[jj];
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (j0 + j < c.top_k) {
                const half2_t h = bits_to_half2(v[j]);
                a = __builtin_fmaf((float)h.x, w[j], a);
                b = __builtin_fmaf((float)h.y, w[j], b);
            }
    }
    half2_t sum;
    sum.x = (half_t)a;
    sum.y = (half_t)b;
    *reinterpret_cast<half2_t*>(c.out + (size_t)t * D + og * 128 + 2 * lane) = sum;
    if (lane == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// grid = (slots * 2 * H/128, ceil((D/128) / 4)); wave w of workgroup (gid, q) owns
// the Hadamard block 4q + w of D for slot s = gid / (2*hblocks), projection
// p = (gid / hblocks) & 1 and column block hg = gid % hblocks.
// part: fp32 [gid][n_wg][128]; counters[s*hblocks + hg] count 2*n_wg workgroups.
template <int K, int CB, int NW>
__global__ __launch_bounds__(NW * 64) void moe_gateup_kernel(
    const uint32_t* __restrict__ gu_trellis, const half_t* __restrict__ x,
    const int* __restrict__ indices, const half_t* __restrict__ gu_suh,
    const half_t* __restrict__ gu_svh, const half_t* __restrict__ dn_suh, half_t* xh_dn,
    float* part, int* counters, int top_k, int E, int D, int H, int activation) {
    __shared__ __attribute__((aligned(16))) half_t xs[NW][kXwRows<1>][kXwLd];
    __shared__ float red[NW][128];
    __shared__ float up_val[128];
    __shared__ int last_flag;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int dblocks = D >> 7, hblocks = H >> 7;
    const int n_wg = gridDim.y;
    const int gid = blockIdx.x;
    const int hg = gid % hblocks, sp = gid / hblocks;
    const int s = sp >> 1, p = sp & 1;
    const int e = clamp_expert(indices[s], E);
    constexpr bool kHalf = NW == 8;
    const int part_idx = blockIdx.y * NW + wave;
    const int blk = kHalf ? part_idx >> 1 : part_idx;
    const int tk0 = blk * 8 + (kHalf ? (part_idx & 1) * 4 : 0);
    float acc[1][2] = {{0.f, 0.f}};
    if (blk < dblocks) {
        const size_t row_words = (size_t)E * 2 * (H >> 4) * (8 * K);
        const uint32_t* base =
            gu_trellis + ((size_t)(p * E + e) * (H >> 4) + 8 * hg) * (8 * K) + lane * K;
        stream_block_rows<K, CB, 1, true, kHalf, true>(base, row_words, tk0, tk0 + (kHalf ? 4 : 8),
                                                 x + (size_t)(s / top_k) * D, (size_t)D, 1,
                                                 gu_suh + ((size_t)e * 2 + p) * D, xs[wave], lane,
                                                 acc);
    }
    const float2_t v = moe_wg_sum<NW>(red, acc, lane, wave);
    int* counter = counters + s * hblocks + hg;
    if (wave == 0) {
        const bool last = moe_publish(part + ((size_t)gid * n_wg + blockIdx.y) * 128, v, counter,
                                      2 * n_wg, lane);
        if (lane == 0) last_flag = last;
    }
    __syncthreads();
    if (!last_flag) return;
    asm volatile("" ::: "memory");
    // waves 0 and 1 finish gate and up, wave 0 then applies the GLU and rotates
    float f0 = 0.f, f1 = 0.f;
    if (wave < 2) {
        const int gid_p = (s * 2 + wave) * hblocks + hg;
        const float2_t sum = moe_sum_rows(part + (size_t)gid_p * n_wg * 128, n_wg, lane);
        const half2_t sv = *reinterpret_cast<const half2_t*>(
            gu_svh + (size_t)e * 2 * H + wave * H + hg * 128 + 2 * lane);
        moe_finish_block(sum, sv, lane, f0, f1);
        if (wave == 1) {
            up_val[2 * lane] = f0;
            up_val[2 * lane + 1] = f1;
        }
    }
    __syncthreads();
    if (wave != 0) return;
    const float h0 = (float)(half_t)glu_act(f0, up_val[2 * lane], activation);
    const float h1 = (float)(half_t)glu_act(f1, up_val[2 * lane + 1], activation);
    const half2_t ds =
        *reinterpret_cast<const half2_t*>(dn_suh + (size_t)e * H + hg * 128 + 2 * lane);
    float a = h0 * (float)ds.x, b = h1 * (float)ds.y;
    wht128_lanes(a, b, lane);
    half2_t o;
    o.x = (half_t)(a * kHadScaleF);
    o.y = (half_t)(b * kHadScaleF);
    *reinterpret_cast<half2_t*>(xh_dn + (size_t)s * H + hg * 128 + 2 * lane) = o;
    if (lane == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Gate and up of one k-chunk in ONE workgroup of eight waves, reduced through 64-bit
// accumulators with returning atomics (see fix_word): waves 0..3 stream gate, waves
// 4..7 up, over the same Hadamard blocks of D - HALF: half a block each, two blocks
// per workgroup; else a block each, four blocks per workgroup. Wave 0 adds the
// workgroup's 128 gate sums and 128 up sums to the accumulators of (slot, column
// block); the workgroup whose add completes the first gate column is the finisher: it
// holds (or polls for, if other workgroups' adds were interleaved with its own) both
// totals, so it goes on to post-Hadamard, svh, GLU and the rotation for the down
// projection without another trip through memory. One round trip instead of the
// three of store / counter / reload.
// grid = (slots * H/128, chunks); sums: uint64 [slots][2][H], zero on entry and exit.
template <int K, int CB, bool HALF>
__global__ __launch_bounds__(512) void moe_gateup_pair_kernel(
    const uint32_t* __restrict__ gu_trellis, const half_t* __restrict__ x, int* indices, MoeRoute route,
    const half_t* __restrict__ gu_suh, const half_t* __restrict__ gu_svh,
    const half_t* __restrict__ dn_suh, half_t* xh_dn, unsigned long long* sums, int top_k, int E, int D, int H,
    int activation, int* status, int spin_limit) {
    __shared__ __attribute__((aligned(16))) half_t xs[8][kXwRows<1>][kXwLd];
    __shared__ float red[8][128];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int dblocks = D >> 7, hblocks = H >> 7;
    const int n_chunks = gridDim.y;
    const int gid = blockIdx.x;
    const int hg = gid % hblocks, s = gid / hblocks;
    const int p = wave >> 2, j = wave & 3;
    const bool writes = blockIdx.y == 0 && hg == 0 && wave == 0 && s % top_k == top_k - 1;
    const int e = clamp_expert(route.logits ? moe_route_slot(route, s, top_k, indices, writes, lane) : indices[s], E);
    const int blk = HALF ? blockIdx.y * 2 + (j >> 1) : blockIdx.y * 4 + j;
    const int tk0 = blk * 8 + (HALF ? (j & 1) * 4 : 0);
    float acc[1][2] = {{0.f, 0.f}};
    if (blk < dblocks) {
        const size_t row_words = (size_t)E * 2 * (H >> 4) * (8 * K);
        const uint32_t* base =
            gu_trellis + ((size_t)(p * E + e) * (H >> 4) + 8 * hg) * (8 * K) + lane * K;
        stream_block_rows<K, CB, 1, true, HALF, true>(base, row_words, tk0, tk0 + (HALF ? 4 : 8),
                                                x + (size_t)(s / top_k) * D, (size_t)D, 1,
                                                gu_suh + ((size_t)e * 2 + p) * D, xs[wave], lane,
                                                acc);
    }
    // Scales of what follows the reduction, requested in front of it: its round trip hides theirs (behind it a shared-expert
    // block of 8 of 256 experts of 2048 x 512 takes 24.5 us a token, so 24.2; without a shared expert there is no difference). In front of
    // the weights they, and the choices of a table's row that is written behind them, cost five registers a lane: at K = 6 and 7 a
    // CU then holds two workgroups in place of three (MCG: three of four), and 7 tokens of 6 slots, 257 experts of 1792 x 512, take 38.9 us in
    // place of 36.8 at K = 6, 6 tokens of 5 slots of 2048 x 384 30.1 in place of 28.3 at K = 7.
    half2_t svg, svu, ds;
    if (wave == 0) {
        const half_t* svh_e = gu_svh + (size_t)e * 2 * H + hg * 128 + 2 * lane;
        svg = *reinterpret_cast<const half2_t*>(svh_e);
        svu = *reinterpret_cast<const half2_t*>(svh_e + H);
        ds = *reinterpret_cast<const half2_t*>(dn_suh + (size_t)e * H + hg * 128 + 2 * lane);
    }
    const int c0 = (lane >> 3) * 16 + (lane & 7);
    red[wave][c0] = acc[0][0];
    red[wave][c0 + 8] = acc[0][1];
    __syncthreads();
    if (wave != 0) return;
    const int bits = fix_count_bits(n_chunks);
    // word q of a lane: projection q >> 1, column 2*lane + (q & 1); wave order within a projection
    unsigned long long w[4];
    unsigned long long* slot[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int col = 2 * lane + (q & 1), w0 = (q >> 1) * 4;
        float v = red[w0][col];
#pragma unroll
        for (int i = 1; i < 4; i++) v = __fadd_rn(v, red[w0 + i][col]);
        slot[q] = sums + ((size_t)s * 2 + (q >> 1)) * H + hg * 128 + col;
        const unsigned long long a = fix_word(v, bits);
        w[q] = __hip_atomic_fetch_add(slot[q], a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + a;
    }
    if (__builtin_amdgcn_readfirstlane(fix_count(w[0], bits)) != n_chunks) return;
    auto all_complete = [&]() {
        bool ok = true;
#pragma unroll
        for (int q = 0; q < 4; q++) ok = ok && fix_count(w[q], bits) == n_chunks;
        return __ballot(ok) == ~0ull;
    };
    bool complete = all_complete();
    for (int spin = 0; !complete && spin < spin_limit; spin++) {
#pragma unroll
        for (int q = 0; q < 4; q++)
            w[q] = __hip_atomic_load(slot[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        complete = all_complete();
    }
    if (!complete) {
        // the counts never became complete (array not zero on entry, or shared with an
        // overlapping call): NaN for this block of the down projection's input (and so
        // for the slot's output), status word set, accumulators left for the caller to zero
        if (status && lane == 0)
            __hip_atomic_fetch_or(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        half2_t bad;
        bad.x = bad.y = bits_to_half(0x7E00);
        *reinterpret_cast<half2_t*>(xh_dn + (size_t)s * H + hg * 128 + 2 * lane) = bad;
        return;
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
        __hip_atomic_store(slot[q], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    float g0, g1, u0, u1;
    moe_finish_block(float2_t{fix_value(w[0], bits), fix_value(w[1], bits)}, svg, lane, g0, g1);
    moe_finish_block(float2_t{fix_value(w[2], bits), fix_value(w[3], bits)}, svu, lane, u0, u1);
    const float h0 = (float)(half_t)glu_act(g0, u0, activation);
    const float h1 = (float)(half_t)glu_act(g1, u1, activation);
    float a = h0 * (float)ds.x, b = h1 * (float)ds.y;
    wht128_lanes(a, b, lane);
    half2_t o;
    o.x = (half_t)(a * kHadScaleF);
    o.y = (half_t)(b * kHadScaleF);
    *reinterpret_cast<half2_t*>(xh_dn + (size_t)s * H + hg * 128 + 2 * lane) = o;
}

// grid = (slots * D/128, ceil((H/128) / 4)); slot s = gid / dblocks, column block
// og = gid % dblocks. xh_dn is already rotated. part: fp32 [gid][n_wg][128].
template <int K, int CB, int NW>
__global__ __launch_bounds__(NW * 64) void moe_down_kernel(
    const uint32_t* __restrict__ dn_trellis, const half_t* __restrict__ xh_dn,
    const int* __restrict__ indices, const half_t* __restrict__ dn_svh, half_t* y, float* part, int* counters,
    MoeCombine combine, int E, int D, int H) {
    __shared__ __attribute__((aligned(16))) half_t xs[NW][kXwRows<1>][kXwLd];
    __shared__ float red[NW][128];
    __shared__ int last_flag;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int dblocks = D >> 7, hblocks = H >> 7;
    const int n_wg = gridDim.y;
    const int gid = blockIdx.x;
    const int og = gid % dblocks, s = gid / dblocks;
    const int e = clamp_expert(indices[s], E);
    constexpr bool kHalf = NW == 8;
    const int part_idx = blockIdx.y * NW + wave;
    const int blk = kHalf ? part_idx >> 1 : part_idx;
    const int tk0 = blk * 8 + (kHalf ? (part_idx & 1) * 4 : 0);
    float acc[1][2] = {{0.f, 0.f}};
    if (blk < hblocks) {
        const size_t row_words = (size_t)E * (D >> 4) * (8 * K);
        const uint32_t* base = dn_trellis + ((size_t)e * (D >> 4) + 8 * og) * (8 * K) + lane * K;
        stream_block_rows<K, CB, 1, false, kHalf>(base, row_words, tk0, tk0 + (kHalf ? 4 : 8),
                                                  xh_dn + (size_t)s * H, (size_t)H, 1, nullptr,
                                                  xs[wave], lane, acc);
    }
    half2_t sv;  // (requested behind the weights, as in moe_gateup_pair_kernel)
    if (wave == 0) sv = *reinterpret_cast<const half2_t*>(dn_svh + (size_t)e * D + og * 128 + 2 * lane);
    float2_t v = moe_wg_sum<NW>(red, acc, lane, wave);
    if (n_wg > 1) {
        int* counter = counters + gid;
        if (wave == 0) {
            const bool last = moe_publish(part + ((size_t)gid * n_wg + blockIdx.y) * 128, v,
                                          counter, n_wg, lane);
            if (lane == 0) last_flag = last;
        }
        __syncthreads();
        if (!last_flag || wave != 0) return;
        asm volatile("" ::: "memory");
        v = moe_sum_rows(part + (size_t)gid * n_wg * 128, n_wg, lane);
        if (lane == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else if (wave != 0) {
        return;
    }
    float o0, o1;
    moe_finish_block(v, sv, lane, o0, o1);
    half2_t o;
    o.x = (half_t)o0;
    o.y = (half_t)o1;
    moe_store_row(combine, y, s, og, D, o, lane);
}

// ---------------------------------------------------------------------------
// The same chain with the slots grouped by expert. With several tokens, slots that
// route to the same expert share one pass over its weights: a workgroup set per entry of the list
// that make_slot_groups() has left, up to four batch rows each (the matrix instructions carry
// four rows at the price of one). The grid holds as many sets as there could be groups (one per
// slot); those past the list leave after one scalar load. Per row the arithmetic, the partial rows and the
// counters are those of the kernels above with partial rows, so the results are bit-identical to theirs where both take
// half blocks, or both whole ones (moe_half_blocks()), and the down weights are not rounded (moe_exact_down()).

struct SlotGroup {
    int n;               // rows; 0 = past the list
    int expert;
    int s0, s1, s2, s3;  // the rows' slots; past n: s0
};

// (both entries are requested together)
__device__ __forceinline__ SlotGroup load_slot_group(const int4* __restrict__ list, int i) {
    const int count = list[0].x;
    const int4 v = list[1 + i];
    SlotGroup g;
    g.n = i < count ? v.y : 0;
    g.expert = v.x;
    g.s0 = v.z & 0xFFFF;
    g.s1 = g.n > 1 ? (int)((uint32_t)v.z >> 16) : g.s0;
    g.s2 = g.n > 2 ? v.w & 0xFFFF : g.s0;
    g.s3 = g.n > 3 ? (int)((uint32_t)v.w >> 16) : g.s0;
    return g;
}

__device__ __forceinline__ int group_slot(const SlotGroup& g, int r) {
    return r == 1 ? g.s1 : (r == 2 ? g.s2 : (r == 3 ? g.s3 : g.s0));
}

// The list for a routing table that is there already.
__global__ __launch_bounds__(kGroupThreads) void moe_groups_kernel(const int* __restrict__ indices, int slots, int E,
                                                                   int4* list) {
    __shared__ GroupScratch scratch;
    make_slot_groups([&](int s) { return clamp_expert(indices[s], E); }, slots, E, list, scratch);
}

// The NW waves' sums of batch row r, added in wave order.
template <int NW>
__device__ __forceinline__ float2_t moe_row_sum(const float (*red)[kGroupRows][128], int r,
                                                int lane) {
    float2_t v{red[0][r][2 * lane], red[0][r][2 * lane + 1]};
#pragma unroll
    for (int w = 1; w < NW; w++) {
        v.x = __fadd_rn(v.x, red[w][r][2 * lane]);
        v.y = __fadd_rn(v.y, red[w][r][2 * lane + 1]);
    }
    return v;
}

// Grid and arguments as moe_gateup_kernel, the list in place of the routing table. Wave r of a
// workgroup takes batch row r through the split reduction and, as the last
// contributor of (slot, column block), through gate finish, up finish, GLU and the
// rotation for the down projection.
template <int K, int CB, int NW>
__global__ __launch_bounds__(NW * 64) void moe_gateup_grouped_kernel(
    const uint32_t* __restrict__ gu_trellis, const half_t* __restrict__ x,
    const int4* __restrict__ groups, const half_t* __restrict__ gu_suh,
    const half_t* __restrict__ gu_svh, const half_t* __restrict__ dn_suh, half_t* xh_dn,
    float* part, int* counters, int top_k, int E, int D, int H, int activation) {
    __shared__ __attribute__((aligned(16))) half_t xs[NW][kXwRows<kGroupRows>][kXwLd];
    __shared__ float red[NW][kGroupRows][128];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int dblocks = D >> 7, hblocks = H >> 7;
    const int n_wg = gridDim.y;
    const int gid = blockIdx.x;
    const int hg = gid % hblocks, sp = gid / hblocks;
    const int p = sp & 1;
    const SlotGroup grp = load_slot_group(groups, sp >> 1);
    if (grp.n == 0) return;
    const int e = grp.expert;
    constexpr bool kHalf = NW == 8;
    const int part_idx = blockIdx.y * NW + wave;
    const int blk = kHalf ? part_idx >> 1 : part_idx;
    const int tk0 = blk * 8 + (kHalf ? (part_idx & 1) * 4 : 0);
    float acc[kGroupRows][2];
#pragma unroll
    for (int m = 0; m < kGroupRows; m++) acc[m][0] = acc[m][1] = 0.f;
    if (blk < dblocks) {
        const size_t row_words = (size_t)E * 2 * (H >> 4) * (8 * K);
        const uint32_t* base =
            gu_trellis + ((size_t)(p * E + e) * (H >> 4) + 8 * hg) * (8 * K) + lane * K;
        const half_t* xrow[kGroupRows];
#pragma unroll
        for (int m = 0; m < kGroupRows; m++) xrow[m] = x + (size_t)(group_slot(grp, m) / top_k) * D;
        stream_block_rows_at<K, CB, kGroupRows, true, kHalf, true, true>(
            base, row_words, tk0, tk0 + (kHalf ? 4 : 8), xrow, grp.n, gu_suh + ((size_t)e * 2 + p) * D, xs[wave],
            lane, acc);
    }
    const int c0 = (lane >> 3) * 16 + (lane & 7);
#pragma unroll
    for (int m = 0; m < kGroupRows; m++) {
        red[wave][m][c0] = acc[m][0];
        red[wave][m][c0 + 8] = acc[m][1];
    }
    __syncthreads();
    if (wave >= grp.n) return;
    const int sr = group_slot(grp, wave);
    const float2_t v = moe_row_sum<NW>(red, wave, lane);
    int* counter = counters + sr * hblocks + hg;
    const size_t gid_r = ((size_t)sr * 2 + p) * hblocks + hg;
    if (!moe_publish(part + (gid_r * n_wg + blockIdx.y) * 128, v, counter, 2 * n_wg, lane)) return;
    asm volatile("" ::: "memory");
    // both projections' partial rows in flight together, and the scales
    const half_t* svh_e = gu_svh + (size_t)e * 2 * H + hg * 128 + 2 * lane;
    const half2_t svg = *reinterpret_cast<const half2_t*>(svh_e), svu = *reinterpret_cast<const half2_t*>(svh_e + H);
    const half2_t ds = *reinterpret_cast<const half2_t*>(dn_suh + (size_t)e * H + hg * 128 + 2 * lane);
    const float* rows_g = part + (((size_t)sr * 2) * hblocks + hg) * n_wg * 128;
    const float* rows_u = part + (((size_t)sr * 2 + 1) * hblocks + hg) * n_wg * 128;
    float2_t sg{0.f, 0.f}, su{0.f, 0.f};
    for (int s0 = 0; s0 < n_wg; s0 += 4) {  // four rows of each projection per round trip
        uint64_t vg[4], vu[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t off = (size_t)min(s0 + i, n_wg - 1) * 128 + 2 * lane;
            vg[i] = __hip_atomic_load(reinterpret_cast<const uint64_t*>(rows_g + off),
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            vu[i] = __hip_atomic_load(reinterpret_cast<const uint64_t*>(rows_u + off),
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (s0 + i < n_wg) {
                const float2_t fg = __builtin_bit_cast(float2_t, vg[i]);
                const float2_t fu = __builtin_bit_cast(float2_t, vu[i]);
                sg.x = __fadd_rn(sg.x, fg.x);
                sg.y = __fadd_rn(sg.y, fg.y);
                su.x = __fadd_rn(su.x, fu.x);
                su.y = __fadd_rn(su.y, fu.y);
            }
        }
    }
    float g0, g1, u0, u1;
    moe_finish_block(sg, svg, lane, g0, g1);
    moe_finish_block(su, svu, lane, u0, u1);
    const float h0 = (float)(half_t)glu_act(g0, u0, activation);
    const float h1 = (float)(half_t)glu_act(g1, u1, activation);
    float a = h0 * (float)ds.x, b = h1 * (float)ds.y;
    wht128_lanes(a, b, lane);
    half2_t o;
    o.x = (half_t)(a * kHadScaleF);
    o.y = (half_t)(b * kHadScaleF);
    *reinterpret_cast<half2_t*>(xh_dn + (size_t)sr * H + hg * 128 + 2 * lane) = o;
    if (lane == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Grid and arguments as moe_down_kernel, the list in place of the routing table; wave r finishes
// batch row r. EXACT: weights rounded to fp16 before the product (moe_exact_down()).
template <int K, int CB, int NW, bool EXACT>
__global__ __launch_bounds__(NW * 64) void moe_down_grouped_kernel(
    const uint32_t* __restrict__ dn_trellis, const half_t* __restrict__ xh_dn,
    const int4* __restrict__ groups, const half_t* __restrict__ dn_svh, half_t* y, float* part, int* counters,
    MoeCombine combine, int E, int D, int H) {
    __shared__ __attribute__((aligned(16))) half_t xs[NW][kXwRows<kGroupRows>][kXwLd];
    __shared__ float red[NW][kGroupRows][128];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int dblocks = D >> 7, hblocks = H >> 7;
    const int n_wg = gridDim.y;
    const int gid = blockIdx.x;
    const int og = gid % dblocks;
    const SlotGroup grp = load_slot_group(groups, gid / dblocks);
    if (grp.n == 0) return;
    const int e = grp.expert;
    constexpr bool kHalf = NW == 8;
    const int part_idx = blockIdx.y * NW + wave;
    const int blk = kHalf ? part_idx >> 1 : part_idx;
    const int tk0 = blk * 8 + (kHalf ? (part_idx & 1) * 4 : 0);
    float acc[kGroupRows][2];
#pragma unroll
    for (int m = 0; m < kGroupRows; m++) acc[m][0] = acc[m][1] = 0.f;
    if (blk < hblocks) {
        const size_t row_words = (size_t)E * (D >> 4) * (8 * K);
        const uint32_t* base = dn_trellis + ((size_t)e * (D >> 4) + 8 * og) * (8 * K) + lane * K;
        const half_t* xrow[kGroupRows];
#pragma unroll
        for (int m = 0; m < kGroupRows; m++) xrow[m] = xh_dn + (size_t)group_slot(grp, m) * H;
        stream_block_rows_at<K, CB, kGroupRows, false, kHalf, true, EXACT>(
            base, row_words, tk0, tk0 + (kHalf ? 4 : 8), xrow, grp.n, nullptr, xs[wave], lane, acc);
    }
    const int c0 = (lane >> 3) * 16 + (lane & 7);
#pragma unroll
    for (int m = 0; m < kGroupRows; m++) {
        red[wave][m][c0] = acc[m][0];
        red[wave][m][c0 + 8] = acc[m][1];
    }
    __syncthreads();
    if (wave >= grp.n) return;
    const int sr = group_slot(grp, wave);
    const half2_t sv = *reinterpret_cast<const half2_t*>(dn_svh + (size_t)e * D + og * 128 + 2 * lane);  // (behind the early exit: eight waves of K = 8 stay at 64 registers)
    float2_t v = moe_row_sum<NW>(red, wave, lane);
    if (n_wg > 1) {
        const size_t gid_r = (size_t)sr * dblocks + og;
        int* counter = counters + gid_r;
        if (!moe_publish(part + (gid_r * n_wg + blockIdx.y) * 128, v, counter, n_wg, lane)) return;
        asm volatile("" ::: "memory");
        v = moe_sum_rows(part + gid_r * n_wg * 128, n_wg, lane);
        if (lane == 0) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    float o0, o1;
    moe_finish_block(v, sv, lane, o0, o1);
    half2_t o;
    o.x = (half_t)o0;
    o.y = (half_t)o1;
    moe_store_row(combine, y, sr, og, D, o, lane);
}

struct MoeWorkspace {
    size_t xh_gu, xh_dn, tables, part_gu, part_dn;
    size_t o_xh_gu, o_xh_dn, o_tables, o_part_gu, o_part_dn, total;
    GemvPlan plan_gu, plan_dn;
    int g_gu, g_dn;
};

// Two-launch chain: whether the waves take half Hadamard blocks, eight to a workgroup, instead of whole
// ones, four to a workgroup (same workgroups, same partial rows). Every slot on its own: where the gate/up launch
// would have fewer than 3200 waves of whole blocks, three to a SIMD: twice the loads in flight then count for
// more than a second rotation (block of 8 slots a token, 256 experts of 2048 x 512: 1 token 22.8 -> 21.1 us, 3 tokens 29.5 ->
// 29.3; 192 of 1536 x 512, 35 slots 29.9 and 32.5, 42 slots 34.3 and 38.1). Grouped slots: below 4096, and from
// K = 5 on always, where the four tile rows that a wave has in flight take 80 registers and more and whole blocks wait
// for their refills (20 tokens of 7 slots, 129 experts of 1664 x 512 K = 4 / 5 / 6 / 8 58.5 -> 58.0, 60.8 -> 59.0, 65.8 ->
// 61.9, 76.4 -> 66.6; 40 of 8 slots, 257 of 2048 x 512 K = 4 115 and 124, K = 8 175 -> 148). EXL3_MOE_HALF_BELOW,
// where it is set, takes the place of both lines.
static bool moe_half_blocks(long long whole_waves, bool grouped, int K) {
    static const int set = env_int("EXL3_MOE_HALF_BELOW", -1, 0, 1 << 20);
    if (set >= 0) return whole_waves < set;
    return grouped ? K >= 5 || whole_waves < 4096 : whole_waves < 3200;
}

// Two-launch chain with several tokens: slots of the same expert in one workgroup (1) or
// every slot on its own (0).
static bool moe_group_slots() {
    static const int v = env_int("EXL3_MOE_GROUP", 1, 0, 1);
    return v != 0;
}

// Calls of a size that the sorted prefill kernels also serve get the rounded weights of those in the down
// projection too, so that the result is no further from the reference's arithmetic whichever is faster
// (7.1e-4 of the output with unsummed halves, 6.8e-4 with rounded weights, against 64 bits). The sizes from which on callers
// turn to the prefill are their own (EXL3SwitchGLU starts out with these); exl3_moe_groups_rounded tells them what holds here.
static bool moe_exact_down(int tokens, int slots, int num_experts) {
    return tokens >= 24 && (slots > 512 || slots >= 2.5 * num_experts);
}

// Whether the slots are grouped by expert: where that is expected to spare enough passes over an expert's
// weights to pay for the list and for reducing through partial rows (3 us and more): a fifth of the slots and 18 of them, or 15 %
// and the passes over 11 experts of 2^20 weights per projection (choices taken as independent and even). From what every entry
// point knows, so that the block and its parts take the same way: that one of the experts may be a shared one, which all tokens have,
// is not asked. us, every slot on its own -> grouped, passes spared of slots: 11 tokens through 257 experts of 2048 x 512 with 9 slots a
// token, K = 4 15.6 of 99 63.2 -> 59.6, 14 tokens 25 of 126 72.5 -> 67.1; 24, 68 of 216 97 -> 86; 17 tokens, 3 of 64 experts of 1024 x 768,
// K = 5 15.3 of 51 38.3 -> 34.7; 10 tokens, 7 of 192 of 1280 x 768, K = 3 8.0 of 70 48.5 -> 51.0; 9 tokens, 8 of 256 of
// 1024 x 384 8.4 of 72 30.7 -> 33.9; 7 tokens, 6 of 33 of 1280 x 256 17 of 42 23.2 -> 26.5. Of 90 calls of 2 to 26 tokens with 11 to 30 % spared
// the 47 on the grouped side take 6 % less, four of them 2 to 8 % more; of the 43 on the single side fourteen would take 4 to 13 % less
// grouped (wide experts, MUL1), as many 3 to 11 % more. Calls that are to have rounded weights in the down
// projection, which the grouped kernel has, are grouped where fewer are spared, too (24 slots of 8 experts: 16).
static bool moe_groups_apply(int tokens, int top_k, int num_experts, int D, int H) {
    const long long slots = (long long)tokens * top_k;
    if (tokens < 2 || slots > kGroupMaxSlots || num_experts > kGroupMaxExperts || !moe_group_slots()) return false;
    const double passes = num_experts * (1.0 - std::pow(1.0 - std::min(1.0, (double)top_k / num_experts), tokens));
    const double spared = slots - passes;
    return spared >= std::max(18.0, 0.2 * slots) ||
           (spared >= std::max(11.0, 0.15 * slots) && spared * D * H >= 11.0 * (1 << 20)) ||
           (moe_exact_down(tokens, (int)slots, num_experts) && slots >= 2.5 * num_experts);
}

// Gate/up launches that would issue more atomics than this reduce through partial rows
// (the memory side retires about 75 000 returning atomics per microsecond).
static long long moe_max_atomics() {
    static const int v = env_int("EXL3_MOE_MAX_ATOMICS", 300000, 0, 1 << 30);
    return v;
}

static MoeWorkspace moe_workspace(int tokens, int top_k, int D, int H) {
    MoeWorkspace w{};
    const int slots = tokens * top_k;
    w.g_gu = slots * 2 * (H / 128);
    w.g_dn = slots * (D / 128);
    w.plan_gu = plan_gemv(1, D / 16, w.g_gu);
    w.plan_dn = plan_gemv(1, H / 16, w.g_dn);
    w.xh_gu = align_up((size_t)slots * 2 * D * 2, 256);
    w.xh_dn = align_up((size_t)slots * H * 2, 256);
    w.tables = align_up((size_t)2 * (w.g_gu + w.g_dn) * sizeof(int), 256);
    // partial rows per group: the chain's split plan or the fused kernels' one row per
    // workgroup of four Hadamard blocks, whichever is larger
    const int rows_gu = std::max(w.plan_gu.n_partials(), (D / 128 + 3) / 4);
    const int rows_dn = std::max(w.plan_dn.n_partials(), (H / 128 + 3) / 4);
    w.part_gu = align_up((size_t)rows_gu * w.g_gu * 128 * sizeof(float), 256);
    w.part_dn = align_up((size_t)rows_dn * w.g_dn * 128 * sizeof(float), 256);
    w.o_xh_gu = 0;
    w.o_xh_dn = w.o_xh_gu + w.xh_gu;
    w.o_tables = w.o_xh_dn + w.xh_dn;
    w.o_part_gu = w.o_tables + w.tables;
    w.o_part_dn = w.o_part_gu + w.part_gu;
    w.total = w.o_part_dn + w.part_dn;
    return w;
}

// ---------------------------------------------------------------------------
// Prefill glue: sort the (token, slot) pairs by expert and build the row-block
// table of the segmented GEMM in ONE launch of one workgroup (the pair counts are
// small: tokens * top_k), and finish gate/up + GLU + down rotation per sorted row.

constexpr int kSortThreads = 1024;

__global__ __launch_bounds__(kSortThreads) void moe_sort_kernel(SortArgs a) {
    extern __shared__ int cursor[];
    sort_pairs<kSortThreads>(a, blockIdx.x, cursor);
}

// One wave per (sorted row, 128-block of H): post-Hadamard + svh of the gate and up
// GEMM outputs, GLU, and the input rotation (dn_suh) of the down projection; the
// same steps and casts as moe_glu_kernel, on fp16 GEMM outputs.
__global__ __launch_bounds__(256) void moe_glu_rows_kernel(
    const half_t* __restrict__ g, const half_t* __restrict__ u, int n_rows, int H,
    const int* __restrict__ sidx, const half_t* __restrict__ gu_svh,
    const half_t* __restrict__ dn_suh, int E, int activation, half_t* __restrict__ xh_dn) {
    const int lane = threadIdx.x & 63;
    const int hblocks = H >> 7;
    const long long wave_id = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wave_id >= (long long)n_rows * hblocks) return;
    const int blk = (int)(wave_id % hblocks);
    const size_t r = (size_t)(wave_id / hblocks);
    const int e = clamp_expert(sidx[r], E);
    const size_t off = r * H + blk * 128 + 2 * lane;
    float v[2][2];
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const half2_t in = *reinterpret_cast<const half2_t*>((p ? u : g) + off);
        float a = (float)in.x, b = (float)in.y;
        wht128_lanes(a, b, lane);
        const half2_t sv = *reinterpret_cast<const half2_t*>(gu_svh + (size_t)e * 2 * H + p * H +
                                                             blk * 128 + 2 * lane);
        v[p][0] = (float)(half_t)(a * kHadScaleF * (float)sv.x);
        v[p][1] = (float)(half_t)(b * kHadScaleF * (float)sv.y);
    }
    const float h0 = (float)(half_t)glu_act(v[0][0], v[1][0], activation);
    const float h1 = (float)(half_t)glu_act(v[0][1], v[1][1], activation);
    const half2_t ds =
        *reinterpret_cast<const half2_t*>(dn_suh + (size_t)e * H + blk * 128 + 2 * lane);
    float a = h0 * (float)ds.x, b = h1 * (float)ds.y;
    wht128_lanes(a, b, lane);
    half2_t o;
    o.x = (half_t)(a * kHadScaleF);
    o.y = (half_t)(b * kHadScaleF);
    *reinterpret_cast<half2_t*>(xh_dn + off) = o;
}

static int launch_moe_sort(SortArgs a, hipStream_t stream) {
    // a workgroup per kSortThreads pairs (64 to a wave), up to kSortMaxGroups, from the size on where
    // one alone takes longer (1025 pairs 5.6 and 6.4 us, 2436 7.3 and 6.7)
    a.groups = a.n_pairs <= 2 * kSortThreads ? 1 : std::min(kSortMaxGroups, (a.n_pairs + kSortThreads - 1) / kSortThreads);
    a.staged = 1;
    a.staged = a.groups == 1 && sort_lds_ints(kSortThreads, a) * sizeof(int) <= (size_t)150 << 10;
    const size_t lds = sort_lds_ints(kSortThreads, a) * sizeof(int);
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(moe_sort_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return EXL3_E_LAUNCH;
    moe_sort_kernel<<<dim3((unsigned)a.groups), dim3(kSortThreads), lds, stream>>>(a);
    return launch_status();
}

}  // namespace exl3

EXL3_EXPORT size_t exl3_moe_workspace_bytes(int tokens, int top_k, int D, int H) {
    if (tokens < 1 || top_k < 1 || D < 128 || H < 128 || D % 128 || H % 128) return 0;
    return exl3::moe_workspace(tokens, top_k, D, H).total;
}

namespace exl3 {

// What the two entry points below share. route.logits: the table `indices` and route.scores are outputs;
// combine.out: y holds the slots' rows in between. `counters` for the combination: combine.counters.
struct MoeCall {
    const uint16_t* x;
    int tokens;
    int32_t* indices;
    int top_k;
    const uint16_t *gu_trellis, *gu_suh, *gu_svh, *dn_trellis, *dn_suh, *dn_svh;
    int num_experts, D, H, K, cb, activation;
    uint16_t* y;
    void* workspace;
    size_t workspace_bytes;
    int32_t* counters;
    size_t counters_len;
    MoeRoute route;
    MoeCombine combine;
};

static int moe_slots(const MoeCall& a, hipStream_t s) {
    const uint16_t *x = a.x, *gu_trellis = a.gu_trellis, *gu_suh = a.gu_suh, *gu_svh = a.gu_svh,
                   *dn_trellis = a.dn_trellis, *dn_suh = a.dn_suh, *dn_svh = a.dn_svh;
    int32_t *indices = a.indices, *counters = a.counters;
    const int tokens = a.tokens, top_k = a.top_k, num_experts = a.num_experts, D = a.D, H = a.H, K = a.K, cb = a.cb,
              activation = a.activation;
    const size_t counters_len = a.counters_len;
    uint16_t* y = a.y;
    if (int rc = check_k_cb(K, cb)) return rc;
    if (!x || !indices || !gu_trellis || !gu_suh || !gu_svh || !dn_trellis || !dn_suh || !dn_svh || !y || !a.workspace)
        return EXL3_E_NULL_POINTER;
    if (tokens < 1 || top_k < 1 || num_experts < 1 || D < 128 || H < 128 || D % 128 || H % 128 ||
        (long long)tokens * top_k > 4096)
        return EXL3_E_BAD_SHAPE;
    if (activation != 0 && activation != 1) return EXL3_E_UNSUPPORTED;
    // the router in a launch of its own (unless the kernel of a few slots does it), with the list of
    // groups if one is wanted
    auto route_table = [&](int4* groups = nullptr, int* arrived = nullptr) {
        const MoeRoute& r = a.route;
        if (!r.logits) {
            if (!groups) return (int)EXL3_OK;
            moe_groups_kernel<<<dim3(1), dim3(kGroupThreads), 0, s>>>(indices, tokens * top_k, num_experts, groups);
            return launch_status();
        }
        if (groups)
            return launch_moe_route_groups(reinterpret_cast<const uint16_t*>(r.logits),
                                           reinterpret_cast<const uint16_t*>(r.shared_logits), tokens, r.n_experts,
                                           top_k - (r.shared_logits != nullptr), r.norm, indices,
                                           reinterpret_cast<uint16_t*>(r.scores), num_experts, groups, arrived, s);
        return exl3_moe_route(r.logits, 0, r.shared_logits, tokens, r.n_experts, top_k - (r.shared_logits != nullptr),
                              r.norm, indices, reinterpret_cast<uint16_t*>(r.scores), s);
    };
    const MoeWorkspace w = moe_workspace(tokens, top_k, D, H);
    if (a.workspace_bytes < w.total) return EXL3_E_WORKSPACE;
    char* base = reinterpret_cast<char*>(a.workspace);
    half_t* xh_gu = reinterpret_cast<half_t*>(base + w.o_xh_gu);
    half_t* xh_dn = reinterpret_cast<half_t*>(base + w.o_xh_dn);
    int* gu_sub = reinterpret_cast<int*>(base + w.o_tables);
    int* gu_tile = gu_sub + w.g_gu;
    int* dn_sub = gu_tile + w.g_gu;
    int* dn_tile = dn_sub + w.g_dn;
    float* part_gu = reinterpret_cast<float*>(base + w.o_part_gu);
    float* part_dn = reinterpret_cast<float*>(base + w.o_part_dn);
    const int slots = tokens * top_k;

    if (counters && !exact_weights()) {
        // two launches: gate/up + GLU + rotation, then down
        const int hblocks = H / 128, dblocks = D / 128;
        if (counters_len < (size_t)slots * (hblocks + dblocks)) return EXL3_E_WORKSPACE;
        const bool grouped = moe_groups_apply(tokens, top_k, num_experts, D, H);
        const bool half = moe_half_blocks((long long)slots * 2 * hblocks * dblocks, grouped, K);
        // every slot on its own, few enough atomics, and counters large enough to hold
        // the accumulators (uint64 [slots][2][H], then the down launch's counters): gate
        // and up of a k-chunk in one workgroup, reduced through returning atomics
        const int pair_chunks = half ? (dblocks + 1) / 2 : (dblocks + 3) / 4;
        const size_t pair_ints = (size_t)slots * 2 * H * 2;
        const bool pair = !grouped && pair_chunks <= kFixMaxContributors &&
                          (long long)slots * 2 * H * pair_chunks <= moe_max_atomics() &&
                          counters_len >= pair_ints + (size_t)slots * dblocks &&
                          (reinterpret_cast<uintptr_t>(counters) & 7) == 0;
        const bool routes = pair && a.route.n_experts <= kInlineRouteExperts;
        // the list takes the place of the chain's tables (2 (2 H + D) / 128 ints per slot: four per slot
        // and four more from two slots on); the counter behind those of the two launches
        int4* const groups = grouped ? reinterpret_cast<int4*>(base + w.o_tables) : nullptr;
        if (!routes)
            if (int rc = route_table(groups, counters + (size_t)slots * (hblocks + dblocks))) return rc;
        auto chain = [&](auto k, auto c, auto nw) {
            constexpr int NW = nw.value;
            if (pair) {
                moe_gateup_pair_kernel<k.value, c.value, NW == 8>
                    <<<dim3((unsigned)(slots * hblocks), (unsigned)pair_chunks), dim3(512), 0, s>>>(
                        reinterpret_cast<const uint32_t*>(gu_trellis),
                        reinterpret_cast<const half_t*>(x), indices, routes ? a.route : MoeRoute{},
                        reinterpret_cast<const half_t*>(gu_suh),
                        reinterpret_cast<const half_t*>(gu_svh),
                        reinterpret_cast<const half_t*>(dn_suh), xh_dn,
                        reinterpret_cast<unsigned long long*>(counters), top_k, num_experts, D, H,
                        activation,
                        counters_status_word(counters, counters_len,
                                             pair_ints + (size_t)slots * dblocks),
                        reduction_spin_limit());
                if (int rc = launch_status()) return rc;
                moe_down_kernel<k.value, c.value, NW>
                    <<<dim3((unsigned)(slots * dblocks), (unsigned)((hblocks + 3) / 4)),
                       dim3(NW * 64), 0, s>>>(reinterpret_cast<const uint32_t*>(dn_trellis), xh_dn,
                                              indices, reinterpret_cast<const half_t*>(dn_svh),
                                              reinterpret_cast<half_t*>(y), part_dn,
                                              counters + pair_ints, a.combine, num_experts, D, H);
                return launch_status();
            }
            if (grouped) {
                moe_gateup_grouped_kernel<k.value, c.value, NW>
                    <<<dim3((unsigned)(slots * 2 * hblocks), (unsigned)((dblocks + 3) / 4)),
                       dim3(NW * 64), 0, s>>>(reinterpret_cast<const uint32_t*>(gu_trellis),
                                              reinterpret_cast<const half_t*>(x), groups,
                                              reinterpret_cast<const half_t*>(gu_suh),
                                              reinterpret_cast<const half_t*>(gu_svh),
                                              reinterpret_cast<const half_t*>(dn_suh), xh_dn,
                                              part_gu, counters, top_k, num_experts, D, H,
                                              activation);
                if (int rc = launch_status()) return rc;
                auto down = [&](auto exact) {
                    moe_down_grouped_kernel<k.value, c.value, NW, exact.value>
                        <<<dim3((unsigned)(slots * dblocks), (unsigned)((hblocks + 3) / 4)),
                           dim3(NW * 64), 0, s>>>(reinterpret_cast<const uint32_t*>(dn_trellis), xh_dn,
                                                  groups, reinterpret_cast<const half_t*>(dn_svh),
                                                  reinterpret_cast<half_t*>(y), part_dn,
                                                  counters + (size_t)slots * hblocks, a.combine,
                                                  num_experts, D, H);
                };
                if (moe_exact_down(tokens, slots, num_experts)) down(std::true_type{});
                else down(std::false_type{});
                return launch_status();
            }
            moe_gateup_kernel<k.value, c.value, NW>
                <<<dim3((unsigned)(slots * 2 * hblocks), (unsigned)((dblocks + 3) / 4)),
                   dim3(NW * 64), 0, s>>>(reinterpret_cast<const uint32_t*>(gu_trellis),
                                          reinterpret_cast<const half_t*>(x), indices,
                                          reinterpret_cast<const half_t*>(gu_suh),
                                          reinterpret_cast<const half_t*>(gu_svh),
                                          reinterpret_cast<const half_t*>(dn_suh), xh_dn, part_gu,
                                          counters, top_k, num_experts, D, H, activation);
            if (int rc = launch_status()) return rc;
            moe_down_kernel<k.value, c.value, NW>
                <<<dim3((unsigned)(slots * dblocks), (unsigned)((hblocks + 3) / 4)), dim3(NW * 64),
                   0, s>>>(reinterpret_cast<const uint32_t*>(dn_trellis), xh_dn, indices,
                           reinterpret_cast<const half_t*>(dn_svh), reinterpret_cast<half_t*>(y),
                           part_dn, counters + (size_t)slots * hblocks, a.combine, num_experts, D, H);
            return launch_status();
        };
        return dispatch_k_cb(K, cb, [&](auto k, auto c) {
            return half ? chain(k, c, std::integral_constant<int, 8>{})
                        : chain(k, c, std::integral_constant<int, 4>{});
        });
    }

    if (int rc = route_table()) return rc;
    {
        const int waves = slots * 2 * (D / 128);
        const int threads = waves * 64 > w.g_gu ? waves * 64 : w.g_gu;
        const int need = threads > w.g_dn ? threads : w.g_dn;
        moe_prep_kernel<<<dim3((need + 255) / 256), dim3(256), 0, s>>>(
            reinterpret_cast<const half_t*>(x), indices, reinterpret_cast<const half_t*>(gu_suh),
            xh_gu, gu_sub, gu_tile, dn_sub, dn_tile, slots, top_k, num_experts, D, H);
        if (int rc = launch_status()) return rc;
    }
    // gate/up: rows = 1, n_sub = 2*slots activation rows, one group per (slot, proj, hg)
    if (int rc = launch_gemv_partials(reinterpret_cast<const uint16_t*>(xh_gu), 1, slots * 2,
                                      gu_trellis, D / 16, num_experts * 2 * (H / 16), K, cb,
                                      gu_sub, gu_tile, w.g_gu, part_gu, w.plan_gu, s))
        return rc;
    {
        const int waves = slots * (H / 128);
        moe_glu_kernel<<<dim3((waves + 3) / 4), dim3(256), 0, s>>>(
            part_gu, w.plan_gu.n_partials(), (size_t)w.g_gu * 128, indices,
            reinterpret_cast<const half_t*>(gu_svh), reinterpret_cast<const half_t*>(dn_suh), xh_dn,
            slots, H, num_experts, activation);
        if (int rc = launch_status()) return rc;
    }
    if (int rc = launch_gemv_partials(reinterpret_cast<const uint16_t*>(xh_dn), 1, slots,
                                      dn_trellis, H / 16, num_experts * (D / 16), K, cb, dn_sub,
                                      dn_tile, w.g_dn, part_dn, w.plan_dn, s))
        return rc;
    {
        const int waves = slots * (D / 128);
        moe_finish_kernel<<<dim3((waves + 3) / 4), dim3(256), 0, s>>>(
            part_dn, w.plan_dn.n_partials(), (size_t)w.g_dn * 128, indices,
            reinterpret_cast<const half_t*>(dn_svh), reinterpret_cast<half_t*>(y), slots, D,
            num_experts);
        if (int rc = launch_status()) return rc;
    }
    if (!a.combine.scores) return EXL3_OK;
    return exl3_moe_combine(y, reinterpret_cast<const uint16_t*>(a.combine.scores), tokens, top_k, D,
                            reinterpret_cast<uint16_t*>(a.combine.out), s);
}

}  // namespace exl3

EXL3_EXPORT int exl3_moe_forward(const uint16_t* x, int tokens, const int32_t* indices, int top_k,
                                 const uint16_t* gu_trellis, const uint16_t* gu_suh,
                                 const uint16_t* gu_svh, const uint16_t* dn_trellis,
                                 const uint16_t* dn_suh, const uint16_t* dn_svh, int num_experts,
                                 int D, int H, int K, int cb, int activation, uint16_t* y,
                                 void* workspace, size_t workspace_bytes, int32_t* counters,
                                 size_t counters_len, void* stream) {
    using namespace exl3;
    return moe_slots({x, tokens, const_cast<int32_t*>(indices), top_k, gu_trellis, gu_suh, gu_svh, dn_trellis, dn_suh,
                      dn_svh, num_experts, D, H, K, cb, activation, y, workspace, workspace_bytes, counters,
                      counters_len, {}, {}},
                     as_stream(stream));
}

EXL3_EXPORT int exl3_moe_groups_rounded(int tokens, int top_k, int num_experts, int D, int H) {
    using namespace exl3;
    return tokens > 0 && top_k > 0 && num_experts > 0 && !exact_weights() &&
           moe_groups_apply(tokens, top_k, num_experts, D, H) && moe_exact_down(tokens, tokens * top_k, num_experts);
}

EXL3_EXPORT size_t exl3_moe_decode_counters(int tokens, int slots_per_token, int D, int H) {
    if (tokens < 1 || slots_per_token < 1 || D < 128 || H < 128) return 0;
    return (size_t)tokens * slots_per_token * ((size_t)4 * H + D / 128) + (size_t)tokens * (D / 128) + 2;
}

EXL3_EXPORT int exl3_moe_decode(const uint16_t* x, int tokens, const uint16_t* logits, const uint16_t* shared_logits,
                                int n_router, int top_k, int norm, const uint16_t* gu_trellis, const uint16_t* gu_suh,
                                const uint16_t* gu_svh, const uint16_t* dn_trellis, const uint16_t* dn_suh,
                                const uint16_t* dn_svh, int num_experts, int D, int H, int K, int cb, int activation,
                                int32_t* indices, uint16_t* scores, uint16_t* slot_rows, uint16_t* out,
                                void* workspace, size_t workspace_bytes, int32_t* counters, size_t counters_len,
                                void* stream) {
    using namespace exl3;
    if (!logits || !indices || !scores || !slot_rows || !out || !counters) return EXL3_E_NULL_POINTER;
    if (tokens < 1 || n_router < 1 || top_k < 1 || top_k > n_router || D < 128 || H < 128 || D % 128 || H % 128 ||
        n_router + (shared_logits != nullptr) > num_experts || (shared_logits && n_router != num_experts - 1))
        return EXL3_E_BAD_SHAPE;
    // whoever ranks, the router's kernel or the experts'
    if (n_router > kRouteMaxExperts || top_k > kRouteMaxTopK) return EXL3_E_UNSUPPORTED;
    if ((reinterpret_cast<uintptr_t>(slot_rows) & 15) || (reinterpret_cast<uintptr_t>(out) & 15)) return EXL3_E_BAD_SHAPE;
    const int kk = top_k + (shared_logits != nullptr);
    if (counters_len < exl3_moe_decode_counters(tokens, kk, D, H)) return EXL3_E_WORKSPACE;
    // the combination's counters lie in front of the status word
    const size_t own = (size_t)tokens * (D / 128);
    int32_t* const combine = counters + counters_len - 2 - own;
    const MoeRoute route{reinterpret_cast<const half_t*>(logits), reinterpret_cast<const half_t*>(shared_logits), n_router,
                         norm, reinterpret_cast<half_t*>(scores)};
    return moe_slots({x, tokens, indices, kk, gu_trellis, gu_suh, gu_svh, dn_trellis, dn_suh, dn_svh, num_experts, D, H, K,
                      cb, activation, slot_rows, workspace, workspace_bytes, counters, counters_len, route,
                      {reinterpret_cast<const half_t*>(scores), reinterpret_cast<half_t*>(out), combine, kk}},
                     as_stream(stream));
}

EXL3_EXPORT int exl3_moe_sort(const int32_t* indices, int n_pairs, int top_k, int n_experts,
                              int block_rows, int32_t* order, int32_t* tok, int32_t* sidx,
                              int32_t* table, int table_len, void* stream) {
    using namespace exl3;
    if (!indices || !order || !tok || !sidx || !table) return EXL3_E_NULL_POINTER;
    if (n_pairs < 1 || top_k < 1 || n_experts < 1 || block_rows < 1 ||
        table_len < n_pairs / block_rows + n_experts)
        return EXL3_E_BAD_SHAPE;
    if (n_experts > kSortMaxExperts) return EXL3_E_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(table) & 15) return EXL3_E_BAD_SHAPE;
    return launch_moe_sort({indices, n_pairs, top_k, n_experts, block_rows, order, tok, sidx,
                            reinterpret_cast<int4*>(table), table_len, 1, 0},
                           as_stream(stream));
}

namespace exl3 {

// Row blocks of the prefill kernels: 32 rows where an average expert's rows fit with room to
// spare (half the matrix work and registers), else 64, decoded again for every further 64.
static int moe_prefill_block_rows(long long pairs, int n_experts) { return pairs <= 24ll * n_experts ? 32 : 64; }

struct MoePrefillWorkspace {
    size_t o_tables, o_table, o_xg, o_xu, o_xd, total;
    int block_rows, table_len;
};

static MoePrefillWorkspace moe_prefill_workspace(long long pairs, int E, int D, int H) {
    MoePrefillWorkspace w{};
    w.block_rows = moe_prefill_block_rows(pairs, E);
    w.table_len = (int)(pairs / w.block_rows + E);
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t o = at;
        at += align_up(bytes, 256);
        return o;
    };
    w.o_tables = take((size_t)pairs * sizeof(int));  // order
    w.o_table = take((size_t)w.table_len * sizeof(int4));
    w.o_xg = take((size_t)pairs * D * 2);  // later the slots' outputs
    w.o_xu = take((size_t)pairs * D * 2);
    w.o_xd = take((size_t)pairs * H * 2);
    w.total = at;
    return w;
}

}  // namespace exl3

EXL3_EXPORT size_t exl3_moe_prefill_workspace_bytes(int tokens, int top_k, int n_experts, int D, int H) {
    if (tokens < 1 || top_k < 1 || n_experts < 1 || D < 128 || H < 128 || D % 128 || H % 128) return 0;
    return exl3::moe_prefill_workspace((long long)tokens * top_k, n_experts, D, H).total;
}

EXL3_EXPORT int exl3_moe_prefill(const uint16_t* x, int tokens, const int32_t* indices, int top_k,
                                 const uint16_t* gu_trellis, const uint16_t* gu_suh,
                                 const uint16_t* gu_svh, const uint16_t* dn_trellis,
                                 const uint16_t* dn_suh, const uint16_t* dn_svh, int num_experts,
                                 int D, int H, int K, int cb, int activation,
                                 const uint16_t* scores, uint16_t* y, void* workspace,
                                 size_t workspace_bytes, void* stream) {
    using namespace exl3;
    if (int rc = check_k_cb(K, cb)) return rc;
    if (!x || !indices || !gu_trellis || !gu_suh || !gu_svh || !dn_trellis || !dn_suh || !dn_svh || !y ||
        !workspace)
        return EXL3_E_NULL_POINTER;
    if (tokens < 1 || top_k < 1 || num_experts < 1 || D < 128 || H < 128 || D % 128 || H % 128 ||
        (long long)tokens * top_k > (1 << 28))
        return EXL3_E_BAD_SHAPE;
    if (activation != 0 && activation != 1) return EXL3_E_UNSUPPORTED;
    if (num_experts > kSortMaxExperts) return EXL3_E_UNSUPPORTED;
    const int N = tokens * top_k, E = num_experts;
    const MoePrefillWorkspace w = moe_prefill_workspace(N, E, D, H);
    if (workspace_bytes < w.total) return EXL3_E_WORKSPACE;
    for (const void* p : {(const void*)workspace, (const void*)y, (const void*)gu_svh, (const void*)dn_suh,
                          (const void*)dn_svh, (const void*)x, (const void*)gu_suh, (const void*)gu_trellis,
                          (const void*)dn_trellis})
        if (reinterpret_cast<uintptr_t>(p) & 15) return EXL3_E_BAD_SHAPE;
    char* base = static_cast<char*>(workspace);
    int* order = reinterpret_cast<int*>(base + w.o_tables);
    int* table = reinterpret_cast<int*>(base + w.o_table);
    uint16_t* xg = reinterpret_cast<uint16_t*>(base + w.o_xg);
    uint16_t* xd = reinterpret_cast<uint16_t*>(base + w.o_xd);
    const size_t xu_offset = (w.o_xu - w.o_xg) / 2;
    hipStream_t s = as_stream(stream);
    const SortArgs sort{indices, N, top_k, E, w.block_rows, order, nullptr, nullptr, reinterpret_cast<int4*>(table), w.table_len, 1, 0};
    // The rotated rows stay in the order of the pairs, which one launch then rotates and sorts, and gate/up gathers
    // them, at 32-bit offsets; beyond those they are put in sorted order, and the sort comes first.
    const bool gather = (unsigned long long)N * D * 2 <= 0xFFFFFFFFull;
    if (!gather)
        if (int rc = launch_moe_sort(sort, s)) return rc;
    if (int rc = launch_had_pre_pairs(x, tokens, top_k, D, gather ? nullptr : order, indices, gu_suh, E, xg, xu_offset,
                                      gather ? &sort : nullptr, s))
        return rc;
    // gate, up, GLU and rotation, then down with its output transform, back in pair order
    uint16_t* slots = scores ? xg : y;
    if (int rc = launch_moe_rows(xg, xg + xu_offset, N, gu_trellis, gu_svh, dn_trellis, dn_suh, dn_svh, E, D, H, K, cb,
                                 activation, table, w.table_len, w.block_rows, order, gather, xd, slots, s))
        return rc;
    return scores ? exl3_moe_combine(slots, scores, tokens, top_k, D, y, stream) : EXL3_OK;
}

EXL3_EXPORT int exl3_moe_glu_rows(const uint16_t* g, const uint16_t* u, int n_rows, int H,
                                  const int32_t* sidx, const uint16_t* gu_svh,
                                  const uint16_t* dn_suh, int n_experts, int activation,
                                  uint16_t* xh_dn, void* stream) {
    using namespace exl3;
    if (!g || !u || !sidx || !gu_svh || !dn_suh || !xh_dn) return EXL3_E_NULL_POINTER;
    if (n_rows < 0 || H < 128 || H % 128 || n_experts < 1) return EXL3_E_BAD_SHAPE;
    if (activation < 0 || activation > 1) return EXL3_E_UNSUPPORTED;
    if (n_rows == 0) return EXL3_OK;
    const long long waves = (long long)n_rows * (H / 128);
    const long long grid = (waves + 3) / 4;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    moe_glu_rows_kernel<<<dim3((unsigned)grid), dim3(256), 0, as_stream(stream)>>>(
        reinterpret_cast<const half_t*>(g), reinterpret_cast<const half_t*>(u), n_rows, H, sidx,
        reinterpret_cast<const half_t*>(gu_svh), reinterpret_cast<const half_t*>(dn_suh), n_experts,
        activation, reinterpret_cast<half_t*>(xh_dn));
    return launch_status();
}
