// Hadamard-128 regularisation kernels (input side with suh, output side with
// split-K reduction + svh + bias).
//
// Narrow form (few rows, fp32 partial sums): one wavefront owns one 128-wide
// block, lane l holds elements 2l and 2l+1 in fp32. The Sylvester transform
// factors into 7 butterfly stages that commute; the stage on element bit 0 is
// in-lane, the other six exchange with lane l ^ (1 << b).
// Wide form (prefill, fp16 in and out): lane l of a 16-lane group holds the 8
// consecutive elements 8l..8l+7 of a block (one 16-byte load), the stages on
// element bits 0..2 are in-lane and the other four exchange inside the group, so
// a wavefront transforms four blocks per 1 KiB load and a workgroup walks along
// one row. Same stage order and the same a+b / a-b per stage as the narrow form,
// hence the same bits. No LDS, no barriers. Arithmetic follows
// ponyexl3/ref/hadamard.py:50-80: multiply by the pre vector in fp32,
// transform, scale by 1/sqrt(128), multiply by the post vector in fp32, and the
// caller-visible casts of ponyexl3/ref/forward.py:34,41,42,45.
#include "exl3_device.hpp"
#include "exl3_host.hpp"
#include "exl3_rows.hpp"
#include "exl3_sort.hpp"

#pragma clang fp contract(off)

namespace exl3 {

constexpr float kHadScale = 0.088388347648318440550f;  // 1/sqrt(128)

__device__ __forceinline__ void wht128(float& a, float& b, int lane) { wht128_lanes(a, b, lane); }

// Optional row gathers / scatter of the wide kernels: kernel row r reads input row
// in_index[r], scale vector scale_index[r] (scale_ld elements apart) and writes
// output row out_index[r]; a NULL table is the identity. The tables come from the
// caller's memory: a row whose input, scale or output index falls outside
// [0, n_in) / [0, n_scale) / [0, n_out) is skipped (nothing is read or written for it).
struct RowMap {
    int per_row;
    const int32_t* in_index;
    const int32_t* scale_index;
    const int32_t* out_index;
    size_t scale_ld;
    unsigned n_in, n_scale, n_out;  // rows behind x, scale and out (per_row mode only)
    __device__ size_t in_row(size_t r) const { return in_index ? (size_t)in_index[r] : r; }
    __device__ size_t scale_row(size_t r) const { return scale_index ? (size_t)scale_index[r] : r; }
    __device__ size_t out_row(size_t r) const { return out_index ? (size_t)out_index[r] : r; }
    __device__ bool row_ok(size_t r, bool uses_scale) const {
        if (!per_row) return true;
        // negative entries wrap to huge unsigned values and fail the same test
        return in_row(r) < (size_t)n_in && out_row(r) < (size_t)n_out &&
               (!uses_scale || scale_row(r) < (size_t)n_scale);
    }
};

// Wide forms: grid.x = number of output rows ((row, sub) pairs for the input side);
// the four waves of a workgroup take consecutive 512-element chunks of the row,
// and grid.y workgroups share a row when there are too few rows to fill the chip.
// All pointers 16-byte aligned, n a multiple of 128.
__global__ __launch_bounds__(256) void had_pre_wide_kernel(const half_t* __restrict__ x,
                                                           const half_t* __restrict__ suh,
                                                           half_t* __restrict__ xh, int n,
                                                           int n_sub, RowMap map) {
    const int lane = threadIdx.x & 63;
    // One workgroup per source row: per-row tables (rows sorted by expert) give its
    // source, scale vector and destination; otherwise the row is rotated once per stacked
    // sibling (scale vector s, destination row r * n_sub + s) from a single read.
    const size_t r = blockIdx.x;
    if (!map.row_ok(r, suh != nullptr)) return;
    const half_t* xr = x + (map.per_row ? map.in_row(r) : r) * (size_t)n;
    const int subs = map.per_row ? 1 : n_sub;
    // up to four 16-byte chunks of the row in flight per lane
    const int c0 = (blockIdx.y * 256 + threadIdx.x) * 8, cstep = 2048 * gridDim.y;
    for (int cb = c0; cb < n; cb += 4 * cstep) {
        uint4_t raw[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (cb + i * cstep < n) raw[i] = *reinterpret_cast<const uint4_t*>(xr + cb + i * cstep);
        for (int s = 0; s < subs; s++) {
            const half_t* sr =
                suh ? suh + (map.per_row ? map.scale_row(r) * map.scale_ld : s * (size_t)n) : nullptr;
            half_t* orow = xh + (map.per_row ? map.out_row(r) : r * n_sub + s) * (size_t)n;
            uint4_t sraw[4];
            if (sr) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (cb + i * cstep < n)
                        sraw[i] = *reinterpret_cast<const uint4_t*>(sr + cb + i * cstep);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int c = cb + i * cstep;
                if (c >= n) break;
                float v[8], sv[8];
                halfs_to_floats(raw[i], v);
                if (sr) {
                    halfs_to_floats(sraw[i], sv);
#pragma unroll
                    for (int j = 0; j < 8; j++) v[j] = v[j] * sv[j];
                }
                wht128_wide(v, lane);
                uint4_t o;
                uint32_t* ow = reinterpret_cast<uint32_t*>(&o);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    half2_t h;
                    h.x = (half_t)(v[2 * k] * kHadScale);
                    h.y = (half_t)(v[2 * k + 1] * kHadScale);
                    ow[k] = half2_to_bits(h);
                }
                *reinterpret_cast<uint4_t*>(orow + c) = o;
            }
        }
    }
}

// Input side on the matrix pipe: a wave rotates 16 rows x one 128-wide block, for
// subs_per_wave of the stacked siblings from one read of x. Plain signs (packed sign words, the
// usual case) are applied to the fp16 bits of x and the block is contracted with entries +-1,
// fp32 sums (the fp32 butterfly's result up to the order of the additions): 32 matrix
// instructions of 16 cycles and 2 VALU instructions per element replace about 18, which the
// butterfly form is bound by. With any other scale value among the wave's rows the products
// need fp32: the butterfly then runs in this kernel, with the bits of the kernels above.
// Row maps (MoE): row r is pair p = pair[r] (r without pair) of token p / top_k and expert pair_expert[p], whose scales are scale_ld halfs from the next expert's; entries
// outside the buffers are clamped.
// Results: out + s * sub_stride + r * row_stride.
//
// What bounds the large ones is the way of the results to memory. From the matrix pipe's layout the
// sixteen lanes of a quarter wave touch sixteen rows, 16 bytes each, and what the L2 holds at the end is written
// back then. STREAM turns the tile in LDS, rows and results alike, so that loads and stores cover four
// rows of 256 bytes in lane order, and stores past the L2. 13 833 pairs of 2048 (113 MB) 38.8 -> 31.6 us (35.8
// with the stores alone turned, 33.6 without the hint), 333 rows of 17408 7.4 -> 5.8. Same bits. Small results are better read back from the L2: see launch_rotate().
struct RotateArgs {
    const half_t* x;
    const half_t* suh;
    half_t* out;
    int rows, n, n_sub, subs_per_wave;
    size_t sub_scale, sub_stride, row_stride;  // halfs from one sibling's scales / results to the next
    const int32_t* pair;
    const int32_t* pair_expert;
    int top_k, n_tokens, n_experts;
    size_t scale_ld;
};

constexpr int kRotateLd = 128 + 8;  // halfs: rows four LDS banks apart

// The LDS tile belongs to one wave: order for the compiler, the hardware keeps it.
__device__ __forceinline__ void rotate_tile_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Four waves from wave 4 `block` on; `tiles`: LDS, 16 x kRotateLd halfs to a wave (STREAM).
template <bool STREAM>
__device__ __forceinline__ void rotate_waves(const RotateArgs& a, unsigned block, half_t* tiles) {
    half_t* const tile = STREAM ? tiles + (threadIdx.x >> 6) * (16 * kRotateLd) : nullptr;
    const int lane = threadIdx.x & 63;
    const int fr = lane & 15, q = lane >> 4;
    const int blocks = a.n >> 7;
    const long long wid = (long long)block * 4 + (threadIdx.x >> 6);
    const int row_tiles = (a.rows + 15) >> 4;
    if (wid >= (long long)row_tiles * blocks) return;
    // consecutive waves take consecutive blocks of the same rows
    const int blk = (int)(wid % blocks), r0 = (int)(wid / blocks) * 16, r = r0 + fr;
    const bool valid = r < a.rows;
    int src = valid ? r : 0, scale_row = 0;
    if (a.pair_expert) {
        const int p = a.pair ? min(max(a.pair[src], 0), a.n_tokens * a.top_k - 1) : src;
        scale_row = min(max(a.pair_expert[p], 0), a.n_experts - 1);
        src = p / a.top_k;
    }
    const size_t col = (size_t)blk * 128 + q * 8;
    uint4_t xv[4];
    if constexpr (STREAM) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t row = (size_t)__shfl(src, 4 * i + q, kWave);
            xv[i] = *reinterpret_cast<const uint4_t*>(a.x + row * a.n + (size_t)blk * 128 + fr * 8);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) *reinterpret_cast<uint4_t*>(tile + (4 * i + q) * kRotateLd + fr * 8) = xv[i];
        rotate_tile_order();
#pragma unroll
        for (int k = 0; k < 4; k++) xv[k] = *reinterpret_cast<const uint4_t*>(tile + fr * kRotateLd + k * 32 + q * 8);
        rotate_tile_order();
    } else {
        const half_t* xr = a.x + (size_t)src * a.n + col;
#pragma unroll
        for (int k = 0; k < 4; k++) xv[k] = *reinterpret_cast<const uint4_t*>(xr + k * 32);
    }
    const HadamardColumns had(lane);
    const int s_begin = blockIdx.y * a.subs_per_wave, s_end = min(s_begin + a.subs_per_wave, a.n_sub);
    for (int s = s_begin; s < s_end; s++) {
        float4_t z[8];
#pragma unroll
        for (int nt = 0; nt < 8; nt++) z[nt] = float4_t{0.f, 0.f, 0.f, 0.f};
        uint4_t sv[4];
        if (a.suh) {
            const half_t* sr = a.suh + (size_t)scale_row * a.scale_ld + (size_t)s * a.sub_scale + col;
#pragma unroll
            for (int k = 0; k < 4; k++) sv[k] = *reinterpret_cast<const uint4_t*>(sr + k * 32);
        }
        if (!a.suh || all_plain_signs(sv)) {
            static_for<0, 4>([&](auto k) {
                const uint4_t flip = a.suh ? sv[k.value] & 0x80008000u : uint4_t{0u, 0u, 0u, 0u};
                const half8_t v = __builtin_bit_cast(half8_t, xv[k.value] ^ flip);
                static_for<0, 8>([&](auto nt) {
                    z[nt.value] = __builtin_amdgcn_mfma_f32_16x16x32_f16(had.template get<nt.value, k.value>(), v,
                                                                         z[nt.value], 0, 0, 0);
                });
            });
        } else {
            float v[4][8];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                float scale[8];
                halfs_to_floats(xv[k], v[k]);
                halfs_to_floats(sv[k], scale);
#pragma unroll
                for (int t = 0; t < 8; t++) v[k][t] = v[k][t] * scale[t];
            }
            wht128_tile(v);
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int t = 0; t < 8; t++) z[2 * k + (t >> 2)][t & 3] = v[k][t];
        }
        half_t* const o = a.out + (size_t)s * a.sub_stride;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            half8_t v;
#pragma unroll
            for (int c = 0; c < 8; c++) v[c] = (half_t)(z[2 * p + (c >> 2)][c & 3] * kHadScale);
            if constexpr (STREAM) *reinterpret_cast<half8_t*>(tile + fr * kRotateLd + p * 32 + q * 8) = v;
            else if (valid) *reinterpret_cast<half8_t*>(o + (size_t)r * a.row_stride + col + p * 32) = v;
        }
        if constexpr (STREAM) {
            rotate_tile_order();
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int ro = r0 + 4 * i + q;
                const uint4_t v = *reinterpret_cast<const uint4_t*>(tile + (4 * i + q) * kRotateLd + fr * 8);
                if (ro < a.rows)
                    __builtin_nontemporal_store(
                        v, reinterpret_cast<uint4_t*>(o + (size_t)ro * a.row_stride + (size_t)blk * 128 + fr * 8));
            }
            rotate_tile_order();
        }
    }
}

constexpr size_t kRotateTileBytes = (size_t)4 * 16 * kRotateLd * sizeof(half_t);

template <bool STREAM>
__global__ __launch_bounds__(256, 4) void had_pre_mfma_kernel(RotateArgs a) {
    __shared__ __attribute__((aligned(16))) half_t tiles[STREAM ? kRotateTileBytes / sizeof(half_t) : 8];
    rotate_waves<STREAM>(a, blockIdx.x, tiles);
}

// Rotation of pairs in their own order and, by the first workgroups, their sort, which nothing in the rotation
// needs: as a launch in front it takes 5 us up to 2000 pairs and 10 us at 13 833, here no more than the
// rotation does. Whole prefill call with the sort in front and the rows in sorted order -> this way: 97 tokens, 194 pairs
// 63.5 -> 58.5 us, 400 tokens, 2000 pairs 65.2 -> 60.5, 1537 tokens 289 -> 278; 58 shapes of 45 to 2048 tokens 4.5 %.
constexpr int kRotateThreads = 256;
template <bool STREAM>
__global__ __launch_bounds__(kRotateThreads, 4) void moe_sort_rotate_kernel(RotateArgs a, SortArgs sort) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    if (blockIdx.x >= (unsigned)sort.groups) rotate_waves<STREAM>(a, blockIdx.x - sort.groups, reinterpret_cast<half_t*>(lds));
    else if (blockIdx.y == 0) sort_pairs<kRotateThreads>(sort, blockIdx.x, reinterpret_cast<int*>(lds));
}

static int launch_rotate(RotateArgs a, const SortArgs* sort, hipStream_t stream) {
    const long long waves = (long long)((a.rows + 15) / 16) * (a.n / 128);
    // few rows: the siblings in parallel; else one read of x for all of them
    a.subs_per_wave = waves * a.n_sub <= 4096 ? 1 : a.n_sub;
    const long long grid = (waves + 3) / 4, gy = (a.n_sub + a.subs_per_wave - 1) / a.subs_per_wave;
    if (grid + (sort ? kSortMaxGroups : 0) > 0x7FFFFFFFLL || gy > 65535) return EXL3_E_BAD_SHAPE;
    // Past the L2 from 8 MB of results on: whole layers of 77 rows x 3 x 5120 (2.4 MB) and 754 x 2304 (3.5 MB) are 0.5 %
    // slower that way, 333 x 17408 (11.6 MB) 1 % faster, the experts of 1537 tokens (113 MB) 0.6 to 1.7 %. Not
    // for more rows than the rows kernels take: the GEMM, which the matrix pipe's clock bounds, gives the time
    // back (2048 x 5120 -> 34816 0.2 % slower).
    const bool stream_results = (a.pair_expert || a.rows <= kLinearRowsMaxRows) &&
                                (size_t)a.rows * a.n * a.n_sub * sizeof(half_t) >= (size_t)8 << 20;
    if (!sort) {
        auto kernel = stream_results ? had_pre_mfma_kernel<true> : had_pre_mfma_kernel<false>;
        kernel<<<dim3((unsigned)grid, (unsigned)gy), dim3(256), 0, stream>>>(a);
        return launch_status();
    }
    SortArgs so = *sort;
    // a workgroup per 1024 pairs, up to kSortMaxGroups; in place of one alone for 2000 pairs two, where the
    // rotation is as short as the sort: 400 tokens 62.3 -> 60.4 us, 273 tokens 59.1 -> 57.5
    so.groups = std::min(kSortMaxGroups, (so.n_pairs + 1023) / 1024);
    so.staged = so.groups == 1;
    const size_t need = sort_lds_ints(kRotateThreads, so) * sizeof(int);
    const size_t lds = stream_results ? std::max(need, kRotateTileBytes) : need;
    auto kernel = stream_results ? moe_sort_rotate_kernel<true> : moe_sort_rotate_kernel<false>;
    kernel<<<dim3((unsigned)(grid + so.groups), (unsigned)gy), dim3(kRotateThreads), lds, stream>>>(a, so);
    return launch_status();
}

__global__ __launch_bounds__(256) void had_post_wide_kernel(const half_t* __restrict__ y,
                                                            const half_t* __restrict__ svh,
                                                            const half_t* __restrict__ bias,
                                                            half_t* out, int n, RowMap map) {
    const int lane = threadIdx.x & 63;
    const size_t rs = blockIdx.x;
    if (!map.row_ok(rs, svh != nullptr)) return;
    if (svh && map.per_row) svh += map.scale_row(rs) * map.scale_ld;
    const half_t* yr = y + map.in_row(rs) * (size_t)n;
    half_t* orow = out + map.out_row(rs) * (size_t)n;
    // up to four 16-byte chunks of the row in flight per lane
    const int c0 = (blockIdx.y * 256 + threadIdx.x) * 8, cstep = 2048 * gridDim.y;
    for (int cb = c0; cb < n; cb += 4 * cstep) {
        uint4_t raw[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (cb + i * cstep < n) raw[i] = *reinterpret_cast<const uint4_t*>(yr + cb + i * cstep);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int c = cb + i * cstep;
            if (c >= n) break;
            float v[8], sv[8];
            halfs_to_floats(raw[i], v);
            wht128_wide(v, lane);
            if (svh) halfs_to_floats(*reinterpret_cast<const uint4_t*>(svh + c), sv);
            uint4_t bq = {0u, 0u, 0u, 0u};
            if (bias) bq = *reinterpret_cast<const uint4_t*>(bias + c);
            const uint32_t* bw = reinterpret_cast<const uint32_t*>(&bq);
            uint4_t o;
            uint32_t* ow = reinterpret_cast<uint32_t*>(&o);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                float a = v[2 * k] * kHadScale, b = v[2 * k + 1] * kHadScale;
                if (svh) {
                    a = a * sv[2 * k];
                    b = b * sv[2 * k + 1];
                }
                half2_t h;
                h.x = (half_t)a;
                h.y = (half_t)b;
                if (bias) {
                    const half2_t bv = bits_to_half2(bw[k]);
                    h.x = h.x + bv.x;
                    h.y = h.y + bv.y;
                }
                ow[k] = half2_to_bits(h);
            }
            *reinterpret_cast<uint4_t*>(orow + c) = o;
        }
    }
}

// xh[r][s][blk] = fp16(wht(x[r][blk] * suh[s][blk]) / sqrt(128))
__global__ __launch_bounds__(256) void had_pre_kernel(const half_t* __restrict__ x,
                                                      const half_t* __restrict__ suh,
                                                      half_t* __restrict__ xh, int rows, int n,
                                                      int n_sub) {
    const int lane = threadIdx.x & 63;
    const int blocks = n >> 7;
    const long long wave_id = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const long long total = (long long)rows * n_sub * blocks;
    if (wave_id >= total) return;
    const int blk = (int)(wave_id % blocks);
    const long long rs = wave_id / blocks;
    const int s = (int)(rs % n_sub);
    const long long r = rs / n_sub;
    const half2_t xv = *reinterpret_cast<const half2_t*>(x + r * n + blk * 128 + 2 * lane);
    float a = (float)xv.x, b = (float)xv.y;
    if (suh) {
        const half2_t sv =
            *reinterpret_cast<const half2_t*>(suh + (size_t)s * n + blk * 128 + 2 * lane);
        a = a * (float)sv.x;
        b = b * (float)sv.y;
    }
    wht128(a, b, lane);
    half2_t o;
    o.x = (half_t)(a * kHadScale);
    o.y = (half_t)(b * kHadScale);
    *reinterpret_cast<half2_t*>(xh + rs * n + blk * 128 + 2 * lane) = o;
}

// out[r][blk] = fp16(wht(fp16(sum_i y[i][r][blk])) / sqrt(128) * svh[blk]) (+ bias)
template <bool kFp32In>
__global__ __launch_bounds__(256) void had_post_kernel(const void* __restrict__ yv, int n_sum,
                                                       size_t sum_stride,
                                                       const half_t* __restrict__ svh,
                                                       const half_t* __restrict__ bias,
                                                       half_t* out, int rows, int n) {
    const int lane = threadIdx.x & 63;
    const int blocks = n >> 7;
    const long long wave_id = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wave_id >= (long long)rows * blocks) return;
    const int blk = (int)(wave_id % blocks);
    const long long r = wave_id / blocks;
    const size_t off = (size_t)r * n + blk * 128 + 2 * lane;
    float a, b;
    if constexpr (kFp32In) {
        const float* y = reinterpret_cast<const float*>(yv);
        // slices are loaded eight at a time and added strictly in index order
        float2_t acc = {0.f, 0.f};
        int i = 0;
        for (; i + 8 <= n_sum; i += 8) {
            float2_t v[8];
#pragma unroll
            for (int j = 0; j < 8; j++)
                v[j] = *reinterpret_cast<const float2_t*>(y + (size_t)(i + j) * sum_stride + off);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                acc.x = acc.x + v[j].x;
                acc.y = acc.y + v[j].y;
            }
        }
        for (; i < n_sum; i++) {
            const float2_t v = *reinterpret_cast<const float2_t*>(y + (size_t)i * sum_stride + off);
            acc.x = acc.x + v.x;
            acc.y = acc.y + v.y;
        }
        a = (float)(half_t)acc.x;  // the matmul result is stored as fp16 before the transform
        b = (float)(half_t)acc.y;
    } else {
        const half2_t v = *reinterpret_cast<const half2_t*>(reinterpret_cast<const half_t*>(yv) + off);
        a = (float)v.x;
        b = (float)v.y;
    }
    wht128(a, b, lane);
    a = a * kHadScale;
    b = b * kHadScale;
    if (svh) {
        const half2_t sv = *reinterpret_cast<const half2_t*>(svh + blk * 128 + 2 * lane);
        a = a * (float)sv.x;
        b = b * (float)sv.y;
    }
    half2_t o;
    o.x = (half_t)a;
    o.y = (half_t)b;
    if (bias) {
        const half2_t bv = *reinterpret_cast<const half2_t*>(bias + blk * 128 + 2 * lane);
        o.x = o.x + bv.x;
        o.y = o.y + bv.y;
    }
    *reinterpret_cast<half2_t*>(out + off) = o;
}

// From this many rows on the wide kernels (one workgroup per row) fill the device
// better than one wave per 128-element block.
constexpr int kWideMinRows = 16;
static inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Workgroups per row of the wide kernels: about four workgroups per CU in total,
// never more than the row has 2048-element chunks.
static unsigned wide_row_parts(long long rows, int n) {
    const long long chunks = (n + 2047) / 2048;
    long long want = (1024 + rows - 1) / rows;
    if (want > chunks) want = chunks;
    return (unsigned)(want < 1 ? 1 : want);
}

int launch_had_pre(const uint16_t* x, int rows, int n, const uint16_t* suh, int n_sub,
                   uint16_t* xh, hipStream_t stream) {
    if (!x || !xh) return EXL3_E_NULL_POINTER;
    if (rows < 0 || n <= 0 || n % 128 || n_sub < 1) return EXL3_E_BAD_SHAPE;
    if (!suh && n_sub != 1) return EXL3_E_BAD_SHAPE;
    if (rows == 0) return EXL3_OK;
    const long long waves = (long long)rows * n_sub * (n / 128);
    const long long grid = (waves + 3) / 4;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    if ((long long)rows * n_sub >= kWideMinRows && aligned16(x) && aligned16(xh) &&
        (!suh || aligned16(suh))) {
        had_pre_wide_kernel<<<dim3((unsigned)rows, wide_row_parts((long long)rows, n)),
                              dim3(256), 0, stream>>>(
            reinterpret_cast<const half_t*>(x), reinterpret_cast<const half_t*>(suh),
            reinterpret_cast<half_t*>(xh), n, n_sub, RowMap{});
        return launch_status();
    }
    had_pre_kernel<<<dim3((unsigned)grid), dim3(256), 0, stream>>>(
        reinterpret_cast<const half_t*>(x), reinterpret_cast<const half_t*>(suh),
        reinterpret_cast<half_t*>(xh), rows, n, n_sub);
    return launch_status();
}

int launch_had_post(const void* y, int y_is_fp32, int n_sum, size_t sum_stride, int rows, int n,
                    const uint16_t* svh, const uint16_t* bias, uint16_t* out, hipStream_t stream) {
    if (!y || !out) return EXL3_E_NULL_POINTER;
    if (rows < 0 || n <= 0 || n % 128 || n_sum < 1) return EXL3_E_BAD_SHAPE;
    if (!y_is_fp32 && n_sum != 1) return EXL3_E_BAD_SHAPE;
    if (rows == 0) return EXL3_OK;
    const long long waves = (long long)rows * (n / 128);
    const long long grid = (waves + 3) / 4;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    const half_t* s = reinterpret_cast<const half_t*>(svh);
    const half_t* b = reinterpret_cast<const half_t*>(bias);
    half_t* o = reinterpret_cast<half_t*>(out);
    if (!y_is_fp32 && rows >= kWideMinRows && aligned16(y) && aligned16(out) &&
        (!svh || aligned16(svh)) && (!bias || aligned16(bias))) {
        had_post_wide_kernel<<<dim3((unsigned)rows, wide_row_parts(rows, n)), dim3(256), 0, stream>>>(
            reinterpret_cast<const half_t*>(y), s, b, o, n, RowMap{});
        return launch_status();
    }
    if (y_is_fp32)
        had_post_kernel<true><<<dim3((unsigned)grid), dim3(256), 0, stream>>>(y, n_sum, sum_stride,
                                                                              s, b, o, rows, n);
    else
        had_post_kernel<false><<<dim3((unsigned)grid), dim3(256), 0, stream>>>(y, 1, 0, s, b, o,
                                                                               rows, n);
    return launch_status();
}

// Per-row scale vectors (rows that belong to different experts): wide kernels only.
int launch_had_rows(const uint16_t* x, int n_in_rows, int rows, int n, const int32_t* in_index,
                    const uint16_t* scale, int n_scale_rows, const int32_t* scale_index,
                    size_t scale_ld, int post, uint16_t* out, int n_out_rows,
                    const int32_t* out_index, hipStream_t stream) {
    if (!x || !out || !scale) return EXL3_E_NULL_POINTER;
    if (rows < 0 || n <= 0 || n % 128 || scale_ld % 8 || n_in_rows < 0 || n_scale_rows < 0 ||
        n_out_rows < 0)
        return EXL3_E_BAD_SHAPE;
    // identity maps must stay inside their buffers as well
    if ((!in_index && rows > n_in_rows) || (!scale_index && rows > n_scale_rows) ||
        (!out_index && rows > n_out_rows))
        return EXL3_E_BAD_SHAPE;
    if (!aligned16(x) || !aligned16(out) || !aligned16(scale)) return EXL3_E_BAD_SHAPE;
    if (rows == 0) return EXL3_OK;
    const RowMap map{1, in_index, scale_index, out_index, scale_ld, (unsigned)n_in_rows,
                     (unsigned)n_scale_rows, (unsigned)n_out_rows};
    if (post)
        had_post_wide_kernel<<<dim3((unsigned)rows, wide_row_parts(rows, n)), dim3(256), 0, stream>>>(
            reinterpret_cast<const half_t*>(x), reinterpret_cast<const half_t*>(scale), nullptr,
            reinterpret_cast<half_t*>(out), n, map);
    else
        had_pre_wide_kernel<<<dim3((unsigned)rows, wide_row_parts(rows, n)), dim3(256), 0, stream>>>(
            reinterpret_cast<const half_t*>(x), reinterpret_cast<const half_t*>(scale),
            reinterpret_cast<half_t*>(out), n, 1, map);
    return launch_status();
}

// The rotation as the layer forwards use it: on the matrix pipe from 64 rows on (16 rows for two
// siblings of 5120: 4.1 us in the butterfly kernel, 5.0 here; 77 rows for three: 5.8 and 5.4;
// 2048 rows: 23.0 and 18.6).
int launch_rotate_layer(const uint16_t* x, int rows, int n, const uint16_t* suh, int n_sub, uint16_t* xh,
                        hipStream_t stream) {
    if (rows < 64 || n < 128 || n % 128 || n_sub < 1 || (!suh && n_sub != 1) || !x || !xh || !aligned16(x) ||
        !aligned16(xh) || (suh && !aligned16(suh)))
        return launch_had_pre(x, rows, n, suh, n_sub, xh, stream);
    RotateArgs a{};
    a.x = reinterpret_cast<const half_t*>(x);
    a.suh = reinterpret_cast<const half_t*>(suh);
    a.out = reinterpret_cast<half_t*>(xh);
    a.rows = rows;
    a.n = n;
    a.n_sub = n_sub;
    a.sub_scale = a.sub_stride = (size_t)n;
    a.row_stride = (size_t)n_sub * n;
    return launch_rotate(a, nullptr, stream);
}

// Rows sorted by expert: both rotations (gate and up signs of the row's expert, gu_suh
// [E][2][n]) of row r = pair order[r], to xg[r] and, sub_stride halfs further, xu[r].
int launch_had_pre_pairs(const uint16_t* x, int tokens, int top_k, int n, const int32_t* order,
                         const int32_t* indices, const uint16_t* gu_suh, int n_experts, uint16_t* xg,
                         size_t sub_stride, const SortArgs* sort, hipStream_t stream) {
    if (!aligned16(x) || !aligned16(gu_suh) || !aligned16(xg) || sub_stride % 8) return EXL3_E_BAD_SHAPE;
    RotateArgs a{};
    a.x = reinterpret_cast<const half_t*>(x);
    a.suh = reinterpret_cast<const half_t*>(gu_suh);
    a.out = reinterpret_cast<half_t*>(xg);
    a.rows = tokens * top_k;
    a.n = n;
    a.n_sub = 2;
    a.sub_scale = (size_t)n;
    a.sub_stride = sub_stride;
    a.row_stride = (size_t)n;
    a.pair = order;
    a.pair_expert = indices;
    a.top_k = top_k;
    a.n_tokens = tokens;
    a.n_experts = n_experts;
    a.scale_ld = (size_t)2 * n;
    return launch_rotate(a, sort, stream);
}

}  // namespace exl3

EXL3_EXPORT int exl3_had128_rows(const uint16_t* x, int n_in_rows, int rows, int n,
                                 const int32_t* in_index, const uint16_t* scale, int n_scale_rows,
                                 const int32_t* scale_index, size_t scale_ld, int post,
                                 uint16_t* out, int n_out_rows, const int32_t* out_index,
                                 void* stream) {
    return exl3::launch_had_rows(x, n_in_rows, rows, n, in_index, scale, n_scale_rows, scale_index,
                                 scale_ld, post, out, n_out_rows, out_index,
                                 exl3::as_stream(stream));
}

EXL3_EXPORT int exl3_had128_pre(const uint16_t* x, int rows, int n, const uint16_t* suh, int n_sub,
                                uint16_t* xh, void* stream) {
    return exl3::launch_had_pre(x, rows, n, suh, n_sub, xh, exl3::as_stream(stream));
}

EXL3_EXPORT int exl3_rotate(const uint16_t* x, int rows, int n, const uint16_t* suh, int n_sub, uint16_t* xh,
                            void* stream) {
    return exl3::launch_rotate_layer(x, rows, n, suh, n_sub, xh, exl3::as_stream(stream));
}

EXL3_EXPORT int exl3_had128_post(const void* y, int y_is_fp32, int n_sum, size_t sum_stride,
                                 int rows, int n, const uint16_t* svh, const uint16_t* bias,
                                 uint16_t* out, void* stream) {
    return exl3::launch_had_post(y, y_is_fp32, n_sum, sum_stride, rows, n, svh, bias, out,
                                 exl3::as_stream(stream));
}
