// Whole layer in one launch for 2..16 rows of a layer that does not fill the chip (linear_batch_applies):
// input Hadamard, decode, products, split reduction, output Hadamard, svh and bias.
//
// The frame is that of linear_small_kernel: a wave rotates the activations it needs itself, streams
// packed words straight into registers and decodes every weight once. Such a launch is bound by the
// chain of steps that one wave goes through, not by the rate of any unit, so the chain is cut:
//
//   * a wave takes half a Hadamard block (four tile rows), all of whose loads are issued at the start;
//   * the rows of the batch are rotated side by side: up to 8 rows a lane holds 2 R elements of one
//     row, so that the fp32 butterfly costs about 18 VALU instructions per row instead of 41 with
//     two elements per lane and short chains; up to 16 rows the matrix pipe does it, and only the wave's half;
//   * products with a block-diagonal A operand (see x_operand_row in exl3_small.hpp): one matrix
//     instruction serves 4 batch rows (16x16x32) or 16 (32x32x16);
//   * the reduction is spread over the waves: wave w owns batch rows w, w + NW, ...
//
// Up to eight rows the products take the unsummed halves of the weights, as linear_small_kernel does;
// above, the weights are rounded to fp16 first, as in the kernels for more rows. Measured, us, against
// linear_small_kernel (rotation kernel and linear_mid_kernel from 9 rows on), K = 4, cold weights:
// 1664 -> 2560 at 4 / 8 / 16 rows 9.6 / 14.8 / 11.2 -> 5.7 / 7.6 / 9.1; 2560 -> 4096 9.5 / 14.7 / 12.5 -> 6.8 / 8.9 / 9.4.
#include "exl3_device.hpp"
#include "exl3_host.hpp"
#include "exl3_rows.hpp"
#include "exl3_small.hpp"

#include <type_traits>

#pragma clang fp contract(off)

namespace exl3 {

// R: batch rows that the kernel stages (4, 8 or 16); up to 8 take unsummed halves where the codebook has them.
template <int R, int CB>
struct BatchTile {
    static constexpr bool EXACT = R > 8 || !kHasHalves<CB>;
    // Up to 8 rows v_mfma_f32_16x16x32_f16, four rows each; above v_mfma_f32_32x32x16_f16, whose 32
    // A rows serve 16 rows in both lane halves.
    static constexpr bool WIDE = R > 8;
    static constexpr int NQ = WIDE ? 1 : R / 4;
    typedef float vec_t __attribute__((ext_vector_type(WIDE ? 16 : 4)));
    struct acc_t {  // batch row m of a column
        vec_t v[NQ];
        __device__ __forceinline__ float row(int m) const { return WIDE ? v[0][m] : v[m >> 2][m & 3]; }
    };
    // halfs per staged row: the 64 values of a half block (unsummed: each twice) and 16 bytes, so that
    // consecutive rows start four LDS banks apart
    static constexpr int LD = (EXACT ? 64 : 128) + 8;
    // Where lane `lane` reads its share of A: k-slots of group (lane >> 4 or >> 5) in A row i hold the
    // batch row whose sums land in that group's lanes, zeros (row R) elsewhere.
    static __device__ __forceinline__ int operand_row(int lane, int part) {
        if constexpr (!WIDE) {
            const int i = lane & 15, m = 4 * part + (i & 3);
            return (i >> 2) == (lane >> 4) ? m : R;
        } else {
            const int i = lane & 31, m = (i & 3) + 4 * (i >> 3);
            return ((i >> 2) & 1) == (lane >> 5) ? m : R;
        }
    }
    static __device__ __forceinline__ void mfma(const uint4_t (&a)[NQ], uint4_t b, acc_t& c) {
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            if constexpr (!WIDE)
                c.v[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a[i]),
                                                                __builtin_bit_cast(half8_t, b), c.v[i], 0, 0, 0);
            else
                c.v[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a[i]),
                                                                __builtin_bit_cast(half8_t, b), c.v[i], 0, 0, 0);
        }
    }
};

// 16 bytes of fp16 data at any (2-byte aligned) address: views of a larger tensor may start anywhere.
typedef uint4_t any_uint4_t __attribute__((aligned(2)));

// Products of a wave's half block: tile rows tk .. tk + 3 (tk a multiple of 4) of the 8 tile columns at
// `base`, against the rotated block's 64 values of its half.
template <int K, int CB, int R>
__device__ __forceinline__ void batch_main(const uint32_t* __restrict__ base, size_t row_words, int tk,
                                           const half_t* __restrict__ x, int in_features, int rows,
                                           const half_t* __restrict__ suh, half_t* xw, int lane,
                                           typename BatchTile<R, CB>::acc_t (&acc)[2]) {
    using T = BatchTile<R, CB>;
    constexpr bool EXACT = T::EXACT;
    const int blk = (tk >> 3) * 128, upper = (tk >> 2) & 1;
    constexpr int kSlots = kStreamSlots;
    uint32_t buf[kSlots][K];
    // the row of zeros
    auto stage_zeros = [&]() {
        if (lane < T::LD / 8) *reinterpret_cast<uint4_t*>(xw + R * T::LD + 8 * lane) = uint4_t{0u, 0u, 0u, 0u};
    };
    // eight rotated values, columns c .. c + 7 of the half, of batch row m
    auto stage8 = [&](int m, int c, const float* z) {
        half8_t o;
#pragma unroll
        for (int i = 0; i < 8; i++) o[i] = (half_t)__fmul_rn(z[i], kHadScaleF);
        if constexpr (EXACT) {
            *reinterpret_cast<half8_t*>(xw + m * T::LD + c) = o;
        } else {
            *reinterpret_cast<half8_t*>(xw + m * T::LD + 2 * c) = __builtin_shufflevector(o, o, 0, 0, 1, 1, 2, 2, 3, 3);
            *reinterpret_cast<half8_t*>(xw + m * T::LD + 2 * c + 8) = __builtin_shufflevector(o, o, 4, 4, 5, 5, 6, 6, 7, 7);
        }
    };
    // xw rows = this half of fp16(had128(x * suh) / sqrt(128))   (ponyexl3/ref/forward.py:32-34).
    // Activations are requested first: loads return in issue order (see stream_block_rows_at).
    if constexpr (R <= 8) {
        // lane = (row fr, elements E q .. E q + E - 1)
        constexpr int E = 2 * R;
        const int fr = lane & (R - 1), q = lane / R;
        uint4_t xq[E / 8], sq[E / 8];
        const half_t* xr = x + (size_t)min(fr, rows - 1) * in_features + blk + q * E;  // rows past the batch: never used
#pragma unroll
        for (int k = 0; k < E / 8; k++) xq[k] = *reinterpret_cast<const any_uint4_t*>(xr + k * 8);
        if (suh) {
#pragma unroll
            for (int k = 0; k < E / 8; k++) sq[k] = *reinterpret_cast<const any_uint4_t*>(suh + blk + q * E + k * 8);
        }
        issue_first_rows<K, true>(base, row_words, tk, 0, buf);
        __builtin_amdgcn_sched_barrier(0);
        stage_zeros();
        float z[E];
#pragma unroll
        for (int k = 0; k < E / 8; k++) {
            float v[8], sc[8];
            halfs_to_floats(xq[k], v);
            if (suh) halfs_to_floats(sq[k], sc);
#pragma unroll
            for (int i = 0; i < 8; i++) z[8 * k + i] = suh ? __fmul_rn(v[i], sc[i]) : v[i];
        }
#pragma unroll
        for (int h = 1; h < E; h <<= 1)
#pragma unroll
            for (int i = 0; i < E; i++)
                if ((i & h) == 0) butterfly_in_lane(z[i], z[i + h]);
        // then lanes R, 2 R, ... 32 apart
        static_for<(R == 4 ? 2 : 3), 4>([&](auto bit) {
            const uint32_t sign = lane_sign_mask(lane, bit.value);
#pragma unroll
            for (int i = 0; i < E; i++) z[i] = butterfly_dpp<bit.value>(z[i], sign);
        });
#pragma unroll
        for (int i = 0; i < E; i += 2) {
            swap_rows16(z[i], z[i + 1]);
            butterfly_in_lane(z[i], z[i + 1]);
            swap_halves32(z[i], z[i + 1]);
            butterfly_in_lane(z[i], z[i + 1]);
            swap_halves32(z[i], z[i + 1]);
            swap_rows16(z[i], z[i + 1]);
        }
        if ((lane >> 5) == upper) {
#pragma unroll
            for (int k = 0; k < E / 8; k++) stage8(fr, (q * E & 63) + 8 * k, z + 8 * k);
        }
    } else {
        // lane = (row fr, elements 32 k + 8 q .. + 7)
        const int fr = lane & 15, q = lane >> 4, col = blk + q * 8;
        uint4_t xq[4], sq[4];
        const half_t* xr = x + (size_t)min(fr, rows - 1) * in_features + col;
#pragma unroll
        for (int k = 0; k < 4; k++) xq[k] = *reinterpret_cast<const any_uint4_t*>(xr + k * 32);
        if (suh) {
#pragma unroll
            for (int k = 0; k < 4; k++) sq[k] = *reinterpret_cast<const any_uint4_t*>(suh + col + k * 32);
        }
        issue_first_rows<K, true>(base, row_words, tk, 0, buf);
        __builtin_amdgcn_sched_barrier(0);
        stage_zeros();
        if (!suh || all_plain_signs(sq)) {
            if (suh) {
#pragma unroll
                for (int k = 0; k < 4; k++) xq[k] ^= sq[k] & 0x80008000u;
            }
            // the upper half's columns differ from the lower half's in the sign of elements 64 .. 127
            const uint32_t flip = upper ? 0x80008000u : 0u;
            xq[2] ^= flip;
            xq[3] ^= flip;
            const HadamardColumns had(lane);
            static_for<0, 2>([&](auto a) {
                float4_t t[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
                static_for<0, 4>([&](auto k) {
                    const half8_t v = __builtin_bit_cast(half8_t, xq[k.value]);
                    t[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(had.template get<2 * a.value, k.value>(), v, t[0], 0, 0, 0);
                    t[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(had.template get<2 * a.value + 1, k.value>(), v, t[1], 0, 0, 0);
                });
                const float z[8] = {t[0][0], t[0][1], t[0][2], t[0][3], t[1][0], t[1][1], t[1][2], t[1][3]};
                stage8(fr, 32 * a.value + 8 * q, z);
            });
        } else {
            // any other scale vector: fp32 butterfly, the bits of wht128_lanes()
            float z[4][8];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                float sc[8];
                halfs_to_floats(xq[k], z[k]);
                halfs_to_floats(sq[k], sc);
#pragma unroll
                for (int c = 0; c < 8; c++) z[k][c] = __fmul_rn(z[k][c], sc[c]);
            }
            wht128_tile(z);
            if (upper) {
                stage8(fr, 8 * q, z[2]);
                stage8(fr, 32 + 8 * q, z[3]);
            } else {
                stage8(fr, 8 * q, z[0]);
                stage8(fr, 32 + 8 * q, z[1]);
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();

    const half_t* xa[T::NQ];
#pragma unroll
    for (int i = 0; i < T::NQ; i++) xa[i] = xw + T::operand_row(lane, i) * T::LD;
    struct Chunk {
        uint4_t v[T::NQ];
    };
    // activations of chunk c (input rows 4c.. of the tile row, each twice; EXACT 8c..)
    auto chunk = [&](int row, int c) {
        Chunk t;
#pragma unroll
        for (int i = 0; i < T::NQ; i++) t.v[i] = *reinterpret_cast<const uint4_t*>(xa[i] + row * (EXACT ? 16 : 32) + 8 * c);
        return t;
    };
    uint32_t prev = neighbour_word(buf[0][K - 1], lane);
    static_for<0, kSlots>([&](auto sc) {
        constexpr int s = sc.value;
        const uint32_t prev_next = s + 1 < kSlots ? neighbour_word(buf[s + 1 < kSlots ? s + 1 : 0][K - 1], lane) : 0u;
        __builtin_amdgcn_sched_barrier(0);
        const LaneWords<K> lw = make_lane_words<K>(prev, buf[s]);
        if constexpr (EXACT) {
            // one column after the other; the first one's products run while the second is decoded
            const Chunk x0 = chunk(s, 0), x1 = chunk(s, 1);
            half2_t wp[2][8];
            auto issue = [&](auto csc) {
                constexpr int cs = decltype(csc)::value;
                const half2_t(&w)[8] = wp[cs];
                T::mfma(x0.v, uint4_t{half2_to_bits(w[0]), half2_to_bits(w[1]), half2_to_bits(w[2]), half2_to_bits(w[3])}, acc[cs]);
                T::mfma(x1.v, uint4_t{half2_to_bits(w[4]), half2_to_bits(w[5]), half2_to_bits(w[6]), half2_to_bits(w[7])}, acc[cs]);
            };
            static_for<0, 8>([&](auto t) {
                constexpr int cs = t.value >> 2, i = t.value & 3, n = 8 * i + 4 * cs;
                static_assert(cw_col_sel(n) == cs && cw_row(n) == 2 * i && cw_row(n + 2) == 2 * i + 8);
                decode_pair2<CB>(lane_codeword<K, n>(lw), lane_codeword<K, n + 1>(lw), lane_codeword<K, n + 2>(lw),
                                 lane_codeword<K, n + 3>(lw), wp[cs][i], wp[cs][4 + i]);
                if constexpr (t.value == 4) issue(std::integral_constant<int, 0>{});
            });
            issue(std::integral_constant<int, 1>{});
        } else {
            // as dot_tile_row(): chunks 0, 2, 1, 3, the instruction of a chunk and column half a chunk late
            auto step_chunk = [](int t) constexpr { return (t >> 1) == 0 ? 0 : (t >> 1) == 1 ? 2 : (t >> 1) == 2 ? 1 : 3; };
            auto pair_n = [](int j, int cs) constexpr { return 8 * (j & 3) + 4 * cs + 2 * (j >> 2); };
            Chunk xc[4];
            uint4_t wb[8];
            xc[0] = chunk(s, 0);
            xc[2] = chunk(s, 2);
            auto issue = [&](auto tc) {
                constexpr int t = tc.value;
                T::mfma(xc[step_chunk(t)].v, wb[t], acc[t & 1]);
            };
            static_for<0, 8>([&](auto tc) {
                constexpr int t = tc.value, c = step_chunk(t), cs = t & 1;
                constexpr int n0 = pair_n(2 * c, cs), n1 = pair_n(2 * c + 1, cs);
                static_assert(cw_col_sel(n0) == cs && cw_row(n0) == 4 * c && cw_row(n1) == 4 * c + 2);
                wb[t].x = scramble<CB>(lane_codeword<K, n0>(lw));
                wb[t].y = scramble<CB>(lane_codeword<K, n0 + 1>(lw));
                if constexpr (t >= 1) issue(std::integral_constant<int, t - 1>{});
                if constexpr (t == 2) xc[1] = chunk(s, 1);
                if constexpr (t == 4) xc[3] = chunk(s, 3);
                wb[t].z = scramble<CB>(lane_codeword<K, n1>(lw));
                wb[t].w = scramble<CB>(lane_codeword<K, n1 + 1>(lw));
            });
            issue(std::integral_constant<int, 7>{});
        }
        __builtin_amdgcn_sched_barrier(0);
        prev = prev_next;
    });
}

// Output transform of MR rows of a 128-column block, two columns per lane: the fp16 cast at
// ponyexl3/ref/forward.py:41, Hadamard, svh, bias (forward.py:42-45).
template <int MR>
__device__ __forceinline__ void batch_finish(float (&a)[MR], float (&b)[MR], bool svh, half2_t sv, bool bias, half2_t bv,
                                             int lane, half2_t (&o)[MR]) {
#pragma unroll
    for (int i = 0; i < MR; i++) {
        a[i] = (float)(half_t)a[i];
        b[i] = (float)(half_t)b[i];
        wht128_lanes(a[i], b[i], lane);
        a[i] = __fmul_rn(a[i], kHadScaleF);
        b[i] = __fmul_rn(b[i], kHadScaleF);
        if (svh) {
            a[i] = __fmul_rn(a[i], (float)sv.x);
            b[i] = __fmul_rn(b[i], (float)sv.y);
        }
        o[i].x = (half_t)a[i];
        o[i].y = (half_t)b[i];
        if (bias) {
            o[i].x = o[i].x + bv.x;
            o[i].y = o[i].y + bv.y;
        }
    }
}

// grid (column groups, partial rows); a wave of a workgroup is one split. The two reductions
// are those of linear_small_kernel, described there.
template <int K, int CB, int R, bool ATOMIC, int NW>
__global__ __launch_bounds__(NW * 64, R > 8 ? 4 : 1) void linear_batch_kernel(
    const uint32_t* __restrict__ trellis, const half_t* __restrict__ x, const half_t* __restrict__ suh,
    const half_t* __restrict__ svh, const half_t* __restrict__ bias, half_t* __restrict__ y, float* partial,
    int* counters, const int* __restrict__ group_sub, int in_tiles, int out_tiles, int rows, int n_groups,
    int* status, int spin_limit) {
    using T = BatchTile<R, CB>;
    constexpr int MR = (R + NW - 1) / NW;  // batch rows per wave in the reduction: wave, wave + NW, ...
    constexpr size_t kXsBytes = sizeof(half_t) * NW * (R + 1) * T::LD;
    constexpr size_t kRedBytes = sizeof(float) * NW * R * 128;
    __shared__ __attribute__((aligned(16))) unsigned char smem[kXsBytes > kRedBytes ? kXsBytes : kRedBytes];
    float (*red)[R][128] = reinterpret_cast<float (*)[R][128]>(smem);
    const int g = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int split = blockIdx.y * NW + wave, n_splits = in_tiles >> 2;
    const int sub = group_sub ? group_sub[g] : 0;
    const int in_features = in_tiles * 16;
    typename T::acc_t acc[2];
#pragma unroll
    for (int cs = 0; cs < 2; cs++)
#pragma unroll
        for (int i = 0; i < T::NQ; i++) {
#pragma unroll
            for (int c = 0; c < (T::WIDE ? 16 : 4); c++) acc[cs].v[i][c] = 0.f;
            if constexpr (!T::WIDE) asm("" : "+a"(acc[cs].v[i]));  // as keep_in_agprs()
        }
    if (split < n_splits)
        batch_main<K, CB, R>(trellis + (size_t)g * 8 * (8 * K) + lane * K, (size_t)out_tiles * (8 * K), split * 4, x,
                             in_features, rows, suh ? suh + (size_t)sub * in_features : nullptr,
                             reinterpret_cast<half_t*>(smem) + wave * (R + 1) * T::LD, lane, acc);
    // requested now, needed only by the finishing workgroup: by then they are here
    const size_t col = (size_t)g * 128 + 2 * lane;
    // (zeros where there are none: batch_finish() takes them by value, and an undefined argument would let the compiler
    // conclude that both pointers are there)
    half2_t sv{(half_t)0.f, (half_t)0.f}, bv = sv;
    if (svh) sv = half2_t{svh[col], svh[col + 1]};
    if (bias) bv = half2_t{bias[col], bias[col + 1]};
    const int c0 = (lane >> 3) * 16 + (lane & 7);
    __syncthreads();  // nobody reads staged activations any more
#pragma unroll
    for (int m = 0; m < R; m++) {
        red[wave][m][c0] = acc[0].row(m);
        red[wave][m][c0 + 8] = acc[1].row(m);
    }
    __syncthreads();
    const size_t out_total = (size_t)n_groups * 128;
    const int wg_splits = (n_splits + NW - 1) / NW;  // partial rows per group
    float va[MR], vb[MR];
#pragma unroll
    for (int i = 0; i < MR; i++) {
        const int m = min(wave + NW * i, R - 1);
        float2_t s = *reinterpret_cast<const float2_t*>(&red[0][m][2 * lane]);
#pragma unroll
        for (int w = 1; w < NW; w++) {  // wave order
            const float2_t t = *reinterpret_cast<const float2_t*>(&red[w][m][2 * lane]);
            s.x = __fadd_rn(s.x, t.x);
            s.y = __fadd_rn(s.y, t.y);
        }
        va[i] = s.x;
        vb[i] = s.y;
    }
    half2_t o[MR];
    if constexpr (ATOMIC) {
        unsigned long long* sums = reinterpret_cast<unsigned long long*>(counters) + col;
        const int bits = fix_count_bits(wg_splits);
        unsigned long long w0[MR], w1[MR];
#pragma unroll
        for (int i = 0; i < MR; i++) {
            w0[i] = w1[i] = 0;
            const int m = wave + NW * i;
            if (m < rows) {
                const unsigned long long ax = fix_word(va[i], bits), ay = fix_word(vb[i], bits);
                unsigned long long* slot = sums + (size_t)m * out_total;
                w0[i] = __hip_atomic_fetch_add(slot, ax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + ax;
                w1[i] = __hip_atomic_fetch_add(slot + 1, ay, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + ay;
            }
        }
        // Finisher = the workgroup whose add brought (row 0, first column of the group) to wg_splits.
        // The adds to other words that are still missing then come from waves that have passed
        // the same barrier: the polls wait for waves that run, not for one to be scheduled.
        __shared__ int finishes, gave_up;
        if (threadIdx.x == 0) {
            finishes = fix_count(w0[0], bits) == wg_splits;
            gave_up = 0;
        }
        __syncthreads();
        if (!finishes) return;
#pragma unroll
        for (int i = 0; i < MR; i++) {
            const int m = wave + NW * i;
            if (m >= rows) break;
            const unsigned long long* slot = sums + (size_t)m * out_total;
            auto complete = [&]() {
                return __ballot(fix_count(w0[i], bits) == wg_splits && fix_count(w1[i], bits) == wg_splits) == ~0ull;
            };
            bool ok = complete();
            for (int spin = 0; !ok && spin < spin_limit; spin++) {
                w0[i] = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                w1[i] = __hip_atomic_load(slot + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ok = complete();
            }
            if (!ok && lane == 0) gave_up = 1;
        }
        __syncthreads();
        const bool bad = gave_up != 0;  // the whole group's outputs become NaN, its accumulators stay
        if (bad && status && threadIdx.x == 0)
            __hip_atomic_fetch_or(status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < MR; i++) {
            if (!bad && wave + NW * i < rows) {
                unsigned long long* slot = sums + (size_t)(wave + NW * i) * out_total;
                __hip_atomic_store(slot, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(slot + 1, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            va[i] = fix_value(w0[i], bits);
            vb[i] = fix_value(w1[i], bits);
        }
        batch_finish<MR>(va, vb, svh, sv, bias, bv, lane, o);
#pragma unroll
        for (int i = 0; i < MR; i++) {
            if (bad) o[i].x = o[i].y = bits_to_half(0x7E00);
            if (wave + NW * i < rows) *reinterpret_cast<half2_t*>(y + (size_t)(wave + NW * i) * out_total + col) = o[i];
        }
    } else {
        __shared__ int last_flag;
#pragma unroll
        for (int i = 0; i < MR; i++) {
            const int m = wave + NW * i;
            if (m < rows)
                __hip_atomic_store(reinterpret_cast<uint64_t*>(partial + ((size_t)blockIdx.y * rows + m) * out_total + col),
                                   __builtin_bit_cast(uint64_t, float2_t{va[i], vb[i]}), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) {
            const int seen = __hip_atomic_fetch_add(&counters[g], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            last_flag = seen == wg_splits - 1;
        }
        __syncthreads();
        if (!last_flag) return;
        asm volatile("" ::: "memory");
        // device-scope loads, eight partial rows of every batch row in flight, added in split order
        // (a batch that runs past the last partial row re-reads that row and drops it)
        constexpr int SB = 8;
#pragma unroll
        for (int i = 0; i < MR; i++) va[i] = vb[i] = 0.f;
        const size_t stride = (size_t)rows * out_total;
        for (int s0 = 0; s0 < wg_splits; s0 += SB) {
            uint64_t v[SB][MR];
#pragma unroll
            for (int j = 0; j < SB; j++)
#pragma unroll
                for (int i = 0; i < MR; i++)
                    v[j][i] = __hip_atomic_load(
                        reinterpret_cast<const uint64_t*>(partial + (size_t)min(s0 + j, wg_splits - 1) * stride +
                                                          (size_t)min(wave + NW * i, rows - 1) * out_total + col),
                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int j = 0; j < SB; j++)
                if (s0 + j < wg_splits) {
#pragma unroll
                    for (int i = 0; i < MR; i++) {
                        const float2_t f = __builtin_bit_cast(float2_t, v[j][i]);
                        va[i] = __fadd_rn(va[i], f.x);
                        vb[i] = __fadd_rn(vb[i], f.y);
                    }
                }
        }
        batch_finish<MR>(va, vb, svh, sv, bias, bv, lane, o);
#pragma unroll
        for (int i = 0; i < MR; i++) {
            const int m = wave + NW * i;
            if (m < rows) *reinterpret_cast<half2_t*>(y + (size_t)m * out_total + col) = o[i];
        }
        if (threadIdx.x == 0) __hip_atomic_store(&counters[g], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Rows that the kernel stages for a batch: 4, 8 or 16.
static int batch_rows(int rows) { return rows <= 4 ? 4 : rows <= 8 ? 8 : 16; }

// Accumulators against partial rows, per launch: the memory side retires about 75 k atomics per
// microsecond, all workgroups reach their reduction at about the same time, and the chain of store, counter and
// reload costs 1-2 us more than a returning atomic. Where the two met in a sweep of 2..8 rows, by
// millions of weights: 10 180 k atomics, 17 200 k, 42 520 k, 52 660 k, 89 1500 k, 178 1750 k; at 3
// rows of 8192 -> 5120 11.9 against 15.0 us, at 8 rows 22.0 against 17.0 (four waves per workgroup).
// Launches that linear_small_kernel would reduce through fp32 partial rows (four whole blocks to each)
// take accumulators only where these are as good: up to 31 contributors, 30 fraction bits.
// EXL3_LINEAR_MAX_ATOMICS, where it is set, takes the place of both lines.
bool linear_batch_uses_atomics(int rows, int n_groups, GemvPlan plan) {
    if (rows > 8 || plan.n_partials() > kFixMaxContributors) return false;
    const long long atomics = (long long)n_groups * plan.n_partials() * 128 * rows;
    if (linear_max_atomics_set() >= 0) return atomics <= linear_small_max_atomics(rows);
    const long long whole_blocks = (long long)n_groups * ((plan.n_splits + 7) / 8) * 128 * rows;
    if (plan.n_partials() > kFixFineContributors && whole_blocks > linear_small_max_atomics(rows)) return false;
    const long long weights = (long long)n_groups * 128 * plan.n_splits * 64;
    return atomics <= 60000 + weights / 100;
}

// Half blocks double the waves and rotate 128 values for 64 rows of weights, which pays while the
// chip is not full: (blocks of the reduction) x (column groups) up to a line that a sweep of 1664 -> 2560
// to 5120 -> 34816 gave. Against the kernels that take over there (us, 3INST / MCG):
//   2..4 rows  8192 -> 5120 (2560) 3 rows K = 4 13.4 -> 11.6; 6144 -> 12288 (4608) K = 4 17.2 -> 18.3, K = 5
//              21.3 -> 18.5; 5120 -> 34816 (10880) K = 4 32.3 -> 33.8, K = 6 39.4 -> 35.4, K = 8 48.8 -> 41.6
//   5..8 rows  1664 -> 2560 (260) 5 rows 11.8 -> 7.2; 5120 -> 10240 (3200) 8 rows K = 4 20.6 -> 19.5; 6144 -> 12288
//              5 rows K = 4 21.7 -> 22.7, K = 6 25.5 -> 23.6
//   9..16 rows 1664 -> 2560 16 rows 11.2 -> 9.1 (with the rotation's launch), 2560 -> 4096 12.5 -> 9.4, 8192 -> 5120
//              21.2 -> 18.5; 5120 -> 10240 20.2 -> 21.7
// Reductions too long for fine accumulators (linear_batch_uses_atomics) at 3..4 rows pay 3 us for their partial
// rows and end earlier: 17408 -> 3328 (3536) K = 4 18.1 -> 17.9, 16384 -> 3456 (3456) K = 4 16.7 -> 17.2, 17408 ->
// 4352 (4624) K = 6 22.7 -> 21.1, 17408 -> 5120 (5440) K = 6 22.7 -> 23.4, K = 8 26.7 -> 25.1.
bool linear_batch_applies(int rows, int in_tiles, int n_groups, int K) {
    if (rows < 2 || rows > kLinearBatchMaxRows) return false;
    const long long units = (long long)(in_tiles / 8) * n_groups;
    if (rows > 8) return units <= 2700;
    if (rows > 4) return units <= (K >= 5 ? 5000 : 3300);
    if (rows > 2 && in_tiles > 32 * kFixFineContributors) return units <= (K >= 7 ? 12000 : K == 6 ? 5000 : 3400);
    // (the top line keeps the partial rows of exl3_linear_forward_static within its array)
    return units <= (K >= 6 ? 12000 : K == 5 ? 5000 : 4096);
}

// Eight waves per workgroup halve the partial rows. Up to four rows the workgroup's sum is one
// round of additions for four waves, and four waves are the better ones while the atomics are few.
GemvPlan plan_linear_batch(int rows, int in_tiles, int n_groups) {
    GemvPlan plan{in_tiles / 4, 4, 4, true};
    if (rows > 4 || !linear_batch_uses_atomics(rows, n_groups, plan)) plan.wg_waves = 8;
    return plan;
}

int launch_linear_batch(const uint16_t* x, int rows, const uint16_t* trellis, int in_tiles, int out_tiles, int K, int cb,
                        const uint16_t* suh, int n_sub, const int32_t* group_sub, const uint16_t* svh,
                        const uint16_t* bias, uint16_t* y, float* partial, int* counters, GemvPlan plan,
                        hipStream_t stream, int* status) {
    if (int rc = check_k_cb(K, cb)) return rc;
    if (!x || !trellis || !y || !counters) return EXL3_E_NULL_POINTER;
    if (rows < 1 || rows > kLinearBatchMaxRows || n_sub < 1 || in_tiles < 8 || out_tiles < 8 || in_tiles % 8 ||
        out_tiles % 8)
        return EXL3_E_BAD_SHAPE;
    if (n_sub > 1 && (!group_sub || !suh)) return EXL3_E_BAD_INDEX;
    const int n_groups = out_tiles / 8, r = batch_rows(rows);
    if (!plan.batch || plan.tk_per_split != 4 || plan.n_splits != in_tiles / 4 || plan.n_partials() > 65535 ||
        !(plan.wg_waves == 8 || (plan.wg_waves == 4 && r == 4)))
        return EXL3_E_BAD_SHAPE;
    const bool atomic = linear_batch_uses_atomics(rows, n_groups, plan);
    if (atomic && (reinterpret_cast<uintptr_t>(counters) & 7)) return EXL3_E_BAD_SHAPE;
    if (!atomic && !partial) return EXL3_E_NULL_POINTER;
    const int spin_limit = reduction_spin_limit();
    const dim3 grid((unsigned)n_groups, (unsigned)plan.n_partials());
    return dispatch_k_cb(K, cb, [&](auto k, auto c) {
        auto launch = [&](auto rc, auto at, auto nw) {
            linear_batch_kernel<k.value, c.value, rc.value, at.value, nw.value><<<grid, dim3(nw.value * 64), 0, stream>>>(
                reinterpret_cast<const uint32_t*>(trellis), reinterpret_cast<const half_t*>(x),
                reinterpret_cast<const half_t*>(suh), reinterpret_cast<const half_t*>(svh),
                reinterpret_cast<const half_t*>(bias), reinterpret_cast<half_t*>(y), partial, counters, group_sub,
                in_tiles, out_tiles, rows, n_groups, status, spin_limit);
        };
        using Y = std::true_type;
        using N = std::false_type;
        using R4 = std::integral_constant<int, 4>;
        using R8 = std::integral_constant<int, 8>;
        if (r == 16) launch(std::integral_constant<int, 16>{}, N{}, R8{});
        else if (r == 8) atomic ? launch(R8{}, Y{}, R8{}) : launch(R8{}, N{}, R8{});
        else if (plan.wg_waves == 8) atomic ? launch(R4{}, Y{}, R8{}) : launch(R4{}, N{}, R8{});
        else if (atomic) launch(R4{}, Y{}, R4{});
        else return (int)EXL3_E_BAD_SHAPE;  // plan_linear_batch() takes eight waves there
        return launch_status();
    });
}

}  // namespace exl3
