// Building blocks of the kernels that take a few dozen rows at a time: the weights go from
// the trellis through registers straight into v_mfma_f32_32x32x16_f16, only the activations
// pass through LDS.
//
// Geometry. A wave decodes 64 columns x 32 reduction rows per step: lanes 0..31 hold four
// tiles of one tile row, lanes 32..63 the same four tile columns of the next one, 32
// codewords per lane = columns u and u + 8 of its tile over 16 rows. Eight consecutive rows
// of a column are one lane's share of a 32x32x16 operand whose k-slots are rows 0..7 (or
// 8..15) of the two tile rows - the order of k-slots is free as long as the activations use
// the same - so the decoded pairs are the operand: no exchange between lanes, no LDS write.
// Against LDS-staged weights this takes 4 KiB of ds_write and 4 KiB of ds_read per 2048
// weights off the LDS pipe, which was as busy as the VALU.
//
// A workgroup holds NKS k-slices (waves that share columns and split the 32 * NKS rows of a
// step among them) of one or more 64-column strips. The activation tile of a step, BM =
// 32 * MR rows x 32 * NKS halfs, is filled two steps ahead by direct loads into one of three
// LDS stages; the trellis words are two steps ahead in registers; one barrier per step.
//
// Per wave and step: about 140 VALU instructions (decode), 4 * MR matrix instructions of 32
// cycles, 2 * MR LDS reads. VALU issue (about 550 cycles) sets the pace up to MR = 4, where
// the matrix pipe catches up; four waves per SIMD hide the latencies.
#pragma once

#include "exl3_device.hpp"

namespace exl3 {

template <int MR, int NKS>
struct RowsTile {
    static_assert(NKS == 2 || NKS == 4, "LDS rows of 128 or 256 bytes");
    static constexpr int BM = 32 * MR, BK = 32 * NKS, CHUNKS = BK / 8;
    static constexpr int STAGE = BM * BK;              // halfs per stage
    static constexpr int FILLS = STAGE * 2 / 1024;     // wave-wide direct loads per stage
    // 16-byte chunk c of row r is stored at chunk c ^ swizzle(r): a fragment read (32 rows,
    // one chunk) then touches every bank equally
    static __device__ __forceinline__ int swizzle(int row) { return NKS == 2 ? (row >> 1) & 7 : row & 15; }
};

// Byte offset in the activation matrix of what lane `lane` of fill `f` of a stage copies
// (relative to the tile's first row and the step's first column); rows past `last_row` repeat
// it.
template <int MR, int NKS>
__device__ __forceinline__ uint32_t rows_fill_offset(int f, int lane, int last_row, size_t ldx) {
    using T = RowsTile<MR, NKS>;
    const int row = f * (64 / T::CHUNKS) + lane / T::CHUNKS;
    const int chunk = (lane % T::CHUNKS) ^ T::swizzle(row);
    return (uint32_t)((size_t)min(row, last_row) * ldx * 2 + chunk * 16);
}

template <int K, int CB, int CS>
__device__ __forceinline__ void decode_column(const LaneWords<K>& lw, half2_t (&wp)[16]) {
    static_for<0, 4>([&](auto i) {
        constexpr int na = 4 * (2 * i.value + CS), nb = na + 2;
        constexpr int ia = 8 * cw_col_sel(na) + (cw_row(na) >> 1);
        constexpr int ib = 8 * cw_col_sel(nb) + (cw_row(nb) >> 1);
        decode_pair2<CB>(lane_codeword<K, na>(lw), lane_codeword<K, na + 1>(lw), lane_codeword<K, nb>(lw),
                         lane_codeword<K, nb + 1>(lw), wp[ia], wp[ib]);
    });
}

// acc[mr][cs] (+)= D of 32x32: column m (lane m of the decode: tile m >> 3, column (m & 7) +
// 8 cs of it) x activation row 32 mr + n. A lane holds n = lane & 31 and m = 8 (i >> 2) +
// 4 (lane >> 5) + (i & 3), i = 0..15.
//   w       the lane's trellis words at step 0; w_step dwords further per step
//   a       activation tile at step 0 (uniform); a_off: rows_fill_offset of the wave's LPW
//           fills, which go to LDS bytes fill_to + 1024 i (fills: whether this wave has any)
//   stages  the activation stages; read_off: the lane's first fragment, see rows_read_base
template <int K, int CB, int MR, int NKS, int LPW>
__device__ __forceinline__ void rows_main(const uint32_t* w, size_t w_step, const char* a,
                                          const uint32_t (&a_off)[LPW], bool fills, uint32_t fill_to,
                                          const half_t* stages, int read_off, int nsteps, int lane, float16_t (&acc)[MR][2]) {
    using T = RowsTile<MR, NKS>;
    const int last = nsteps - 1;
    uint32_t words[2][K];
    auto load_w = [&](int t, auto slot) {
        constexpr int s = decltype(slot)::value;
        const uint32_t* q = w + (size_t)min(t, last) * w_step;
        // the origin of the address is hidden from the optimiser, which could otherwise move
        // the load across the waits below that count it
        asm volatile("" : "+v"(q));
        const auto p = (const uint32_t __attribute__((address_space(1)))*)q;
#pragma unroll
        for (int i = 0; i < K; i++) words[s][i] = __builtin_nontemporal_load(p + i);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_a = [&](int t, int stage) {
        if (!fills) return;
        const char* p = a + (size_t)min(t, last) * (T::BK * 2);
#pragma unroll
        for (int i = 0; i < LPW; i++) load_lds16(p, a_off[i], fill_to + (uint32_t)(stage * T::STAGE + i * 512) * 2);
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    // Memory operations retire in order. A fill is followed by the trellis loads of its step (K
    // dwords: at least (K + 3) / 4), the next step's fills and that step's trellis loads: with
    // no more than those outstanding it has landed.
    constexpr int kAfterFill = LPW + 2 * ((K + 3) / 4);
    load_a(0, 0);
    load_w(0, S0{});
    load_a(1, 1);
    load_w(1, S1{});
    barrier_with_loads_in_flight<kAfterFill>();
    int s0 = 0, s2 = 2;  // stage of step t and of step t + 2
    auto step = [&](int t, auto slot) {
        const LaneWords<K> lw = finish_lane_words<K>(words[decltype(slot)::value], lane);
        __builtin_amdgcn_sched_barrier(0);
        load_a(t + 2, s2);
        __builtin_amdgcn_sched_barrier(0);
        const half_t* r = stages + s0 * T::STAGE;
        half8_t af[MR][2];
#pragma unroll
        for (int mr = 0; mr < MR; mr++)
#pragma unroll
            for (int kh = 0; kh < 2; kh++)
                af[mr][kh] = *reinterpret_cast<const half8_t*>(r + (read_off ^ (kh * 8)) + mr * 32 * T::BK);
        half2_t wp[16];
        auto contract = [&](auto csc) {
            constexpr int cs = decltype(csc)::value;
#pragma unroll
            for (int kh = 0; kh < 2; kh++) {
                const uint4_t q = {half2_to_bits(wp[8 * cs + 4 * kh]), half2_to_bits(wp[8 * cs + 4 * kh + 1]),
                                   half2_to_bits(wp[8 * cs + 4 * kh + 2]), half2_to_bits(wp[8 * cs + 4 * kh + 3])};
#pragma unroll
                for (int mr = 0; mr < MR; mr++)
                    acc[mr][cs] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, q), af[mr][kh],
                                                                         acc[mr][cs], 0, 0, 0);
            }
        };
        decode_column<K, CB, 0>(lw, wp);
        contract(S0{});
        decode_column<K, CB, 1>(lw, wp);
        contract(S1{});
        // behind the decode, so that the words can come back to the registers they left
        __builtin_amdgcn_sched_barrier(0);
        load_w(t + 2, slot);
        barrier_with_loads_in_flight<kAfterFill>();
        s0 = s0 == 2 ? 0 : s0 + 1;
        s2 = s2 == 2 ? 0 : s2 + 1;
    };
    int t = 0;
    for (; t + 1 < nsteps; t += 2) {
        step(t, S0{});
        step(t + 1, S1{});
    }
    if (t < nsteps) step(t, S0{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no fill lands in LDS after this
    __syncthreads();
}

// Halfs from the stage's start to the lane's first fragment (k-slice ks); the second 8 rows
// flip chunk bit 0, further 32-row blocks are at multiples of 32 * BK.
template <int MR, int NKS>
__device__ __forceinline__ int rows_read_base(int ks, int lane) {
    using T = RowsTile<MR, NKS>;
    const int row = lane & 31, chunk = ks * 4 + (lane >> 5) * 2;
    return row * T::BK + (chunk ^ T::swizzle(row)) * 8;
}

// Hadamard-128 on the matrix pipe with outputs eight columns to a lane. Column tile nt of
// block half a = nt >> 1 is laid out so that matrix row m stands for column 32 a + 8 (m >> 2)
// + 4 (nt & 1) + (m & 3): after a pair of tiles a lane (q = lane >> 4, activation row lane &
// 15) holds columns 32 a + 8 q .. + 7. Entry (k, n) of H has sign parity(k & n); with k = 32 ks
// + 8 q + t that is parity(t & 3 & n) ^ parity(q & m >> 2), which the lane knows, t bit 2 in
// odd tiles, and parity(ks & a) for all lanes.
struct HadamardColumns {
    uint32_t w0, w1;  // +-1 for t = 0, 1 and t = 2, 3
    __device__ __forceinline__ explicit HadamardColumns(int lane) {
        const int m = lane & 15, q = lane >> 4;
        const uint32_t flip = (__builtin_popcount(q & (m >> 2)) & 1) ? 0x80008000u : 0u;
        w0 = 0x3C003C00u ^ ((uint32_t)(m & 1) << 31) ^ flip;
        w1 = 0x3C003C00u ^ ((uint32_t)((m >> 1) & 1) << 15) ^
             ((uint32_t)(__builtin_popcount(m & 3) & 1) << 31) ^ flip;
    }
    template <int NT, int KS>
    __device__ __forceinline__ half8_t get() const {
        constexpr uint32_t uni = (__builtin_popcount((NT >> 1) & KS) & 1) ? 0x80008000u : 0u;
        constexpr uint32_t hi = uni ^ ((NT & 1) ? 0x80008000u : 0u);
        return __builtin_bit_cast(half8_t, uint4_t{w0 ^ uni, w1 ^ uni, w0 ^ hi, w1 ^ hi});
    }
    // the same for column tile 2 a + ODD with a (uniform) not known at compile time
    template <int ODD, int KS>
    __device__ __forceinline__ half8_t get_part(int a) const {
        const uint32_t uni = (__builtin_popcount(a & KS) & 1) ? 0x80008000u : 0u;
        const uint32_t hi = uni ^ (ODD ? 0x80008000u : 0u);
        return __builtin_bit_cast(half8_t, uint4_t{w0 ^ uni, w1 ^ uni, w0 ^ hi, w1 ^ hi});
    }
};

constexpr float kHadNorm = 0.088388347648318440550f;  // 1/sqrt(128)

// fp16 pair (hi, lo) with hi + lo = v up to the last bits of a 22-bit product
__device__ __forceinline__ void split_halves(float v, half_t& hi, half_t& lo) {
    hi = (half_t)v;
    lo = (half_t)(v - (float)hi);
}

// Eight halfs of a column block as bits, for the "all zero" test of a low part.
__device__ __forceinline__ uint32_t any_bits(half8_t v) {
    const uint4_t u = __builtin_bit_cast(uint4_t, v) & 0x7FFF7FFFu;
    return u.x | u.y | u.z | u.w;
}

}  // namespace exl3
