// Building blocks of the kernels that take a few dozen rows at a time: the weights go from
// the trellis through registers straight into v_mfma_f32_32x32x16_f16; activations and packed
// words pass through LDS, decoded weights do not.
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
// 32 * MR rows x 32 * NKS halfs, and the waves' trellis words are filled two steps ahead by
// direct loads into one of three LDS stages; one barrier per step, in its middle.
//
// Per wave and step: about 140 VALU instructions (decode), 4 * MR matrix instructions of 32
// cycles, 2 * MR + 2 LDS reads. VALU issue (about 550 cycles) sets the pace up to MR = 4, where
// the matrix pipe catches up. Two workgroups of 64 rows share a CU up to K = 5, from there on and
// with more rows one has it to itself. 333 rows of 17408 -> 5120 (K = 5), whole layer: 115 us with
// words in registers and the barrier at the step's end, 101 in this form, 97 with half quads and
// direct loads one by one between the matrix instructions; the prefill GEMM 115. 1537 tokens
// through 257 experts: gate/up 150 us, down 87 with two k-slices, 73 with one.
#pragma once

#include "exl3_device.hpp"

namespace exl3 {

template <int MR, int NKS>
struct RowsTile {
    static_assert(NKS == 1 || NKS == 2 || NKS == 4, "LDS rows of 64, 128 or 256 bytes");
    static constexpr int BM = 32 * MR, BK = 32 * NKS, CHUNKS = BK / 8;
    static constexpr int STAGE = BM * BK;              // halfs per stage
    static constexpr int FILLS = STAGE * 2 / 1024;     // wave-wide direct loads per stage
    // 16-byte chunk c of row r is stored at chunk c ^ swizzle(r): a fragment read (32 rows,
    // one chunk) then touches every bank equally
    static __device__ __forceinline__ int swizzle(int row) {
        return NKS == 1 ? (row >> 2) & 3 : NKS == 2 ? (row >> 1) & 7 : row & 15;
    }
};

// Byte offset in the activation matrix of what lane `lane` of fill `f` of a stage copies
// (relative to the tile's first row and the step's first column); rows past `last_row` repeat
// it. row_of: where in the matrix a row of the tile is.
template <int MR, int NKS, typename RowOf>
__device__ __forceinline__ uint32_t rows_fill_offset(int f, int lane, int last_row, size_t ldx, RowOf row_of) {
    using T = RowsTile<MR, NKS>;
    const int row = f * (64 / T::CHUNKS) + lane / T::CHUNKS;
    const int chunk = (lane % T::CHUNKS) ^ T::swizzle(row);
    return (uint32_t)((size_t)row_of(min(row, last_row)) * ldx * 2 + chunk * 16);
}
template <int MR, int NKS>
__device__ __forceinline__ uint32_t rows_fill_offset(int f, int lane, int last_row, size_t ldx) {
    return rows_fill_offset<MR, NKS>(f, lane, last_row, ldx, [](int row) { return row; });
}

// Half H of quad I (0..3) of column tile pair CS: the quad is rows 2I, 2I + 1 and 2I + 8, 2I + 9
// of the lane's column; its first half leaves two codewords scrambled in `x`.
template <int K, int CB, int CS, int I, int H>
__device__ __forceinline__ void decode_half_quad(const LaneWords<K>& lw, uint32_t (&x)[2], half2_t (&wp)[2][4]) {
    constexpr int na = 4 * (2 * I + CS), nb = na + 2;
    static_assert(cw_col_sel(na) == CS && cw_row(na) == 2 * I && cw_row(nb) == 2 * I + 8);
    if constexpr (CB == CB_MUL1) {
        wp[H][I] = decode_mul1_pair(lane_codeword<K, na + 2 * H>(lw), lane_codeword<K, na + 2 * H + 1>(lw));
    } else if constexpr (H == 0) {
        x[0] = scramble<CB>(lane_codeword<K, na>(lw));
        x[1] = scramble<CB>(lane_codeword<K, na + 1>(lw));
    } else {
        add_halves_pack2(x[0], x[1], scramble<CB>(lane_codeword<K, nb>(lw)), scramble<CB>(lane_codeword<K, nb + 1>(lw)),
                         wp[0][I], wp[1][I]);
    }
}

// Trellis words of a wave and step, in LDS as in memory: 64 lanes x K dwords.
template <int K>
struct RowsWords {
    static constexpr int STAGE = 64 * K;                // dwords of one wave and stage
    static constexpr int LOADS = (16 * K + 63) / 64;    // wave-wide direct loads of 16 bytes a lane
};

// acc[mr][cs] = D of 32x32: column m (lane m of the decode: tile m >> 3, column (m & 7) +
// 8 cs of it) x activation row 32 mr + n. A lane holds n = lane & 31 and m = 8 (i >> 2) +
// 4 (lane >> 5) + (i & 3), i = 0..15.
//   w         the wave's trellis words at step 0 (uniform): four tiles of its first tile row;
//             w_row dwords further the second; w_step dwords further per step
//   a         activation tile at step 0 (uniform); a_off: rows_fill_offset of the wave's LPW
//             fills, which go to LDS bytes fill_to + 1024 i (fills: whether this wave has any)
//   stages    the activation stages; read_off: the lane's first fragment, see rows_read_base
//   words     the wave's first word stage (16-byte aligned); word_stage dwords to its next
//
// Everything that comes from memory goes to LDS by direct loads, two steps and more ahead, so no
// register waits for memory and the only wait is the counted one at the barrier: the compiler
// cannot count the direct loads, and its waits for trellis words in registers drained them
// to one step. One barrier in the middle of a step: before it the matrix pipe works on column
// tile pair 0 while pair 1 is decoded, behind it on pair 1 while pair 0 of the next step is
// decoded and that step's fragments are read, so that a wave keeps both pipes busy by itself
// (decode of a pair: about 68 VALU instructions of 4 cycles between its 2 MR matrix
// instructions of 32 cycles).
template <int K, int CB, int MR, int NKS, int LPW>
__device__ __forceinline__ void rows_main(const uint32_t* w, size_t w_row, size_t w_step, const char* a,
                                          const uint32_t (&a_off)[LPW], bool fills, uint32_t fill_to,
                                          const half_t* stages, int read_off, const uint32_t* words, int word_stage,
                                          int nsteps, int lane, float16_t (&acc)[MR][2]) {
    using T = RowsTile<MR, NKS>;
    using W = RowsWords<K>;
    constexpr int kBatch = LPW + W::LOADS;
    const int last = nsteps - 1;
    uint32_t w_off[W::LOADS];
#pragma unroll
    for (int i = 0; i < W::LOADS; i++) {
        const int c = 64 * i + lane;  // 16-byte chunk
        w_off[i] = c < 8 * K ? 16u * c : (uint32_t)w_row * 4u + 16u * (c - 8 * K);
    }
    const uint32_t words_to = lds_byte_address(words);
    // direct load I of step t's batch
    auto load_one = [&](int t, int stage, auto ic) {
        constexpr int i = ic.value;
        const int tc = min(t, last);
        if constexpr (i < LPW) {
            if (fills)
                load_lds16(a + (size_t)tc * (T::BK * 2), a_off[i], fill_to + (uint32_t)(stage * T::STAGE + i * 512) * 2);
        } else {
            constexpr int j = i - LPW;
            if (64 * (j + 1) <= 16 * K || lane < 16 * K - 64 * j)
                load_lds16(w + (size_t)tc * w_step, w_off[j], words_to + (uint32_t)(stage * word_stage + j * 256) * 4);
        }
    };
    auto load_batch = [&](int t, int stage) { static_for<0, kBatch>([&](auto i) { load_one(t, stage, i); }); };
    // All but the last `n` batches of this wave have landed, and all waves have got here.
    auto arrive = [&](auto n) {
        constexpr int b = decltype(n)::value;
        if (fills) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(b * kBatch) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(b * W::LOADS) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    LaneWords<K> lw;
    const int prev = ((lane & ~7) | ((lane + 7) & 7)) * K + K - 1;
    auto read_words = [&](int stage) {
        const uint32_t* q = words + stage * word_stage;
        lw.w[0] = q[prev];
#pragma unroll
        for (int i = 0; i < K; i++) lw.w[i + 1] = q[lane * K + i];
    };
    half8_t af[MR][2];
    auto read_a = [&](int stage, auto kh) {
        const half_t* r = stages + stage * T::STAGE;
#pragma unroll
        for (int mr = 0; mr < MR; mr++)
            af[mr][kh.value] = *reinterpret_cast<const half8_t*>(r + (read_off ^ (kh.value * 8)) + mr * 32 * T::BK);
    };
    half2_t wp[2][2][4];  // [cs][kh]
    // 2 MR matrix instructions of pair cs; the eight half quads of pair ds, and whatever
    // after(i) issues, go evenly between them
    uint32_t x[2];
    auto half_step = [&](auto csc, auto dsc, auto after) {
        constexpr int cs = decltype(csc)::value, ds = decltype(dsc)::value;
        static_for<0, 2 * MR>([&](auto ic) {
            constexpr int i = ic.value, kh = i / MR, mr = i % MR;
            const uint4_t q = {half2_to_bits(wp[cs][kh][0]), half2_to_bits(wp[cs][kh][1]),
                               half2_to_bits(wp[cs][kh][2]), half2_to_bits(wp[cs][kh][3])};
            acc[mr][cs] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, q), af[mr][kh],
                                                                 acc[mr][cs], 0, 0, 0);
            after(ic);
            static_for<8 * i / (2 * MR), 8 * (i + 1) / (2 * MR)>(
                [&](auto h) { decode_half_quad<K, CB, ds, h.value / 2, h.value % 2>(lw, x, wp[ds]); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using N0 = std::integral_constant<int, 0>;
    using N1 = std::integral_constant<int, 1>;
    using N2 = std::integral_constant<int, 2>;
    load_batch(0, 0);
    load_batch(1, 1);
    load_batch(2, 2);
    // zeros by the matrix pipe, which idles here: 2 MR instructions in place of 32 MR moves (twice that
    // where the compiler joins a loop that may not run at all; nsteps >= 1)
#pragma unroll
    for (int mr = 0; mr < MR; mr++)
#pragma unroll
        for (int cs = 0; cs < 2; cs++)
            acc[mr][cs] = __builtin_amdgcn_mfma_f32_32x32x16_f16(half8_t{}, half8_t{}, float16_t{}, 0, 0, 0);
    arrive(N2{});
    read_words(0);
    read_a(0, N0{});
    read_a(0, N1{});
    static_for<0, 8>([&](auto h) { decode_half_quad<K, CB, 0, h.value / 2, h.value % 2>(lw, x, wp[0]); });
    // no scalar load is under way in the loop, so that waits there can count the LDS reads
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    int s0 = 0, s1 = 1;  // stages of step t and t + 1
    int t = 0;
    do {
        half_step(N0{}, N1{}, [](auto) {});
        arrive(N1{});  // step t + 1 is in LDS; stage s0 has been read by every wave
        read_words(s1);
        __builtin_amdgcn_sched_barrier(0);
        half_step(N1{}, N0{}, [&](auto ic) {
            constexpr int i = ic.value;
            if constexpr (i == MR - 1) read_a(s1, N0{});
            if constexpr (i == 2 * MR - 1) read_a(s1, N1{});
            static_for<kBatch * i / (2 * MR), kBatch * (i + 1) / (2 * MR)>([&](auto j) { load_one(t + 3, s0, j); });
        });
        s0 = s1;
        s1 = s1 == 2 ? 0 : s1 + 1;
    } while (++t < nsteps);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no direct load lands in LDS after this
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

// Sums of two k-slices: the wave of slice ks keeps columns cs = ks. `ex` holds MR*4 float4 per
// lane and wave; every wave passes its other half to its partner (wave ^ 1).
template <int MR>
__device__ __forceinline__ void rows_add_slices2(float16_t (&acc)[MR][2], float4_t* ex, int wave, int lane,
                                                 float16_t (&sum)[MR]) {
    const bool second = wave & 1;
#pragma unroll
    for (int mr = 0; mr < MR; mr++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float4_t v;
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] = second ? acc[mr][0][4 * i + c] : acc[mr][1][4 * i + c];
            ex[((wave ^ 1) * MR * 4 + mr * 4 + i) * 64 + lane] = v;
        }
    __syncthreads();
#pragma unroll
    for (int mr = 0; mr < MR; mr++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float4_t v = ex[(wave * MR * 4 + mr * 4 + i) * 64 + lane];
#pragma unroll
            for (int c = 0; c < 4; c++)
                sum[mr][4 * i + c] = __fadd_rn(second ? acc[mr][1][4 * i + c] : acc[mr][0][4 * i + c], v[c]);
        }
    __syncthreads();
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

// Whether the scale values of all lanes are +-1, eight halfs at a time (packed sign words, the
// usual case): a sign flip on fp16 bits is then all the product needs.
template <int N>
__device__ __forceinline__ bool all_plain_signs(const uint4_t (&s)[N]) {
    uint32_t not_one = 0;
#pragma unroll
    for (int k = 0; k < N; k++) {
        const uint4_t m = (s[k] & 0x7FFF7FFFu) ^ 0x3C003C00u;
        not_one |= m.x | m.y | m.z | m.w;
    }
    return __ballot(not_one != 0) == 0;
}

// Unnormalised Hadamard-128 in fp32 on the layout of HadamardColumns: v[k][t] = element 32 k +
// 8 (lane >> 4) + t of row lane & 15. Stages in the order of the element bits, a + b and a - b
// each: the bits of wht128_lanes() and wht128_wide(). For rows whose scale vector is general: a
// product of two halfs has 22 bits and reaches 2^32, which no pair of halfs holds (a high part
// above 65504 is infinite, a low part below 2^-24 is lost).
// wht32_tile: element bits 0..4, one column part; wht128_tile: all seven.
__device__ __forceinline__ void wht32_tile(float (&v)[8]) {
#pragma unroll
    for (int h = 1; h < 8; h <<= 1)
#pragma unroll
        for (int t = 0; t < 8; t++)
            if ((t & h) == 0) butterfly_in_lane(v[t], v[t + h]);
#pragma unroll
    for (int t = 0; t < 8; t += 2) {
        swap_rows16(v[t], v[t + 1]);
        butterfly_in_lane(v[t], v[t + 1]);
        swap_halves32(v[t], v[t + 1]);
        butterfly_in_lane(v[t], v[t + 1]);
        swap_halves32(v[t], v[t + 1]);
        swap_rows16(v[t], v[t + 1]);
    }
}
__device__ __forceinline__ void wht128_tile(float (&v)[4][8]) {
#pragma unroll
    for (int k = 0; k < 4; k++) wht32_tile(v[k]);
#pragma unroll
    for (int h = 1; h < 4; h <<= 1)
#pragma unroll
        for (int k = 0; k < 4; k++)
            if ((k & h) == 0) {
#pragma unroll
                for (int t = 0; t < 8; t++) butterfly_in_lane(v[k][t], v[k + h][t]);
            }
}

}  // namespace exl3
