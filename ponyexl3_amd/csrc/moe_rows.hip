// Routed experts of a prefill chunk: the (token, slot) rows are sorted by expert, a
// workgroup takes up to 64 rows of one expert through 128 columns of gate AND up or 256
// columns of down (see exl3_rows.hpp for the contraction): 64-column strips times NKS k-slices.
//
// What bounds them: issue of the decode. 1537 tokens through 257 experts, NKS = 2: VALU issue 85 % and
// 77 % (gate/up, down) of the time that CUs are busy, which is 81 and 84 % of the time (2.2 and 4.4
// rounds of workgroups); 25 and 36 % of the VALU instructions stood outside the main loop. SiLU without the
// scaling that its range does not need and accumulators that the matrix pipe clears, whole call: 1537 tokens 309 -> 301 us, 400 through 65
// experts of 1024 x 256 67.9 -> 65.2; over 58 shapes of 45 to 2048 tokens 2 %. Looping
// workgroups, one launch of as many as the chip holds, were slower (gate/up 158 -> 162 us, down 94 -> 103).
//
// moe_gateup_rows_kernel ends with everything that stands between the two products: output
// transform of gate and up (ponyexl3/ref/forward.py:41-42), GLU, rotation for the down
// projection - a Hadamard block of H is exactly one 128-column group - so gate and up never
// reach memory. moe_down_rows_kernel applies its output transform and stores rows at their
// (token, slot) place.
#include "exl3_device.hpp"
#include "exl3_host.hpp"
#include "exl3_rows.hpp"
#include "exl3_glu.hpp"

#pragma clang fp contract(off)

namespace exl3 {

constexpr int kYPad = 8;  // halfs: 16-byte reads of 16 tile rows hit all banks

// The fp16 casts of the sums to an LDS tile [BM][ld], first column `col` of the wave's strip.
template <int MR>
__device__ __forceinline__ void rows_store_half(const float16_t (&sum)[MR], half_t* tile, int ld, int col, int cs,
                                                int lane) {
#pragma unroll
    for (int mr = 0; mr < MR; mr++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            half4_t o;
#pragma unroll
            for (int c = 0; c < 4; c++) o[c] = (half_t)sum[mr][4 * i + c];
            *reinterpret_cast<half4_t*>(tile + (mr * 32 + (lane & 31)) * ld + col + 16 * i + 8 * cs +
                                        4 * (lane >> 5)) = o;
        }
}

// The products of a wave (64 columns from `col`) as fp16 in an LDS tile [32 MR][ld], after the sum of
// two k-slices if there are (`ex`: LDS of the exchange, over which the tile may lie).
template <int MR, int NKS>
__device__ __forceinline__ void rows_to_tile(float16_t (&acc)[MR][2], void* ex, half_t* tile, int ld, int col, int wave,
                                             int lane) {
    if constexpr (NKS == 2) {
        float16_t sum[MR];
        rows_add_slices2<MR>(acc, static_cast<float4_t*>(ex), wave, lane, sum);
        rows_store_half<MR>(sum, tile, ld, col, wave & 1, lane);
    } else {
#pragma unroll
        for (int mr = 0; mr < MR; mr++)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                half4_t o;
#pragma unroll
                for (int c = 0; c < 4; c++) o[c] = (half_t)acc[mr][i & 1][4 * (i >> 1) + c];
                *reinterpret_cast<half4_t*>(tile + (mr * 32 + (lane & 31)) * ld + col + 8 * i + 4 * (lane >> 5)) = o;
            }
    }
}

// grid: unit = (row block b, 128-column block hg of H), dealt so that the units of a row block
// land on one XCD (they read the same activations): b = 8 (u / (8 hblocks)) + u % 8.
// table[b] = {expert, first row, end row of the expert, 0}, empty if first >= end. gather: row r of xg and xu is
// at gather[r] (or at r).
template <int K, int CB, int MR, int NKS>
__global__ __launch_bounds__(256 * NKS, 4) void moe_gateup_rows_kernel(
    const uint32_t* __restrict__ trellis, const half_t* __restrict__ xg, const half_t* __restrict__ xu,
    const int4* __restrict__ table, int n_blocks, const half_t* __restrict__ gu_svh,
    const half_t* __restrict__ dn_suh, const int* __restrict__ gather, half_t* __restrict__ xd, int n_rows, int E, int D,
    int H, int activation) {
    using T = RowsTile<MR, NKS>;
    constexpr int kFillWaves = 2 * NKS, LPW = T::FILLS / kFillWaves;
    constexpr int kParts = 2 * MR / NKS;  // of a wave, of the four 32-column parts of a row tile
    constexpr int kLd = 128 + kYPad;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int hblocks = H >> 7;
    const int set = blockIdx.x / (8 * hblocks), in_set = blockIdx.x % (8 * hblocks);
    const int b = set * 8 + (in_set & 7), hg = in_set >> 3;
    if (b >= n_blocks) return;
    const int4 blk = table[b];
    const int e = blk.x, m0 = blk.y, end = min(blk.z, n_rows);
    if (e < 0 || e >= E || m0 < 0 || m0 >= end) return;
    const int valid = min(end - m0, T::BM);

    const int proj = wave / (2 * NKS), cq = (wave / NKS) & 1, ks = wave % NKS;
    const size_t row_words = (size_t)E * 2 * (H >> 4) * (8 * K);
    const uint32_t* w = trellis + (size_t)(2 * ks) * row_words +
                        ((size_t)(proj * E + e) * (H >> 4) + hg * 8 + cq * 4) * (8 * K);
    half_t* stages = reinterpret_cast<half_t*>(lds) + proj * 3 * T::STAGE;
    uint32_t a_off[LPW];
#pragma unroll
    for (int i = 0; i < LPW; i++) 
        a_off[i] = rows_fill_offset<MR, NKS>(wave % kFillWaves * LPW + i, lane, valid - 1, D,
                                             [&](int row) { return gather ? gather[m0 + row] : row; });
    float16_t acc[MR][2];
    uint32_t* words = reinterpret_cast<uint32_t*>(reinterpret_cast<half_t*>(lds) + 2 * 3 * T::STAGE) +
                      wave * RowsWords<K>::STAGE;
    rows_main<K, CB, MR, NKS, LPW>(w, row_words, 2 * NKS * row_words,
                                   reinterpret_cast<const char*>((proj ? xu : xg) + (gather ? 0 : (size_t)m0 * D)), a_off, true,
                                   lds_byte_address(stages) + wave % kFillWaves * LPW * 1024, stages,
                                   rows_read_base<MR, NKS>(ks, lane), words, 4 * NKS * RowsWords<K>::STAGE,
                                   D / (32 * NKS), lane, acc);

    half_t* tile = reinterpret_cast<half_t*>(lds);  // [gate | up][BM][kLd]
    rows_to_tile<MR, NKS>(acc, lds, tile + proj * T::BM * kLd, kLd, cq * 64, wave, lane);
    __syncthreads();

    // Output transform, GLU and rotation: a wave takes a 16-row tile and kParts of the four
    // 32-column parts of the block.
    const int rt = wave % (2 * MR), part = wave / (2 * MR);
    const int fr = lane & 15, q = lane >> 4;
    const HadamardColumns had(lane);
    const half_t* yrow = tile + (rt * 16 + fr) * kLd + q * 8;
    auto transform = [&](const half8_t (&y)[4], auto a_const, float (&z)[8]) {
        float4_t t[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        constexpr int a = decltype(a_const)::value;
        static_for<0, 4>([&](auto k) {
            t[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(had.template get<2 * a, k.value>(), y[k.value], t[0], 0, 0, 0);
            t[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(had.template get<2 * a + 1, k.value>(), y[k.value], t[1], 0, 0, 0);
        });
#pragma unroll
        for (int c = 0; c < 8; c++) z[c] = t[c >> 2][c & 3];
    };
    // f(a) for the wave's parts a, which are compile-time values in each branch
    auto for_parts = [&](auto f) {
        static_for<0, 4 / kParts>([&](auto p) {
            if (part == p.value)
                static_for<0, kParts>([&](auto i) { f(std::integral_constant<int, p.value * kParts + i.value>{}, i); });
        });
    };
    half8_t h[kParts];
    {
        half8_t yg[4], yu[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            yg[k] = *reinterpret_cast<const half8_t*>(yrow + k * 32);
            yu[k] = *reinterpret_cast<const half8_t*>(yrow + T::BM * kLd + k * 32);
        }
        for_parts([&](auto a, auto i) {
            const int col = hg * 128 + a.value * 32 + q * 8;
            const half8_t sg = *reinterpret_cast<const half8_t*>(gu_svh + (size_t)e * 2 * H + col);
            const half8_t su = *reinterpret_cast<const half8_t*>(gu_svh + (size_t)e * 2 * H + H + col);
            float zg[8], zu[8];
            transform(yg, a, zg);
            transform(yu, a, zu);
#pragma unroll
            for (int c = 0; c < 8; c++) {
                zg[c] = (float)(half_t)(zg[c] * kHadNorm * (float)sg[c]);
                zu[c] = (float)(half_t)(zu[c] * kHadNorm * (float)su[c]);
            }
            if (activation == 1) {
#pragma unroll
                for (int c = 0; c < 8; c++) h[i.value][c] = (half_t)glu_act(zg[c], zu[c], 1);
            } else {
#pragma unroll
                for (int c = 0; c < 8; c++) h[i.value][c] = (half_t)glu_act(zg[c], zu[c], 0);
            }
        });
    }
    uint4_t ds[4];  // the expert's scales of the block, in the layout of a row
#pragma unroll
    for (int k = 0; k < 4; k++)
        ds[k] = *reinterpret_cast<const uint4_t*>(dn_suh + (size_t)e * H + hg * 128 + k * 32 + q * 8);
    __syncthreads();
    for_parts([&](auto a, auto i) {
        *reinterpret_cast<half8_t*>(tile + (rt * 16 + fr) * kLd + a.value * 32 + q * 8) = h[i.value];
    });
    __syncthreads();
    const bool store = rt * 16 + fr < valid;
    half_t* out = xd + (size_t)(m0 + rt * 16 + fr) * H + hg * 128 + q * 8;
    auto put = [&](int a, const float (&z)[8]) {
        half8_t o;
#pragma unroll
        for (int c = 0; c < 8; c++) o[c] = (half_t)(z[c] * kHadNorm);
        if (store) *reinterpret_cast<half8_t*>(out + a * 32) = o;
    };
    if (all_plain_signs(ds)) {
        half8_t v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = __builtin_bit_cast(half8_t, *reinterpret_cast<const uint4_t*>(yrow + k * 32) ^ (ds[k] & 0x80008000u));
        for_parts([&](auto a, auto) {
            float z[8];
            transform(v, a, z);
            put(a, z);
        });
    } else {
        // in fp32: column part k of the row up to element bit 4, twice over, then bits 5 and 6
        // for the wave's own parts
        auto five_stages = [&](int k, float (&v)[8]) {
            float scale[8];
            halfs_to_floats(*reinterpret_cast<const uint4_t*>(yrow + k * 32), v);
            halfs_to_floats(ds[k], scale);
#pragma unroll
            for (int t = 0; t < 8; t++) v[t] = v[t] * scale[t];
            wht32_tile(v);
        };
#pragma unroll
        for (int i = 0; i < kParts; i++) {
            const int a = part * kParts + i;
            float t[2][8], u[8], z[8];
#pragma unroll
            for (int half = 0; half < 2; half++) {
                five_stages(2 * half, t[half]);
                five_stages(2 * half + 1, u);
#pragma unroll
                for (int c = 0; c < 8; c++) t[half][c] = a & 1 ? __fsub_rn(t[half][c], u[c]) : __fadd_rn(t[half][c], u[c]);
            }
#pragma unroll
            for (int c = 0; c < 8; c++) z[c] = a & 2 ? __fsub_rn(t[0][c], t[1][c]) : __fadd_rn(t[0][c], t[1][c]);
            put(a, z);
        }
    }
}

// unit = (row block b, 256-column block g of D), XCD order as above; rows go to out[order[r]].
template <int K, int CB, int MR, int NKS>
__global__ __launch_bounds__(256 * NKS, 4) void moe_down_rows_kernel(
    const uint32_t* __restrict__ trellis, const half_t* __restrict__ xd, const int4* __restrict__ table, int n_blocks,
    const half_t* __restrict__ dn_svh, const int* __restrict__ order, half_t* __restrict__ out, int n_rows, int E,
    int D, int H) {
    using T = RowsTile<MR, NKS>;
    constexpr int LPW = 1;
    constexpr int kParts = 4 * MR / NKS;  // of a wave, of the eight 32-column parts of a row tile
    static_assert(T::FILLS <= 4 * NKS, "a fill a wave");
    constexpr int kLd = 256 + kYPad;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int gblocks = (D + 255) >> 8;
    const int set = blockIdx.x / (8 * gblocks), in_set = blockIdx.x % (8 * gblocks);
    const int b = set * 8 + (in_set & 7), g = in_set >> 3;
    if (b >= n_blocks) return;
    const int4 blk = table[b];
    const int e = blk.x, m0 = blk.y, end = min(blk.z, n_rows);
    if (e < 0 || e >= E || m0 < 0 || m0 >= end) return;
    const int valid = min(end - m0, T::BM);
    // a last block of 128 columns: its upper half repeats the lower half's and is not stored
    const bool full = g * 256 + 128 < D;

    const int cq = wave / NKS, ks = wave % NKS;
    const size_t row_words = (size_t)E * (D >> 4) * (8 * K);
    const uint32_t* w = trellis + (size_t)(2 * ks) * row_words +
                        ((size_t)e * (D >> 4) + g * 16 + (full ? cq : cq & 1) * 4) * (8 * K);
    half_t* stages = reinterpret_cast<half_t*>(lds);
    uint32_t a_off[LPW];
#pragma unroll
    for (int i = 0; i < LPW; i++) a_off[i] = rows_fill_offset<MR, NKS>(wave * LPW + i, lane, valid - 1, H);
    float16_t acc[MR][2];
    uint32_t* words = reinterpret_cast<uint32_t*>(stages + 3 * T::STAGE) + wave * RowsWords<K>::STAGE;
    rows_main<K, CB, MR, NKS, LPW>(w, row_words, 2 * NKS * row_words, reinterpret_cast<const char*>(xd + (size_t)m0 * H),
                                   a_off, wave < T::FILLS, lds_byte_address(stages) + wave * LPW * 1024, stages,
                                   rows_read_base<MR, NKS>(ks, lane), words, 4 * NKS * RowsWords<K>::STAGE,
                                   H / (32 * NKS), lane, acc);
    half_t* tile = reinterpret_cast<half_t*>(lds);  // [BM][kLd]
    rows_to_tile<MR, NKS>(acc, lds, tile, kLd, cq * 64, wave, lane);
    __syncthreads();

    // output transform: a wave takes a 16-row tile and kParts of the eight 32-column parts
    const int rt = wave % (2 * MR), part = wave / (2 * MR);
    const int fr = lane & 15, q = lane >> 4;
    const HadamardColumns had(lane);
    const int r = rt * 16 + fr;
    const size_t dst_row = r < valid ? (size_t)order[m0 + r] : 0;
    static_for<0, 8 / kParts>([&](auto p) {
        if (part != p.value) return;
        static_for<0, kParts>([&](auto i) {
            constexpr int c = p.value * kParts + i.value, half = c >> 2, a = c & 3;
            if (half && !full) return;
            const half_t* yrow = tile + (rt * 16 + fr) * kLd + half * 128 + q * 8;
            float4_t t[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            static_for<0, 4>([&](auto k) {
                const half8_t y = *reinterpret_cast<const half8_t*>(yrow + k.value * 32);
                t[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(had.template get<2 * a, k.value>(), y, t[0], 0, 0, 0);
                t[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(had.template get<2 * a + 1, k.value>(), y, t[1], 0, 0, 0);
            });
            const int col = g * 256 + half * 128 + a * 32 + q * 8;
            const half8_t sv = *reinterpret_cast<const half8_t*>(dn_svh + (size_t)e * D + col);
            half8_t o;
#pragma unroll
            for (int j = 0; j < 8; j++) o[j] = (half_t)(t[j >> 2][j & 3] * kHadNorm * (float)sv[j]);
            if (r < valid) *reinterpret_cast<half8_t*>(out + dst_row * D + col) = o;
        });
    });
}

template <int K, int MR, int NKS>
static constexpr size_t rows_lds_bytes(int tiles, int tile_cols) {
    const size_t stages = (size_t)3 * (tiles * RowsTile<MR, NKS>::STAGE * 2 + 4 * NKS * RowsWords<K>::STAGE * 4);
    const size_t exchange = NKS == 2 ? (size_t)8 * MR * 4 * 64 * 16 : 0;
    const size_t y = (size_t)tiles * RowsTile<MR, NKS>::BM * (tile_cols + kYPad) * 2;
    return stages > exchange ? (stages > y ? stages : y) : (exchange > y ? exchange : y);
}

// Workgroups of four waves (NKS = 1) instead of eight: no exchange between k-slices, twice the steps
// for a prologue and an epilogue, and four to a CU that are at different points of their work; but
// half the waves where there are too few units to fill the chip. Over 48 shapes (33 to 1537 tokens,
// 32 to 257 experts, D 1024..2048, H 256..768, K 2..8), whole prefill call:
// down, from 800 units on (by the table's length, which is 1.1 to 1.8 times the units with rows): 1 to 10 us
//   less of 45 to 320, none slower (2048 x 512, 257 experts, 9 a token: 1537 tokens K = 4 293.6 ->
//   276.1); below 1.1 us less to 2.1 us more;
// gate/up, where LDS holds one workgroup of eight waves on a CU (64 rows, K >= 6), from 400 units on:
//   1000 tokens K = 6 312.1 -> 275.6, 820 tokens through 64 experts K = 7 137.7 -> 132.5, none slower;
//   264 units 80.6 -> 84.9;
// gate/up, where it holds two, from 1300 units on: 1.3 % less of whole calls (1600 tokens, top-8 of 128 experts of
//   1152 x 768 271 -> 263, 1536 of 256 of 1024 x 384 146 -> 141; two of 13 slower, 219 -> 223 at most); below, 4 to 14 % more
//   up to 400 units and 2 % less to 2 % more on from there (1104 units 148 -> 145, 1152 158 -> 162).
constexpr long long kDownNarrowUnits = 800, kGateUpNarrowUnits = 400, kGateUpManyUnits = 1300;
constexpr size_t kLdsBytes = (size_t)160 << 10;

// block_rows: 32 or 64
int launch_moe_rows(const uint16_t* xg, const uint16_t* xu, int n_rows, const uint16_t* gu_trellis,
                    const uint16_t* gu_svh, const uint16_t* dn_trellis, const uint16_t* dn_suh,
                    const uint16_t* dn_svh, int E, int D, int H, int K, int cb, int activation,
                    const int32_t* table, int n_blocks, int block_rows, const int32_t* order, bool gather, uint16_t* xd,
                    uint16_t* out, hipStream_t stream) {
    const long long sets = (n_blocks + 7) / 8;
    const long long gu_grid = sets * 8 * (H / 128), dn_grid = sets * 8 * ((D + 255) / 256);
    if (gu_grid > 0x7FFFFFFFLL || dn_grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    auto H_ = [](const uint16_t* p) { return reinterpret_cast<const half_t*>(p); };
    return dispatch_k_cb(K, cb, [&](auto k, auto c) {
        auto go = [&](auto mrc, auto gnc, auto dnc) {
            constexpr int MR = mrc.value, GN = gnc.value, DN = dnc.value;
            constexpr size_t gu_lds = rows_lds_bytes<k.value, MR, GN>(2, 128), dn_lds = rows_lds_bytes<k.value, MR, DN>(1, 256);
            auto gu = moe_gateup_rows_kernel<k.value, c.value, MR, GN>;
            auto dn = moe_down_rows_kernel<k.value, c.value, MR, DN>;
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(gu), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)gu_lds) != hipSuccess ||
                hipFuncSetAttribute(reinterpret_cast<const void*>(dn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)dn_lds) != hipSuccess)
                return (int)EXL3_E_LAUNCH;
            gu<<<dim3((unsigned)gu_grid), dim3(256 * GN), gu_lds, stream>>>(
                reinterpret_cast<const uint32_t*>(gu_trellis), H_(xg), H_(xu), reinterpret_cast<const int4*>(table),
                n_blocks, H_(gu_svh), H_(dn_suh), gather ? order : nullptr, reinterpret_cast<half_t*>(xd), n_rows, E, D, H, activation);
            if (int rc = launch_status()) return rc;
            dn<<<dim3((unsigned)dn_grid), dim3(256 * DN), dn_lds, stream>>>(
                reinterpret_cast<const uint32_t*>(dn_trellis), H_(xd), reinterpret_cast<const int4*>(table), n_blocks,
                H_(dn_svh), order, reinterpret_cast<half_t*>(out), n_rows, E, D, H);
            return launch_status();
        };
        using N1 = std::integral_constant<int, 1>;
        using N2 = std::integral_constant<int, 2>;
        const bool many_dn = dn_grid >= kDownNarrowUnits;
        if (block_rows == 32) return many_dn ? go(N1{}, N2{}, N1{}) : go(N1{}, N2{}, N2{});
        constexpr bool one_per_cu = 2 * rows_lds_bytes<k.value, 2, 2>(2, 128) > kLdsBytes;
        if (gu_grid >= (one_per_cu ? kGateUpNarrowUnits : kGateUpManyUnits))
            return many_dn ? go(N2{}, N1{}, N1{}) : go(N2{}, N1{}, N2{});
        return many_dn ? go(N2{}, N2{}, N1{}) : go(N2{}, N2{}, N2{});
    });
}

}  // namespace exl3
