// Layer on a few dozen to a few hundred rows (takes the lower end of the rows > 16 ladder of
// ponyexl3/mlx/exl3_linear.py:137-161): the decode still costs more than the product, so every
// weight is decoded once per up to 128 rows and goes from registers into 32x32x16 matrix
// instructions (see exl3_rows.hpp for the contraction).
//
// Workgroup = one 128-column group (one block of the output Hadamard) x one row block of 32 MR
// rows x one range of the reduction; its waves are two 64-column strips x NKS (four or two) k-slices
// of a 32 NKS deep step. A whole reduction ends with the output transform
// (ponyexl3/ref/forward.py:41-45) on the matrix pipe; ranges write fp32 partial rows that
// the output transform kernel adds in range order.
//
// What bounds it: issue of the decode, and the matrix pipe next to it. 333 rows of 17408 -> 5120
// (K = 4): VALU issue 49 % and matrix pipe 39 % of the SIMD cycles, which overlap only in part,
// 30 % of the wave time in waits and barriers; the layer 88 us where the GEMM takes 108.
// Half of a quad between two matrix instructions, rather than a whole quad between pairs of
// them, and direct loads spread the same way gave 5 %.
//
// x is already rotated: fp16 [rows][n_sub][in].
#include "exl3_device.hpp"
#include "exl3_host.hpp"
#include "exl3_rows.hpp"

#pragma clang fp contract(off)

namespace exl3 {

constexpr int kLinRowsLd = 128 + 8;  // halfs: 16-byte reads of 16 tile rows hit all banks

struct LinRowsArgs {
    const uint32_t* trellis;
    const half_t* xh;
    const half_t* svh;
    const half_t* bias;
    half_t* y;
    float* partial;
    const int* group_sub;  // rotation of each column group, or NULL
    size_t ldx, sub_stride;
    int rows, block_rows, n_row_blocks, n_units, n_splits, steps_per_split, in_steps, out_tiles, xcd_chunk;
};

// Sums of the four k-slices of a strip. On return the wave of slice ks holds column tile pair
// cs = ks >> 1 and, of each of its 32-row blocks, accumulators 8 (ks & 1) .. + 7 of sixteen:
// two exchanges of half of what a wave holds, every wave busy in both.
template <int MR>
__device__ __forceinline__ void rows_add_slices4(float16_t (&acc)[MR][2], float4_t* ex, int wave, int lane,
                                                 float (&sum)[MR][8]) {
    const bool upper = wave & 2, odd = wave & 1;
#pragma unroll
    for (int mr = 0; mr < MR; mr++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float4_t v;
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] = upper ? acc[mr][0][4 * i + c] : acc[mr][1][4 * i + c];
            ex[((wave ^ 2) * MR * 4 + mr * 4 + i) * 64 + lane] = v;
        }
    __syncthreads();
    float half_sum[MR][16];
#pragma unroll
    for (int mr = 0; mr < MR; mr++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float4_t v = ex[(wave * MR * 4 + mr * 4 + i) * 64 + lane];
#pragma unroll
            for (int c = 0; c < 4; c++)
                half_sum[mr][4 * i + c] = __fadd_rn(upper ? acc[mr][1][4 * i + c] : acc[mr][0][4 * i + c], v[c]);
        }
    __syncthreads();
#pragma unroll
    for (int mr = 0; mr < MR; mr++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            float4_t v;
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] = odd ? half_sum[mr][4 * i + c] : half_sum[mr][8 + 4 * i + c];
            ex[((wave ^ 1) * MR * 2 + mr * 2 + i) * 64 + lane] = v;
        }
    __syncthreads();
#pragma unroll
    for (int mr = 0; mr < MR; mr++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float4_t v = ex[(wave * MR * 2 + mr * 2 + i) * 64 + lane];
#pragma unroll
            for (int c = 0; c < 4; c++)
                sum[mr][4 * i + c] = __fadd_rn(odd ? half_sum[mr][8 + 4 * i + c] : half_sum[mr][4 * i + c], v[c]);
        }
    __syncthreads();
}

// Workgroups are dealt to the eight XCDs by index: the row blocks of one (column group, range)
// unit u land on one XCD, whose L2 then reads their trellis words once. Whole units in turn (xcd_chunk = 0) can leave one
// XCD with more workgroups than another; else each gets xcd_chunk, an eighth of them, neighbours, so that the row blocks of seven units at most
// lie across a border, and units of one range are neighbours too. See rows_deal_evenly(). Each has its own way to the unit: one for both made the
// kernel of short layers up to 7 % slower that are not dealt evenly (27 rows of 4992 -> 28672, MCG at K = 2, 33.3 and 36.5 us).
// Up to 32 rows three workgroups fit on a CU by their LDS, and the register bound keeps them to that: 87 registers in place of 72 at K = 4 made
// it two (17 rows of 4736 -> 22400 32.8 and 34.0 us).
template <int K, int CB, int MR, int NKS>
__global__ __launch_bounds__(128 * NKS, MR == 1 ? 6 : MR == 2 ? 4 : NKS == 2 && MR == 3 ? 3 : 2) void linear_rows_kernel(LinRowsArgs p) {
    using T = RowsTile<MR, NKS>;
    constexpr int LPW = T::FILLS / (2 * NKS);
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int g, split, rb;
    if (p.xcd_chunk) {
        const unsigned id = (blockIdx.x >> 3) + (blockIdx.x & 7) * p.xcd_chunk;
        const int u = id / (unsigned)p.n_row_blocks, n_groups = p.out_tiles >> 3;
        rb = id % (unsigned)p.n_row_blocks;
        if (u >= p.n_units) return;
        split = u / n_groups;
        g = u % n_groups;
    } else {
        const int set = blockIdx.x / (8 * p.n_row_blocks), in_set = blockIdx.x % (8 * p.n_row_blocks);
        const int u = set * 8 + (in_set & 7);
        rb = in_set >> 3;
        if (u >= p.n_units) return;
        g = u / p.n_splits;
        split = u % p.n_splits;
    }
    const int k0 = split * p.steps_per_split;
    const int nsteps = min(p.steps_per_split, p.in_steps - k0);
    const int m0 = rb * p.block_rows;
    const int valid = min(p.block_rows, p.rows - m0);

    const int cq = wave / NKS, ks = wave % NKS;
    const size_t row_words = (size_t)p.out_tiles * (8 * K);
    const uint32_t* w = p.trellis + ((size_t)k0 * 8 + 2 * ks) * row_words + (size_t)(g * 8 + cq * 4) * (8 * K);
    const half_t* x = p.xh + (size_t)m0 * p.ldx + (size_t)k0 * 128;
    if (p.group_sub) x += (size_t)p.group_sub[g] * p.sub_stride;
    half_t* stages = reinterpret_cast<half_t*>(lds);
    uint32_t a_off[LPW];
#pragma unroll
    for (int i = 0; i < LPW; i++) a_off[i] = rows_fill_offset<MR, NKS>(wave * LPW + i, lane, valid - 1, p.ldx);
    float16_t acc[MR][2];
    uint32_t* words = reinterpret_cast<uint32_t*>(stages + 3 * T::STAGE) + wave * RowsWords<K>::STAGE;
    rows_main<K, CB, MR, NKS, LPW>(w, row_words, 2 * NKS * row_words, reinterpret_cast<const char*>(x), a_off, true,
                                   lds_byte_address(stages) + wave * LPW * 1024, stages,
                                   rows_read_base<MR, NKS>(ks, lane), words, 2 * NKS * RowsWords<K>::STAGE,
                                   nsteps * (4 / NKS), lane, acc);
    // lane: row lane & 31 of each 32-row block, columns col + 16 i + 0..3, i < NI
    constexpr int NI = 8 / NKS;
    std::conditional_t<NKS == 4, float[MR][8], float16_t[MR]> sum;
    if constexpr (NKS == 4) rows_add_slices4<MR>(acc, reinterpret_cast<float4_t*>(lds), wave, lane, sum);
    else rows_add_slices2<MR>(acc, reinterpret_cast<float4_t*>(lds), wave, lane, sum);
    const int col = cq * 64 + (NKS == 4 ? 32 * (ks & 1) + 8 * (ks >> 1) : 8 * ks) + 4 * (lane >> 5);
    const size_t n_out = (size_t)p.out_tiles * 16;
    if (p.n_splits > 1) {
        float* dst = p.partial + ((size_t)split * p.rows + m0) * n_out + (size_t)g * 128 + col;
#pragma unroll
        for (int mr = 0; mr < MR; mr++) {
            const int r = mr * 32 + (lane & 31);
            if (r < valid) {
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    float4_t v;
#pragma unroll
                    for (int c = 0; c < 4; c++) v[c] = sum[mr][4 * i + c];
                    *reinterpret_cast<float4_t*>(dst + (size_t)r * n_out + 16 * i) = v;
                }
            }
        }
        return;
    }
    // Scales of the output transform: of the lane's columns, which are the same in all row tiles of a wave. Requested
    // in front of the barrier, and eight as one load where the vector allows it: as eight loads of two bytes for every row tile behind
    // it they were up to a tenth of a layer. Us, before -> now: 100 rows of 4096 -> 24576 with bias 45.3 -> 41.1, 40 of
    // 1536 -> 17408 19.0 -> 17.2, 306 of 2944 -> 11776 (K = 6) 57.4 -> 54.4, 700 of 2048 -> 6144 48.4 -> 48.4. (In front of the exchanges, and with
    // it on the way of the ranges too, these took 41.3, 17.6 and 54.2, and layers of ranges 1 % more than without.)
    static_assert(2 * NKS % 4 == 0);
    const int fr = lane & 15, q = lane >> 4, part = wave & 3, c0 = g * 128 + part * 32 + q * 8;
    half8_t sv, bv;
    auto eight = [](const half_t* v) {
        if ((reinterpret_cast<uintptr_t>(v) & 15) == 0) return *reinterpret_cast<const half8_t*>(v);  // (the same for all lanes)
        half8_t r;
#pragma unroll
        for (int c = 0; c < 8; c++) r[c] = v[c];
        return r;
    };
    if (p.svh) sv = eight(p.svh + c0);
    if (p.bias) bv = eight(p.bias + c0);
    half_t* tile = reinterpret_cast<half_t*>(lds);  // [BM][kLinRowsLd]
#pragma unroll
    for (int mr = 0; mr < MR; mr++)
#pragma unroll
        for (int i = 0; i < NI; i++) {
            half4_t o;
#pragma unroll
            for (int c = 0; c < 4; c++) o[c] = (half_t)sum[mr][4 * i + c];
            *reinterpret_cast<half4_t*>(tile + (mr * 32 + (lane & 31)) * kLinRowsLd + col + 16 * i) = o;
        }
    __syncthreads();
    // output transform: 2 MR 16-row tiles x four 32-column parts
    const HadamardColumns had(lane);
#pragma unroll
    for (int j = 0; j < 4 * MR / NKS; j++) {
        const int rt = (wave + 2 * NKS * j) >> 2;
        const half_t* yrow = tile + (rt * 16 + fr) * kLinRowsLd + q * 8;
        float4_t t[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        static_for<0, 4>([&](auto k) {
            const half8_t yv = *reinterpret_cast<const half8_t*>(yrow + k.value * 32);
            t[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(had.template get_part<0, k.value>(part), yv, t[0], 0, 0, 0);
            t[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(had.template get_part<1, k.value>(part), yv, t[1], 0, 0, 0);
        });
        const int r = rt * 16 + fr;
        if (r >= valid) continue;
        half8_t o;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            float v = __fmul_rn(t[c >> 2][c & 3], kHadNorm);
            if (p.svh) v = __fmul_rn(v, (float)sv[c]);
            o[c] = (half_t)v;
            if (p.bias) o[c] = o[c] + bv[c];
        }
        half_t* dst = p.y + (size_t)(m0 + r) * n_out + c0;
        *reinterpret_cast<half4_t*>(dst) = half4_t{o[0], o[1], o[2], o[3]};
        *reinterpret_cast<half4_t*>(dst + 4) = half4_t{o[4], o[5], o[6], o[7]};
    }
}

// Microseconds of one 128-deep step of a workgroup, measured at 16..333 rows of 5120 x 10240,
// 17408 x 5120, 5120 x 34816 (K = 4): a CU holds two workgroups of up to 64 rows or one of more.
// Only the number of ranges is chosen by it, the same at every K: pricing the one workgroup that a
// CU holds at 33..64 rows from K = 6 on changed no choice among 1666 layers.
static double rows_step_us(int mr, bool pair) {
    if (mr == 1) return pair ? 1.1 : 0.70;
    if (mr == 2) return pair ? 1.27 : 0.73;
    return mr == 3 ? 0.92 : 1.02;
}
constexpr double kRowsFillSteps = 5;      // pipeline fill and reduction of a workgroup
constexpr double kRowsPostUs = 3;         // launch of the pass that adds the ranges
constexpr double kRowsPartialRate = 8e6;  // bytes of partial rows written and read back per us

LinRowsPlan plan_linear_rows(int rows, int in_tiles, int n_groups) {
    LinRowsPlan p{};
    p.n_row_blocks = (rows + 127) / 128;
    p.block_rows = (rows + p.n_row_blocks - 1) / p.n_row_blocks;
    p.mr = (p.block_rows + 31) / 32;
    const int steps = in_tiles / 8;
    p.n_splits = 1;
    p.steps_per_split = steps;
    double best = 1e30;
    for (int s = 1; s <= 16 && (s == 1 || steps / s >= 2); s++) {
        const int per = (steps + s - 1) / s;
        if ((steps + per - 1) / per != s) continue;  // some range would be empty
        const long long n = (long long)p.n_row_blocks * n_groups * s;
        double us;  // per step of all workgroups
        if (p.mr <= 2)
            us = n <= 256 ? rows_step_us(p.mr, false)
                          : rows_step_us(p.mr, true) * (n <= 512 ? 1.0 : (double)n / 512 + 0.15);
        else
            us = rows_step_us(p.mr, false) * (double)((n + 255) / 256);
        us *= per + kRowsFillSteps;
        if (s > 1) us += kRowsPostUs + (double)s * rows * n_groups * 128 * 8 / kRowsPartialRate;
        if (us < best) {
            best = us;
            p.n_splits = s;
            p.steps_per_split = per;
        }
    }
    return p;
}

// Workgroups of four waves (two k-slices) instead of eight, where there are more of eight than the
// chip holds at once: with half the registers and LDS to a workgroup a CU holds four of them up to 64
// rows (three from K = 6 on), three (two from K = 6 on) up to 96, two above, where it held one of
// eight waves from 65 rows on or at K = 6, two else: 12 waves where there were 8, and the last round is
// of smaller pieces. 70 layers of 46 to 994 rows beyond that line, without the rotation: 18 % less at
// 77 rows of 5120 -> 34816 (80.8 -> 66.1 us), 21 % at 64 rows with K = 6 (77.5 -> 60.9), 15 % at 700
// rows of 2048 -> 6144 (50.9 -> 43.1), 11 % at the median, more (0.3 to 3 %) in three; below it
// mostly slower (256 rows of 5120 -> 10240 46.7 and 58.1). Up to 32 rows a CU holds three of eight
// waves, and the line is beyond the layers measured.
static int rows_per_cu(int mr, int nks, int K) {
    const int lds = 3 * (mr * 32 * nks * 32 * 2 + 2 * nks * 64 * K * 4), fit = (160 << 10) / lds;
    const int waves = mr <= 2 ? 16 : nks == 2 && mr == 3 ? 12 : 8;  // of a CU, by registers
    return std::min(fit, waves / (2 * nks));
}
static long long rows_workgroups(const LinRowsPlan& p, int n_groups) {
    return (long long)p.n_row_blocks * n_groups * p.n_splits;
}
static bool rows_narrow(const LinRowsPlan& p, int n_groups, int K) {
    return p.mr >= 2 && rows_workgroups(p, n_groups) > 256 * rows_per_cu(p.mr, 4, K);
}

// Whether the workgroups are dealt to the XCDs one by one and not in whole units: where an XCD gets more of them than its 32 CUs hold
// at once, and fewer that way (12 row blocks of 19 units: 36 on three XCDs, 24 on the others, one to a CU; evenly 29). Layers,
// whole units -> evenly, us: 514 rows of 13184 -> 6272 (K = 6) 206 -> 126, 788 of 6912 -> 1536 62.5 -> 40.7, 1309 of 2688 -> 2176
// 59.5 -> 35.6. Of 700 layers of 33 to 2048 rows 37 in workgroups of eight waves take 33 % less that way, 167 of four waves 4 %. Where all are resident at once whole units, which
// spread neighbouring trellis words over the XCDs, are as good or better (224 rows of 4992 -> 3072 28.6 and 29.9,
// 333 of 17408 -> 5120 92.3 and 93.2, 300 of 5120 -> 8192 48.3 and 48.7).
static bool rows_deal_evenly(const LinRowsPlan& p, int n_groups, int K) {
    const long long units = (long long)n_groups * p.n_splits, most = (units + 7) / 8 * p.n_row_blocks;
    return most > 32 * rows_per_cu(p.mr, rows_narrow(p, n_groups, K) ? 2 : 4, K) && most > (units * p.n_row_blocks + 7) / 8;
}

// Time of a plan in workgroups of four waves, fitted to the same layers (4 % root mean square): rounds of as many as the chip holds, a last one that costs between its share
// and that of its fullest CU.
static double rows_narrow_estimate_us(const LinRowsPlan& p, int n_groups, int K, int cb) {
    static const double step[3] = {0.615, 0.695, 0.817}, mul1[3] = {1.036, 1.149, 1.075};
    const int m = p.mr - 2, per_cu = rows_per_cu(p.mr, 2, K);
    const long long n = rows_workgroups(p, n_groups), full = n / (256 * per_cu), rest = n % (256 * per_cu);
    double load = full * (per_cu + 0.54);
    if (rest) load += 0.66 * (double)((rest + 255) / 256) + 0.34 * (double)rest / 256 + 0.54;
    return step[m] * (p.steps_per_split + 5) * load * (K > 4 ? 1 + 0.013 * (K - 4) : 1.0) *
               (cb == CB_MUL1 ? mul1[m] : 1.0) + 4;
}

// Estimate of a plan's time for the choice between this kernel and the prefill GEMM, without the
// input rotation. Alone on its CU, two to a CU, and in several rounds a workgroup's 128-deep step
// takes: {65..96, 97..128 rows} 0.915 and 1.08 us alone, 0.93 and 1.19 in rounds; up to 64 rows
// 0.765 alone, 1.40 for two, and 0.85 in rounds where LDS holds one (K = 6 and more: three stages
// of activations and trellis words). Bit windows take more instructions from K = 5 on. MUL1's factors, here, above and in
// gemm_estimate_us(), are those of a decode of 5.5 instructions a weight in place of decode_mul1_pair()'s 2.5: see linear_rows_applies().
static double rows_estimate_us(const LinRowsPlan& p, int rows, int n_groups, int K, int cb) {
    static const double alone[3] = {0.765, 0.915, 1.08}, rounds[3] = {0.85, 0.93, 1.19}, mul1[3] = {1.28, 1.21, 1.12};
    const int m = p.mr <= 2 ? 0 : p.mr - 2;
    const long long n = rows_workgroups(p, n_groups);
    const double split_us =
        p.n_splits > 1 ? kRowsPostUs + (double)p.n_splits * rows * n_groups * 128 * 8 / kRowsPartialRate : 0;
    if (rows_narrow(p, n_groups, K)) return rows_narrow_estimate_us(p, n_groups, K, cb) + split_us;
    const size_t lds = 3 * ((size_t)p.mr * 32 * 128 * 2 + (size_t)8 * 64 * K * 4);
    double us;
    if (n <= 256) us = alone[m];
    else if (p.mr <= 2 && 2 * lds <= (size_t)160 << 10) us = 1.40 * (n <= 512 ? 1.0 : (double)n / 512 + 0.15);
    else us = rounds[m] * (double)((n + 255) / 256);
    us *= (p.steps_per_split + kRowsFillSteps) * (K > 4 ? 1 + 0.014 * (K - 4) : 1.0) * (cb == CB_MUL1 ? mul1[m] : 1.0);
    return us + split_us;
}

// Whether the layer takes this kernel rather than the prefill GEMM, which has larger tiles (256
// columns and up to 256 rows). Both estimates were fitted to the choice over 2816 layers of 40 to
// 1024 rows (in 1024..17408, out 1024..65536, K = 2..8, all codebooks), before MUL1 was decoded in pairs and before this kernel's shorter
// epilogue and even dealing: as they were then the layer was slower than
// through the GEMM by more than 3 % in seven of them, 8 % at most, and 0.5 % slower than the
// better of the two on average. As they are now the line errs to the GEMM: of 129 MUL1 layers drawn from 33 to 1024 rows ten take more than
// 5 % more than through this kernel, 1.1 % on average (GEMM and this kernel, us: 405 rows of 1792 -> 8960 45.2 and 32.4, 200 of 4096 -> 24576
// 75.8 and 67.1, 384 of 5120 -> 34816 at K = 2 187 and 170), of 65 3INST and MCG layers six, 1.3 % (830 of 1152 -> 22528 at K = 8 89.9 and 69.6);
// none that comes here takes more than through the GEMM. Workgroups of four waves have lines of their own: over 140 layers that
// take them (33 to 994 rows), where the line of the eight-wave estimate lost 1 % (96 rows), 3 % (128 rows,
// and MUL1 from 65 on), 5 % (64 rows, K <= 5) and 14 % (64 rows, K >= 6) to the better of the two, these
// lost 0.2, 1.9, 0.3, 0.1 and 3 %, and no layer went to the slower one that did not before. Up to 64
// rows the GEMM's estimate is 11 % low, and with K <= 5 it was faster in one of 17 layers, by 2 %.
// Measured (layer, GEMM and this kernel, us): 5120 -> 10240 at 77 rows 41.1 and 28.8; 17408 -> 5120 (K = 5) at 333 rows 115 and 97; 5120 -> 34816 at 64 rows 63.7
// and 59.3 at K = 4, but 69.0 and 73.0 at K = 6.
bool linear_rows_applies(int rows, int in_tiles, int out_tiles, int K, int cb) {
    static const int max_rows = env_int("EXL3_LINEAR_ROWS_MAX_ROWS", kLinearRowsMaxRows, 0, kLinearRowsMaxRows);
    // fewer than four 128-deep steps do not fill the three stages of the pipeline
    if (rows < 1 || rows > max_rows || in_tiles < 32 || in_tiles % 8 || out_tiles < 8 || out_tiles % 8) return false;
    if (rows <= kLinearMidMaxRows) return true;
    const LinRowsPlan p = plan_linear_rows(rows, in_tiles, out_tiles / 8);
    const double us = rows_estimate_us(p, rows, out_tiles / 8, K, cb), gemm_us = gemm_estimate_us(rows, in_tiles, out_tiles, K, cb);
    if (!rows_narrow(p, out_tiles / 8, K)) return us < 0.95 * gemm_us;
    if (p.mr == 2) return K <= 5 || us < 1.05 * gemm_us;
    return us < (cb == CB_MUL1 ? 0.92 : p.mr == 3 ? 1.0 : 0.9) * gemm_us;
}

// Whether a layer of more rows than kLinearRowsMaxRows, which the prefill GEMM takes, goes to this kernel all the same, where its
// partial rows fit what the call's workspace holds for the GEMM. Layers too small to fill the GEMM's 256 x 256 tiles, or with few
// steps to a tile. The estimates are those for 3INST, which was fitted up to 1024 rows; past them
//  * reductions of 24 steps and more take longer than estimated the more rows there are (every XCD reads all of them: 1.0 times at 1300
//    rows, 1.2 at 2000), and the GEMM, whose pieces of such a reduction are long ones, is as fast as estimated;
//  * ranges in workgroups of four waves were 1 % slower than the GEMM on average, some by 14 % (50 layers of 3INST and MCG);
//  * the GEMM's estimate is low for MUL1, high from 150 us on and, below K = 4, where both are those of K = 4, 4 % high.
// 609 layers that the estimates alone would send here (in 1024..17408, out 1024..34816, K = 2..8, all codebooks), the two kernels in turn on one
// GPU: 40 of them are more than 2 % slower than through the GEMM, by up to 14 %. Of the 432 left two are, by 2.3 %; what the others gained
// is 1.1 % of the whole.
// GEMM -> this kernel, us: 1167 rows of 1024 -> 3072 38.1 -> 22.1, 1388 of 10880 -> 2944 143 -> 114, 1118 of 3456 -> 6656 98.8 -> 74.2,
// 1659 of 7552 -> 2176 89.1 -> 78.3; beyond the line 1097 of 16512 -> 2048 (K = 7) 117 and 136, 1907 of 12928 -> 1792 127 and 135,
// 2014 of 6656 -> 3584 127 and 136, 1257 of 13568 -> 1920 (K = 7) 105 and 117.
bool linear_rows_long_applies(int rows, int in_tiles, int out_tiles, int K, int cb) {
    static const int max_rows = env_int("EXL3_LINEAR_ROWS_MAX_ROWS", kLinearRowsMaxRows, 0, kLinearRowsMaxRows);
    if (rows <= kLinearRowsMaxRows || rows > kLinearRowsLongMaxRows || max_rows < kLinearRowsMaxRows || in_tiles < 32 ||
        in_tiles % 8 || out_tiles < 8 || out_tiles % 8 ||
        linear_rows_partial_bytes(rows, in_tiles, out_tiles / 8) > (size_t)rows * out_tiles * 32 + gemm_workspace_bytes(rows, in_tiles, out_tiles))
        return false;
    const LinRowsPlan p = plan_linear_rows(rows, in_tiles, out_tiles / 8);
    const double gemm_us = gemm_estimate_us(rows, in_tiles, out_tiles, K, CB_3INST);
    double us = rows_estimate_us(p, rows, out_tiles / 8, K, CB_3INST) * (K < 4 ? 1.04 : 1.0);
    const bool mul1 = cb == CB_MUL1;
    if (us >= (gemm_us >= 150 ? 0.94 : mul1 ? 1.05 : 1.02) * gemm_us) return false;
    if (!mul1 && p.n_splits > 1 && rows_narrow(p, out_tiles / 8, K)) return false;
    if (p.steps_per_split < 24) return true;
    if (rows > 1300) us *= 1 + 0.2 * (rows - 1300) / 700;
    return us < (mul1 ? 1.04 : 0.96) * gemm_us;
}

// Up to 16 rows the rows kernel spends twice the matrix work and half the publishing of the medium-batch kernel, and
// which one is faster hangs on how evenly each fills 256 CUs: the rows kernel with whole reductions as one
// workgroup for every CU or two, nearly, or with few steps; with ranges where nearly two workgroups to a CU have 10 to 20 steps each
// (30 below K = 4, where the decode is shorter) and the medium-batch kernel's workgroups leave 7 % and more
// of their last round empty. Layer, medium-batch -> rows kernel, us: 15 rows of 1536 -> 64896 26.6 -> 21.7, 15 of 1024 -> 61568
// 22.5 -> 17.3, 15 of 2560 -> 29440 24.3 -> 20.1, 14 of 9216 -> 5248 22.3 -> 19.0, 12 of 12288 -> 10368 34.6 -> 29.4. Beyond the lines: 11 rows of
// 2560 -> 43008 (336 workgroups of 20 steps) 35.8 and 40.7, 10 of 8192 -> 21632 (507 of 22) 34.8 and 36.5, 14 of 4096 -> 19072 (447) 22.8
// and 24.0, 12 of 7168 -> 12288 (768 medium-batch workgroups, three to a CU) 22.8
// and 24.9. Of 225 layers of 9 to 16 rows on both sides of the lines the 71 that changed from the medium-batch kernel take 8.3 %
// less, one of them 1.7 % more (12 rows of 1024 -> 49152 21.6 and 22.0); the others, same kernel, repeat within 4 %.
bool linear_rows_before_mid(int rows, int K, int in_tiles, int out_tiles) {
    if (rows > 16 || K >= 5 || in_tiles >= 2 * out_tiles) return true;
    const int n_groups = out_tiles / 8;
    const LinRowsPlan p = plan_linear_rows(rows, in_tiles, n_groups);
    const long long n = rows_workgroups(p, n_groups);
    if (n > 512) return false;
    if (p.n_splits == 1) return n >= 430 || (n >= 340 && p.steps_per_split <= 14) || (n <= 256 && (n >= 200 || p.steps_per_split <= 16));
    const int mid = n_groups * plan_linear_mid(rows, in_tiles, n_groups).n_splits, rounds = (mid + 255) / 256;
    return n >= 450 && p.steps_per_split >= 10 && p.steps_per_split <= (K == 4 ? 20 : 30) && mid < 0.93 * 256 * rounds;
}

bool linear_rows_ever_applies(int rows, int in_tiles, int out_tiles) {
    for (int cb : {(int)CB_3INST, (int)CB_MUL1})
        for (int K = 8; K >= 4; K--)  // (below it the estimates are those of K = 4)
            if (linear_rows_applies(rows, in_tiles, out_tiles, K, cb)) return true;
    return false;
}

size_t linear_rows_partial_bytes(int rows, int in_tiles, int n_groups) {
    const LinRowsPlan p = plan_linear_rows(rows, in_tiles, n_groups);
    return p.n_splits > 1 ? (size_t)p.n_splits * rows * n_groups * 128 * sizeof(float) : 0;
}

LinRowsShape linear_rows_shape(int rows, int in_tiles, int n_groups, int K) {
    const LinRowsPlan p = plan_linear_rows(rows, in_tiles, n_groups);
    return {p.n_row_blocks, p.n_splits, rows_narrow(p, n_groups, K) ? 4 : 8, rows_deal_evenly(p, n_groups, K)};
}

int launch_linear_rows(const uint16_t* xh, int rows, size_t ldx, size_t sub_stride, const uint16_t* trellis,
                       int in_tiles, int out_tiles, int K, int cb, const int32_t* group_sub,
                       const uint16_t* svh, const uint16_t* bias, uint16_t* y, float* partial, hipStream_t stream) {
    if (int rc = check_k_cb(K, cb)) return rc;
    if (!xh || !trellis || !y) return EXL3_E_NULL_POINTER;
    if (rows < 1 || in_tiles < 8 || in_tiles % 8 || out_tiles < 8 || out_tiles % 8 || ldx % 8 ||
        ldx < (size_t)in_tiles * 16 || ldx * 2 * 128 >= (1ull << 31))  // 32-bit row offsets inside a block
        return EXL3_E_BAD_SHAPE;
    if ((reinterpret_cast<uintptr_t>(xh) & 15) || (reinterpret_cast<uintptr_t>(trellis) & 15) ||
        (reinterpret_cast<uintptr_t>(y) & 7))
        return EXL3_E_BAD_SHAPE;
    const int n_groups = out_tiles / 8;
    const LinRowsPlan plan = plan_linear_rows(rows, in_tiles, n_groups);
    if (plan.n_splits > 1 && (!partial || (reinterpret_cast<uintptr_t>(partial) & 15))) return EXL3_E_WORKSPACE;
    const long long units = (long long)n_groups * plan.n_splits;
    const long long chunk = rows_deal_evenly(plan, n_groups, K) ? (units * plan.n_row_blocks + 7) / 8 : 0;
    const long long grid = chunk ? 8 * chunk : (units + 7) / 8 * 8 * plan.n_row_blocks;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    auto H_ = [](const uint16_t* q) { return reinterpret_cast<const half_t*>(q); };
    const LinRowsArgs a{reinterpret_cast<const uint32_t*>(trellis), H_(xh), H_(svh), H_(bias),
                        reinterpret_cast<half_t*>(y), partial, group_sub, ldx, sub_stride, rows,
                        plan.block_rows, plan.n_row_blocks, (int)units, plan.n_splits, plan.steps_per_split,
                        in_tiles / 8, out_tiles, (int)chunk};
    const int rc = dispatch_k_cb(K, cb, [&](auto k, auto c) {
        auto go = [&](auto mrc, auto nks) {
            constexpr int MR = mrc.value, NKS = nks.value;
            constexpr size_t stages = (size_t)3 * (RowsTile<MR, NKS>::STAGE * 2 + 2 * NKS * RowsWords<k.value>::STAGE * 4),
                             exchange = (size_t)2 * NKS * MR * 4 * 64 * 16;
            constexpr size_t bytes = stages > exchange ? stages : exchange;
            static_assert(bytes >= (size_t)32 * MR * kLinRowsLd * 2, "the fp16 tile fits");
            auto kernel = linear_rows_kernel<k.value, c.value, MR, NKS>;
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
                return (int)EXL3_E_LAUNCH;
            kernel<<<dim3((unsigned)grid), dim3(128 * NKS), bytes, stream>>>(a);
            return launch_status();
        };
        using N2 = std::integral_constant<int, 2>;
        using N4 = std::integral_constant<int, 4>;
        const bool narrow = rows_narrow(plan, n_groups, k.value);
        switch (plan.mr) {
            case 1: return go(std::integral_constant<int, 1>{}, N4{});
            case 2: return narrow ? go(N2{}, N2{}) : go(N2{}, N4{});
            case 3: return narrow ? go(std::integral_constant<int, 3>{}, N2{}) : go(std::integral_constant<int, 3>{}, N4{});
            default: return narrow ? go(N4{}, N2{}) : go(N4{}, N4{});
        }
    });
    if (rc != EXL3_OK || plan.n_splits == 1) return rc;
    return launch_had_post(partial, 1, plan.n_splits, (size_t)rows * out_tiles * 16, rows, out_tiles * 16, svh, bias,
                           y, stream);
}

}  // namespace exl3
