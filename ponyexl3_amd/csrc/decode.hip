// exl3_decode_full and its two layout variants: packed trellis -> fp16 W_inner,
// bit-exact with ponyexl3/ref/decode.py:32-81.
//
// Row-major (in, out) and expert-grouped (E, in, out_e): one wavefront decodes
// the 8 tiles (tk, tn0..tn0+7): its 64 lanes read 256*K contiguous bytes, each
// lane decodes 32 codewords in registers, the 16x128 block is transposed through
// LDS and written as 16-byte chunks (half a tile row each, so a tile can be
// steered to its expert's slab).
//
// Transposed (out, in): one wavefront decodes the 8 tiles (tk0..tk0+7, tn), so
// that each of the tile column's 16 output rows receives 128 contiguous halfs.
//
// exl3_public_weight: the same decode with both Hadamard transforms and scale vectors
// applied on the way out (public_weight_kernel).
#include "exl3_device.hpp"
#include "exl3_host.hpp"

namespace exl3 {

constexpr int kDecPad = 8;  // halfs of padding per staged row (keeps 16 B alignment)

template <int K, int CB>
__global__ __launch_bounds__(256) void decode_full_kernel(const uint32_t* __restrict__ trellis,
                                                          half_t* __restrict__ w_out, int in_tiles,
                                                          int out_tiles, int tn_offset,
                                                          int tn_count, int tiles_per_group) {
    __shared__ __attribute__((aligned(16))) half_t stage[4][16][128 + kDecPad];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int groups = (tn_count + 7) >> 3;
    const long long wid = (long long)blockIdx.x * 4 + wave;
    const bool active = wid < (long long)in_tiles * groups;
    const int g = active ? (int)(wid % groups) : 0;
    const int tk = active ? (int)(wid / groups) : 0;
    const int tile_local = g * 8 + (lane >> 3);
    const bool valid = active && tile_local < tn_count;
    // lanes of a tile past the slice re-read the last valid tile (never stored)
    const int tn = tn_offset + (valid ? tile_local : tn_count - 1);
    const uint32_t* p = trellis + ((size_t)tk * out_tiles + tn) * (8 * K) + (lane & 7) * K;
    uint32_t own[K];
#pragma unroll
    for (int i = 0; i < K; i++) own[i] = p[i];
    const LaneWords<K> lw = finish_lane_words<K>(own, lane);
    half2_t wp[16];
    decode_lane<K, CB>(lw, wp);
    const int c0 = (lane >> 3) * 16 + (lane & 7);
#pragma unroll
    for (int cs = 0; cs < 2; cs++)
#pragma unroll
        for (int j = 0; j < 8; j++) {
            stage[wave][2 * j][c0 + 8 * cs] = wp[8 * cs + j].x;
            stage[wave][2 * j + 1][c0 + 8 * cs] = wp[8 * cs + j].y;
        }
    __syncthreads();
    if (!active) return;
    // tiles_per_group == 0: one (in, 16*tn_count) matrix. Otherwise tile column t
    // goes to slab t / tiles_per_group, an (in, 16*tiles_per_group) matrix of its own.
    const int chunk = lane & 15;  // 8 halfs each; two chunks per tile
    const int t = g * 8 + (chunk >> 1);
    if (t >= tn_count) return;
    size_t ld = (size_t)tn_count * 16, col = (size_t)t * 16, slab = 0;
    if (tiles_per_group > 0) {
        ld = (size_t)tiles_per_group * 16;
        col = (size_t)(t % tiles_per_group) * 16;
        slab = (size_t)(t / tiles_per_group) * in_tiles * 16 * ld;
    }
#pragma unroll
    for (int pass = 0; pass < 4; pass++) {
        const int row = pass * 4 + (lane >> 4);
        const uint4_t v = *reinterpret_cast<const uint4_t*>(&stage[wave][row][chunk * 8]);
        *reinterpret_cast<uint4_t*>(w_out + slab + ((size_t)tk * 16 + row) * ld + col +
                                    (chunk & 1) * 8) = v;
    }
}

// W^T (16*tn_count, in): lanes 8t..8t+7 of a wave decode tile (tk0 + t, tn).
template <int K, int CB>
__global__ __launch_bounds__(256) void decode_full_t_kernel(const uint32_t* __restrict__ trellis,
                                                            half_t* __restrict__ w_out,
                                                            int in_tiles, int out_tiles,
                                                            int tn_offset, int tn_count) {
    __shared__ __attribute__((aligned(16))) half_t stage[4][16][128 + kDecPad];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int kgroups = (in_tiles + 7) >> 3;
    const long long wid = (long long)blockIdx.x * 4 + wave;
    const bool active = wid < (long long)tn_count * kgroups;
    const int kg = active ? (int)(wid % kgroups) : 0;
    const int tn_local = active ? (int)(wid / kgroups) : 0;
    const int tk_lane = kg * 8 + (lane >> 3);
    // lanes of a tile row past the matrix re-read the last tile row (never stored)
    const int tk = tk_lane < in_tiles ? tk_lane : in_tiles - 1;
    const uint32_t* p =
        trellis + ((size_t)tk * out_tiles + tn_offset + tn_local) * (8 * K) + (lane & 7) * K;
    uint32_t own[K];
#pragma unroll
    for (int i = 0; i < K; i++) own[i] = p[i];
    const LaneWords<K> lw = finish_lane_words<K>(own, lane);
    half2_t wp[16];
    decode_lane<K, CB>(lw, wp);
    // pair j of column u + 8*cs holds input rows 2j, 2j+1 of the tile: one 4-byte store
    const int u = lane & 7, r0 = (lane >> 3) * 16;
#pragma unroll
    for (int cs = 0; cs < 2; cs++)
#pragma unroll
        for (int j = 0; j < 8; j++)
            *reinterpret_cast<half2_t*>(&stage[wave][u + 8 * cs][r0 + 2 * j]) = wp[8 * cs + j];
    __syncthreads();
    if (!active) return;
    const size_t ld = (size_t)in_tiles * 16;
    const int chunk = lane & 15;
    if (kg * 8 + (chunk >> 1) >= in_tiles) return;
#pragma unroll
    for (int pass = 0; pass < 4; pass++) {
        const int c = pass * 4 + (lane >> 4);  // output row = column of the tile
        const uint4_t v = *reinterpret_cast<const uint4_t*>(&stage[wave][c][chunk * 8]);
        *reinterpret_cast<uint4_t*>(w_out + ((size_t)tn_local * 16 + c) * ld + (size_t)kg * 128 +
                                    chunk * 8) = v;
    }
}

// Public weight W_pub = diag(suh) . H . W_inner . H . diag(svh) of one 128 x 128 block per
// workgroup, in (in, out) or (T) transposed (out, in) order, with the runtime's cast points:
// the result of pushing an fp16 identity through rotation, GEMM and output transform
// (ponyexl3/mlx/native.py:49-70) without the identity. Row i of the rotated identity is
// q_i * sign(H[i][:]) with q_i = fp16(suh_i / sqrt(128)), so the GEMM is a Hadamard product
// over the rows of the block:
//   Y[i][n] = fp16(sum_j +-q_i W[j][n]),   Z[i][m] = fp16(sum_n +-Y[i][n] / sqrt(128) * svh_m)
// Both run on the matrix pipe (v_mfma_f32_16x16x32_f16, fp32 sums in the order of the
// prefill GEMM), the fragments of H made from sign words each lane holds. The decoded weights are
// operands of the first product without a trip through LDS: a wave takes 32 columns over all 128 rows, its
// loads put neighbouring pairs of tile rows on lane bits 4 and 5, and one exchange of 16-lane rows a
// register brings rows 0..7 and 8..15 of a tile into the lanes that the operand wants them in.
// For 5120 x 17408 at K = 4 VALU issue (decode, signs, conversions: 730 instructions a wave, and 108 of the matrix pipe) is busy for
// 82 % of the time that the CUs are, the matrix pipe for 41 %, and waves wait 25 % of theirs; a plain fill of the result would take
// 26 us. What is left are the phases of a workgroup, of which four share a CU (one 34 KiB LDS tile, 128 registers): decode and first
// product, second product, store, with three barriers between. The result goes out through LDS in 256-byte row pieces,
// non-temporal (nobody reads it soon).
// Measured, us, transposed: decoded weights through LDS (five barriers, scales loaded where they are used, a wait
// each) -> operands from registers, scales in front -> words of the next block requested ahead:
//   5120 x 17408 K = 2 / 4 / 8: 63.5 / 65.5 / 71.6 -> 56.3 / 56.5 / 63.1 -> 54.0 / 52.8 / 55.6,
//   not transposed K = 4 69.7 -> 58.5 -> 54.2; 2048 x 2048 7.4 -> 5.7 -> 5.8.
// On other GPUs of the kind 50.9 to 55 at K = 4 (4.1 to 4.4 TB/s of trellis and result). That is one layer again and again, whose words the last-level
// cache can keep. Twelve layers in turn, each one's words from memory, first -> last of these forms: 60 / 62 / 72 -> 48.5 / 53.7 / 57.5.
// The identity through the prefill kernels, the concatenation of its column stripes and the transposed copy took 1420.
//
// Workgroups that start together: 256 CUs of four. The one this many places on gets the place of this one, and as a
// multiple of eight on the same XCD, whose L2 then has its words.
constexpr unsigned kPubAhead = 1024;
constexpr int kPubLd = 128 + kDecPad;  // halfs per row: 16-byte reads of 16 rows hit all banks

// Signs of a fragment of H128 for rows / columns 16 nt + fr and k = 32 ks + 8 q + 0..7: entry
// (k, n) has sign parity(k & n), which splits into a part the lane knows (fr, q and the k
// inside the fragment), a part that needs nt & 1, and one that is the same for every lane
// (nt >> 1 and ks). get() is the fragment times `mag`, an fp16 value in both halves.
struct HadamardFragments {
    uint4_t base, odd;  // sign bits for nt even, nt odd
    __device__ __forceinline__ HadamardFragments(int lane) {
        const int fr = lane & 15, q = lane >> 4;
        const uint32_t flip = ((fr >> 3) & q & 1) ? 0x80008000u : 0u;
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t lo = __builtin_popcount(fr & 7 & (2 * i)) & 1;
            const uint32_t hi = __builtin_popcount(fr & 7 & (2 * i + 1)) & 1;
            w[i] = (lo << 15) ^ (hi << 31) ^ flip;
        }
        base = uint4_t{w[0], w[1], w[2], w[3]};
        odd = base ^ ((q >> 1) ? 0x80008000u : 0u);
    }
    template <int NT, int KS>
    __device__ __forceinline__ half8_t get(uint32_t mag) const {
        constexpr bool neg = (((NT >> 1) & KS & 1) ^ ((NT >> 2) & (KS >> 1) & 1)) != 0;
        return __builtin_bit_cast(half8_t, ((NT & 1) ? odd : base) ^ (neg ? mag ^ 0x80008000u : mag));
    }
};

template <int K, int CB, bool T>
__global__ __launch_bounds__(256, 4) void public_weight_kernel(
    const uint32_t* __restrict__ trellis, const half_t* __restrict__ suh,
    const half_t* __restrict__ svh, half_t* __restrict__ w_out, int out_tiles, int tn_offset,
    int blocks_fast, size_t ldw) {
    constexpr float kScale = 0.088388347648318440550f;  // 1/sqrt(128)
    __shared__ __attribute__((aligned(16))) half_t tile[128 * kPubLd];
    __shared__ __attribute__((aligned(16))) float sv_s[128];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int fr = lane & 15, q = lane >> 4;
    // consecutive workgroups write consecutive pieces of the same output rows
    const int fast = blockIdx.x % blocks_fast, slow = blockIdx.x / blocks_fast;
    const int bi = T ? fast : slow, bn = T ? slow : fast;

    // Wave w takes columns 32w .. 32w + 31, i.e. two tile columns (lane bit 3) of all eight tile rows: 4r + 2 (lane
    // bit 4) + (lane bit 5) in load r.
    uint32_t own[2][K];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const uint32_t* p = trellis +
                            ((size_t)(bi * 8 + 4 * r + (lane >> 3 & 2) + (lane >> 5)) * out_tiles + tn_offset + bn * 8 + 2 * wave +
                             (lane >> 3 & 1)) * (8 * K) + (lane & 7) * K;
#pragma unroll
        for (int i = 0; i < K; i++) own[r][i] = __builtin_nontemporal_load(p + i);
    }
    // one dword of each 128-byte line of the words of the block ahead
    uint32_t ahead = 0;
    {
        const unsigned nb = blockIdx.x + kPubAhead;
        const int nfast = nb % blocks_fast, nslow = nb / blocks_fast;
        const int ni = T ? nfast : nslow, nn = T ? nslow : nfast;
        constexpr int kLines = 2 * K;  // of a tile row
        if (nb < gridDim.x && lane < 2 * kLines)
            ahead = trellis[((size_t)(ni * 8 + 2 * wave + lane / kLines) * out_tiles + tn_offset + nn * 8) * (8 * K) +
                            lane % kLines * 32];
    }
    // scales: one branch and one wait each, in front of everything that needs them
    half_t su[8];
    if (suh) {
#pragma unroll
        for (int nt = 0; nt < 8; nt++) su[nt] = suh[bi * 128 + nt * 16 + fr];
    } else {
#pragma unroll
        for (int nt = 0; nt < 8; nt++) su[nt] = (half_t)1.0f;
    }
    if (threadIdx.x < 128) sv_s[threadIdx.x] = svh ? (float)svh[bn * 128 + threadIdx.x] : 1.0f;
    const HadamardFragments had(lane);

    // A lane has rows 0..7 and 8..15 of its tile; the exchange of 16-lane rows makes of the two tile rows that lane
    // bit 4 tells apart two operands of 32 rows, k = 8 q + t (column u + 8 cs of tile column lane >> 3 & 1 in
    // operand row lane & 15).
    half8_t w[4][2];  // [32-row step][cs]
    static_for<0, 2>([&](auto r) {
        const LaneWords<K> lw = finish_lane_words<K>(own[r.value], lane);
        half2_t wp[16];
        decode_lane<K, CB>(lw, wp);
#pragma unroll
        for (int cs = 0; cs < 2; cs++) {
            uint32_t a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                a[i] = half2_to_bits(wp[8 * cs + i]);
                b[i] = half2_to_bits(wp[8 * cs + 4 + i]);
            }
            // the exchange wants two wait states behind a VALU write of its registers; the compiler does not see
            // those of the asm in add_halves_pack2()
            asm("s_nop 1" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]));
            uint4_t lo, hi;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const auto x = __builtin_amdgcn_permlane16_swap(a[i], b[i], false, false);
                lo[i] = x[0];
                hi[i] = x[1];
            }
            w[2 * r.value][cs] = __builtin_bit_cast(half8_t, lo);
            w[2 * r.value + 1][cs] = __builtin_bit_cast(half8_t, hi);
        }
    });
    // Y^T[n][i] = sum_j W^T[n][j] H[j][i]: a lane gets four consecutive n of one i
    static_for<0, 8>([&](auto nt) {
        const uint32_t qi = half_to_bits((half_t)__fmul_rn((float)su[nt.value], kScale)) * 0x10001u;
        float4_t y[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        static_for<0, 4>([&](auto ks) {
            const half8_t h = had.template get<nt.value, ks.value>(qi);
#pragma unroll
            for (int cs = 0; cs < 2; cs++)
                y[cs] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[ks.value][cs], h, y[cs], 0, 0, 0);
        });
#pragma unroll
        for (int cs = 0; cs < 2; cs++) {
            half4_t o;
#pragma unroll
            for (int c = 0; c < 4; c++) o[c] = (half_t)y[cs][c];
            *reinterpret_cast<half4_t*>(tile + (nt.value * 16 + fr) * kPubLd + wave * 32 + (q >> 1) * 16 + cs * 8 + (q & 1) * 4) = o;
        }
    });
    asm volatile("" ::"v"(ahead));  // (its wait: long there)
    __syncthreads();

    // Z: a lane gets four consecutive i of one m (T) or four consecutive m of one i
    half8_t op[2][4];  // rows 32 wave .. + 31 of the tile, all 128 k
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
            op[rt][ks] = *reinterpret_cast<const half8_t*>(tile + (wave * 32 + rt * 16 + fr) * kPubLd + ks * 32 + q * 8);
    __syncthreads();
    float4_t acc[2][8];
    static_for<0, 4>([&](auto ks) {
        static_for<0, 8>([&](auto nt) {
            const half8_t h = had.template get<nt.value, ks.value>(0x3C003C00u);
#pragma unroll
            for (int rt = 0; rt < 2; rt++)
                acc[rt][nt.value] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    T ? op[rt][ks.value] : h, T ? h : op[rt][ks.value],
                    ks.value == 0 ? float4_t{0.f, 0.f, 0.f, 0.f} : acc[rt][nt.value], 0, 0, 0);
        });
    });
#pragma unroll
    for (int nt = 0; nt < 8; nt++) {
        float s[4];
#pragma unroll
        for (int c = 0; c < 4; c++) s[c] = sv_s[T ? nt * 16 + fr : nt * 16 + q * 4 + c];
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {
            half4_t o;
#pragma unroll
            for (int c = 0; c < 4; c++) o[c] = (half_t)__fmul_rn(__fmul_rn(acc[rt][nt][c], kScale), s[c]);
            half_t* dst = T ? tile + (nt * 16 + fr) * kPubLd + wave * 32 + rt * 16 + q * 4
                            : tile + (wave * 32 + rt * 16 + fr) * kPubLd + nt * 16 + q * 4;
            *reinterpret_cast<half4_t*>(dst) = o;
        }
    }
    __syncthreads();
    half_t* out = w_out + (size_t)(T ? bn : bi) * 128 * ldw + (size_t)(T ? bi : bn) * 128;
#pragma unroll
    for (int it = 0; it < 8; it++) {
        const int row = it * 16 + (threadIdx.x >> 4), c = (threadIdx.x & 15) * 8;
        __builtin_nontemporal_store(*reinterpret_cast<const uint4_t*>(tile + row * kPubLd + c),
                                    reinterpret_cast<uint4_t*>(out + (size_t)row * ldw + c));
    }
}

// Packed tiles -> their 256 16-bit codewords in kernel (stream) order
// (unpack_trellis, ponyexl3/ref/trellis.py:153-214). Lanes 8t..8t+7 of a wave own
// tile t of eight consecutive tiles; lane u extracts codewords 32u..32u+31 and
// writes them as 64 contiguous bytes.
template <int K>
__global__ __launch_bounds__(256) void unpack_trellis_kernel(const uint32_t* __restrict__ trellis,
                                                             uint16_t* __restrict__ codewords,
                                                             long long n_tiles) {
    const int lane = threadIdx.x & 63;
    const long long wid = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const long long tile_lane = wid * 8 + (lane >> 3);
    // lanes past the last tile re-read it (never stored)
    const long long tile = tile_lane < n_tiles ? tile_lane : n_tiles - 1;
    const uint32_t* p = trellis + tile * (8 * K) + (lane & 7) * K;
    uint32_t own[K];
#pragma unroll
    for (int i = 0; i < K; i++) own[i] = p[i];
    const LaneWords<K> lw = finish_lane_words<K>(own, lane);
    uint32_t packed[16];
    static_for<0, 16>([&](auto i) {
        packed[i.value] = lane_codeword<K, 2 * i.value>(lw) | (lane_codeword<K, 2 * i.value + 1>(lw) << 16);
    });
    if (tile_lane >= n_tiles) return;
    uint4_t* dst = reinterpret_cast<uint4_t*>(codewords + tile * 256 + (lane & 7) * 32);
#pragma unroll
    for (int i = 0; i < 4; i++)
        dst[i] = uint4_t{packed[4 * i], packed[4 * i + 1], packed[4 * i + 2], packed[4 * i + 3]};
}

// Shared argument checks and launch of the row-major / expert-grouped kernel.
static int launch_decode_full(const uint16_t* trellis, int in_tiles, int out_tiles, int K, int cb,
                              int tn_offset, int tn_count, int tiles_per_group, uint16_t* w_out,
                              void* stream) {
    if (int rc = check_k_cb(K, cb)) return rc;
    if (!trellis || !w_out) return EXL3_E_NULL_POINTER;
    if (in_tiles < 0 || out_tiles < 0 || tn_offset < 0 || tn_count < 0 ||
        tn_offset + tn_count > out_tiles)
        return EXL3_E_BAD_SHAPE;
    if (in_tiles == 0 || tn_count == 0) return EXL3_OK;
    if ((reinterpret_cast<uintptr_t>(w_out) & 15) || (reinterpret_cast<uintptr_t>(trellis) & 3))
        return EXL3_E_BAD_SHAPE;
    const long long waves = (long long)in_tiles * ((tn_count + 7) / 8);
    const long long grid = (waves + 3) / 4;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    return dispatch_k_cb(K, cb, [&](auto k, auto c) {
        decode_full_kernel<k.value, c.value><<<dim3((unsigned)grid), dim3(256), 0, as_stream(stream)>>>(
            reinterpret_cast<const uint32_t*>(trellis), reinterpret_cast<half_t*>(w_out), in_tiles,
            out_tiles, tn_offset, tn_count, tiles_per_group);
        return launch_status();
    });
}

}  // namespace exl3

EXL3_EXPORT int exl3_decode_full(const uint16_t* trellis, int in_tiles, int out_tiles, int K,
                                 int cb, int tn_offset, int tn_count, uint16_t* w_out,
                                 void* stream) {
    return exl3::launch_decode_full(trellis, in_tiles, out_tiles, K, cb, tn_offset, tn_count, 0,
                                    w_out, stream);
}

EXL3_EXPORT int exl3_decode_full_eg(const uint16_t* trellis, int in_tiles, int out_tiles, int K,
                                    int cb, int tiles_per_e, uint16_t* w_out, void* stream) {
    if (tiles_per_e < 1 || out_tiles < 0 || out_tiles % tiles_per_e) return EXL3_E_BAD_SHAPE;
    return exl3::launch_decode_full(trellis, in_tiles, out_tiles, K, cb, 0, out_tiles, tiles_per_e,
                                    w_out, stream);
}

EXL3_EXPORT int exl3_decode_full_t(const uint16_t* trellis, int in_tiles, int out_tiles, int K,
                                   int cb, int tn_offset, int tn_count, uint16_t* w_out_t,
                                   void* stream) {
    using namespace exl3;
    if (int rc = check_k_cb(K, cb)) return rc;
    if (!trellis || !w_out_t) return EXL3_E_NULL_POINTER;
    if (in_tiles < 0 || out_tiles < 0 || tn_offset < 0 || tn_count < 0 ||
        tn_offset + tn_count > out_tiles)
        return EXL3_E_BAD_SHAPE;
    if (in_tiles == 0 || tn_count == 0) return EXL3_OK;
    if ((reinterpret_cast<uintptr_t>(w_out_t) & 15) || (reinterpret_cast<uintptr_t>(trellis) & 3))
        return EXL3_E_BAD_SHAPE;
    const long long waves = (long long)tn_count * ((in_tiles + 7) / 8);
    const long long grid = (waves + 3) / 4;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    return dispatch_k_cb(K, cb, [&](auto k, auto c) {
        decode_full_t_kernel<k.value, c.value>
            <<<dim3((unsigned)grid), dim3(256), 0, as_stream(stream)>>>(
                reinterpret_cast<const uint32_t*>(trellis), reinterpret_cast<half_t*>(w_out_t),
                in_tiles, out_tiles, tn_offset, tn_count);
        return launch_status();
    });
}

EXL3_EXPORT int exl3_public_weight(const uint16_t* trellis, int in_tiles, int out_tiles, int K,
                                   int cb, const uint16_t* suh, const uint16_t* svh, int tn_offset,
                                   int tn_count, int transposed, uint16_t* w_out, void* stream) {
    using namespace exl3;
    if (int rc = check_k_cb(K, cb)) return rc;
    if (!trellis || !w_out) return EXL3_E_NULL_POINTER;
    if (in_tiles < 0 || out_tiles < 0 || tn_offset < 0 || tn_count < 0 || in_tiles % 8 ||
        tn_count % 8 || tn_offset + tn_count > out_tiles)
        return EXL3_E_BAD_SHAPE;
    if (in_tiles == 0 || tn_count == 0) return EXL3_OK;
    if ((reinterpret_cast<uintptr_t>(w_out) & 15) || (reinterpret_cast<uintptr_t>(trellis) & 3))
        return EXL3_E_BAD_SHAPE;
    const int blocks_in = in_tiles / 8, blocks_out = tn_count / 8;
    const long long grid = (long long)blocks_in * blocks_out;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    return dispatch_k_cb(K, cb, [&](auto k, auto c) {
        auto kernel = transposed ? public_weight_kernel<k.value, c.value, true>
                                 : public_weight_kernel<k.value, c.value, false>;
        kernel<<<dim3((unsigned)grid), dim3(256), 0, as_stream(stream)>>>(
            reinterpret_cast<const uint32_t*>(trellis), reinterpret_cast<const half_t*>(suh),
            reinterpret_cast<const half_t*>(svh), reinterpret_cast<half_t*>(w_out), out_tiles,
            tn_offset, transposed ? blocks_in : blocks_out,
            (size_t)(transposed ? in_tiles : tn_count) * 16);
        return launch_status();
    });
}

EXL3_EXPORT int exl3_unpack_trellis(const uint16_t* trellis, long long n_tiles, int K,
                                    uint16_t* codewords, void* stream) {
    using namespace exl3;
    if (K < 1 || K > 8) return EXL3_E_BAD_K;
    if (n_tiles < 0) return EXL3_E_BAD_SHAPE;
    if (n_tiles == 0) return EXL3_OK;
    if (!trellis || !codewords) return EXL3_E_NULL_POINTER;
    if ((reinterpret_cast<uintptr_t>(trellis) & 3) || (reinterpret_cast<uintptr_t>(codewords) & 15))
        return EXL3_E_BAD_SHAPE;
    const long long grid = (n_tiles + 31) / 32;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    return dispatch_k_cb(K, 0, [&](auto k, auto) {
        unpack_trellis_kernel<k.value><<<dim3((unsigned)grid), dim3(256), 0, as_stream(stream)>>>(
            reinterpret_cast<const uint32_t*>(trellis), codewords, n_tiles);
        return launch_status();
    });
}
