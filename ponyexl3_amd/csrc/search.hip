// Encoder side of the trellis: exl3_quantize_tiles (tail-biting Viterbi search
// over the bitshift trellis) and exl3_pack_trellis (K-bit symbols -> packed tile).
//
// The search follows the arithmetic of the reference's production kernel
// (ponyexl3/convert/metal_search.py:63-196) step for step so that both choose the
// same path: compressed state e = the newest 16-K bits of the codeword; the
// candidate for (fresh, e) is cw = (fresh << (16-K)) | e with predecessor
// cw >> K; path costs are kept as fp16 between steps, the update is one fp32 fma
// clamped to 65504, ties keep the lowest fresh. Pass 0 starts at position 128,
// runs once around the tile and backtracks to the state in front of position 0;
// pass 1 starts at position 0 pinned to that state and has to end in it.
//
// One workgroup of 1024 lanes per CU evaluates all 65536 codewords of a step, 64 per
// lane, and keeps only the minimum per state: which fresh value won matters for the 256
// states on the final path alone, so the backtrack works it out again for those from the
// cost rows of the pass (kept in the caller's workspace, fp16, all of them or every other one)
// instead of every state paying for a select per candidate. A candidate then costs a
// subtraction, an fma and half of a three-operand minimum. The backtrack of one tile is a
// chain of dependent loads; a workgroup keeps two tiles in flight and one of its waves
// walks the chain of one tile while all of them run the forward steps of the other.
#include "exl3_device.hpp"
#include "exl3_host.hpp"

#include <type_traits>

namespace exl3 {

constexpr float kCostInf = 65504.0f;

// fp32 values of four codewords.
template <int CB>
__device__ __forceinline__ void decode4_f32(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                            float (&v)[4]) {
    half2_t a, b;
    decode_pair2<CB>(c0, c1, c2, c3, a, b);
    v[0] = (float)a.x;
    v[1] = (float)a.y;
    v[2] = (float)b.x;
    v[3] = (float)b.y;
}

template <int CB>
__device__ __forceinline__ float decode1_f32(uint32_t cw) {
    float v[4];
    decode4_f32<CB>(cw, cw, cw, cw, v);
    return v[0];
}

// Where things sit for one K. A compressed state e (16-K bits) splits in two ways:
//   as the target of a step   e = p << K | l      (p: 16-2K bits, l: K bits)
//   as its source             e = f << P | p      (f: the K bits above, P = 16-2K)
// The 2^K candidates of a target (p, l) are the sources (f, p), f = 0 .. 2^K - 1, and all
// 2^K targets of one p share them. A cost row is therefore stored as [p][f]: the costs a
// lane needs for one p are one consecutive run of LDS words.
// A lane owns 2^G source groups p (the ones that differ in the low bits of the top K bits
// of their targets, so that the 2^G costs it produces for one l are neighbours in the next
// row: one store) times 2^S targets l of each; from K = 6 on one target, whose candidates
// are shared among FS lanes at K = 7 and 8.
template <int K>
struct SearchMap {
    static constexpr int KR = 16 - K, P = 16 - 2 * K, KK = 1 << K, EDGES = 1 << KR;
    static constexpr int G = K == 2 || K == 3 ? 2 : K == 4 ? 1 : 0;
    static constexpr int S = K <= 6 ? 6 - K - G : 0;
    static constexpr int FS = K <= 6 ? 1 : 1 << (K - 6);
    static constexpr int NG = 1 << G, NS = 1 << S, NF = KK / FS;  // NG * NS * NF = 64
    // Costs are fp16 values. Up to K = 5 a lane uses a cost it has read for 2 (K = 2: 4) targets; there the
    // fma gets it as fp32: with three plain registers it runs at the rate of the simple
    // operations (2.5 cycles per wave and SIMD against 4 for the mixed one, where runs of them
    // meet). K = 3..5: the rows in LDS hold fp32; K = 2, where a lane writes as many costs as it
    // reads, they are converted when read. From K = 6 on every cost is used once. With fp16 rows and the
    // mixed fma instead, all else as it is, ms at 4096 / 64 tiles: K = 2 11.4 / 0.79 against 11.0 / 0.73,
    // 3 11.0 / 0.77 against 9.4 / 0.62, 4 10.6 / 0.77 against 9.0 / 0.60, 5 10.5 / 0.78 against 8.4 / 0.61.
    static constexpr bool PLAIN_FMA = K <= 5, WIDE = K >= 3 && K <= 5;
    // Rows go to the history by the lanes that make them, [lane][target][group], a store each, or (not
    // DIRECT) as 16-byte pieces of the finished LDS row in the next step. K = 3, 4096 tiles: 9.36 ms against
    // 9.67, 64 tiles 0.62 against 0.67; K = 5 8.37 against 8.39; K = 2 10.9 against 10.6, K = 4 8.8 against 8.5.
    static constexpr bool DIRECT = K == 3 || K == 5;
    static constexpr int COST = WIDE ? 4 : 2, ROW_BYTES = COST * EDGES;  // row in LDS
    static constexpr int HIST_BYTES = 2 * EDGES;                          // row in the history, fp16
    typedef std::conditional_t<WIDE, float, half_t> cost_t;
    // Steps that a move of the backtrack goes back. Two up to K = 3, where the 2^2K sources of the sources
    // fit the lanes: only every other row is kept, and those rows are what the search writes most
    // of (K = 2: 32 KB per step, at 256 CUs 6 TB/s). One step at a time, ms at 4096 / 64 tiles: K = 2 13.0 / 0.77
    // against 11.0 / 0.73, K = 3 10.3 / 0.66 against 9.4 / 0.62. At K = 4 there are four to a lane, which cost
    // more registers and time than the rows (64 tiles 604 -> 660 us).
    static constexpr int BACK = K <= 3 ? 2 : 1;
    // Byte offset of source (f, p) in a cost row. The 16-byte units are permuted by exclusive-or so
    // that the lanes of a wave hit different LDS banks in both directions: consecutive p when
    // they read, p that differ in bits K and up when they write. fp32: a plane of 2^P units for every
    // four f; fp16: rows of one p together.
    static __device__ __forceinline__ uint32_t at(uint32_t p, uint32_t f) {
        if constexpr (WIDE) {
            const uint32_t q = f >> 2;
            uint32_t u;
            if constexpr (K == 3) u = p ^ ((p >> 3) & 7) ^ (((p >> 6) & 1) << 3);
            else if constexpr (K == 4) u = p ^ ((p >> 4) & 15);
            else u = p ^ (q & 7) ^ (((p >> 5) & 1) << 3);
            return (((q << P) + u) << 4) + 4 * (f & 3);
        } else if constexpr (K == 2) {
            return ((p ^ ((p >> 4) & 3)) << 3) + 2 * f;  // 8-byte units
        } else if constexpr (K == 6) {
            return (((8 * p + (f >> 3)) ^ (p & 7)) << 4) + 2 * (f & 7);
        } else {
            return (p << (K + 1)) + 2 * f;
        }
    }
    // The same in a row of the history: 16-byte pieces of eight costs, piece i from hist_piece().
    static __device__ __forceinline__ uint32_t hist_at(uint32_t p, uint32_t f) {
        if constexpr (DIRECT) {  // the lane that made state (f, p)
            const uint32_t e = (f << P) | p, ps = e >> K, l = e & (KK - 1);
            constexpr int PL = P - K;
            const uint32_t hi = ps >> PL, t = (ps & ((1u << PL) - 1)) | (hi >> G) << PL | (l >> S) << (P - G);
            return (((t * NS + (l & (NS - 1))) * NG) + (hi & (NG - 1))) * 2;
        } else if constexpr (WIDE) {
            return ((((f >> 3) << P) + p) << 4) + 2 * (f & 7);
        } else {
            return at(p, f);
        }
    }
    static __device__ __forceinline__ uint4_t hist_piece(const unsigned char* row, uint32_t i) {
        if constexpr (!WIDE) {
            return *reinterpret_cast<const uint4_t*>(row + 16 * i);
        } else {
            const uint32_t p = i & ((1u << P) - 1), f = (i >> P) * 8;
            const float4_t a = *reinterpret_cast<const float4_t*>(row + at(p, f));
            const float4_t b = *reinterpret_cast<const float4_t*>(row + at(p, f + 4));
            half8_t h;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                h[c] = (half_t)a[c];  // exact
                h[4 + c] = (half_t)b[c];
            }
            return __builtin_bit_cast(uint4_t, h);
        }
    }
    // p of group g, l of target s and first fresh value of lane `tid`
    static __device__ __forceinline__ uint32_t lane_p(uint32_t tid, int g) {
        if constexpr (K <= 5) {
            constexpr int PL = P - K;  // bits of p below the top K
            const uint32_t plow = tid & ((1u << PL) - 1), phigh = (tid >> PL) & ((1u << (K - G)) - 1);
            return (((phigh << G) | (uint32_t)g) << PL) | plow;
        } else {
            return (tid / FS) >> K;
        }
    }
    static __device__ __forceinline__ uint32_t lane_l(uint32_t tid, int s) {
        if constexpr (K <= 5) return ((tid >> (P - G)) << S) | (uint32_t)s;
        else return (tid / FS) & (KK - 1);
    }
    static __device__ __forceinline__ uint32_t lane_f(uint32_t tid) { return (tid & (FS - 1)) * NF; }
};

constexpr int kSearchThreads = 1024;

template <int CTRL>
__device__ __forceinline__ uint32_t min_dpp(uint32_t v) {
    const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
    return o < v ? o : v;
}

// Minimum over the wave of values that repeat every 2^K lanes.
template <int K>
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
    v = min_dpp<0xB1>(v);                               // lanes 1 apart
    v = min_dpp<0x4E>(v);                               // 2 apart
    if constexpr (K > 2) v = min_dpp<0x141>(v);         // half-row mirror: 4 apart
    if constexpr (K > 3) v = min_dpp<0x140>(v);         // row mirror: 8 apart
    if constexpr (K > 4) {
        float a = __builtin_bit_cast(float, v), b = a;  // 16 apart
        swap_rows16(a, b);
        const uint32_t x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
        v = x < y ? x : y;
    }
    if constexpr (K > 5) {
        float a = __builtin_bit_cast(float, v), b = a;  // 32 apart
        swap_halves32(a, b);
        const uint32_t x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
        v = x < y ? x : y;
    }
    return v;
}

// One step of the backtrack: the predecessor of state `edge` given the costs before the
// step (cost[j] = that of fresh value lane + 64 j, repeating if there are fewer than 64).
// The first fresh value that attains the minimum wins; 0 if no candidate stays under the
// bound, as in the reference. Errors are non-negative, so their bits order like they do.
template <int K, int CB>
__device__ __forceinline__ uint32_t search_predecessor(const half_t (&cost)[K > 6 ? 1 << (K - 6) : 1],
                                                       uint32_t edge, float target, int lane) {
    using M = SearchMap<K>;
    constexpr int NB = K > 6 ? 1 << (K - 6) : 1;
    uint32_t err[NB], best = __builtin_bit_cast(uint32_t, kCostInf);
    const uint32_t bound = best;
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const uint32_t f = (uint32_t)(lane + 64 * j) & (M::KK - 1);
        const float dh = decode1_f32<CB>((f << M::KR) | edge) - target;
        err[j] = __builtin_bit_cast(uint32_t, __builtin_fmaf(dh, dh, (float)cost[j]));
        best = err[j] < best ? err[j] : best;
    }
    best = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_min<K>(best));
    uint32_t f = 0;
#pragma unroll
    for (int j = NB - 1; j >= 0; j--) {
        const unsigned long long hit = __ballot(err[j] == best);
        if (hit) f = (uint32_t)(64 * j + __builtin_ctzll(hit));
    }
    return best < bound ? (f << M::P) | (edge >> K) : 0u;
}

// Minimum over all lanes of values that are equal within aligned groups of 2^K lanes (K = 2, 3).
template <int K>
__device__ __forceinline__ uint32_t groups_min(uint32_t v) {
    if constexpr (K == 2) v = min_dpp<0x141>(v);
    v = min_dpp<0x140>(v);
    if constexpr (K == 3) {  // (K = 2: the sixteen lanes repeat)
        float a = __builtin_bit_cast(float, v), b = a;
        swap_rows16(a, b);
        uint32_t x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
        v = x < y ? x : y;
        a = __builtin_bit_cast(float, v), b = a;
        swap_halves32(a, b);
        x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
        v = x < y ? x : y;
    }
    return v;
}

// Two steps of the backtrack at once (K <= 3): lane (f1, f2), f2 the low K bits, has in `cost` the cost, two
// steps back, of the source f2 of the source f1 of state `edge`. The costs in between are those of the
// forward pass: minimum over f2, rounded to fp16. t1, t2: targets of the later and the earlier step.
// Returns the state in between and sets `edge` to the one before; `fetch` gives the costs of the
// sources of state 0, which stands in where no candidate stays under the bound.
template <int K, int CB, class Fetch>
__device__ __forceinline__ uint32_t search_two_back(half_t cost, uint32_t& edge, float t1, float t2, int lane,
                                                    Fetch&& fetch) {
    using M = SearchMap<K>;
    constexpr uint32_t KK = M::KK;
    const uint32_t bound = __builtin_bit_cast(uint32_t, kCostInf), p = edge >> K;
    const uint32_t f2 = lane & (KK - 1), f1 = ((uint32_t)lane >> K) & (KK - 1);
    const float d2 = decode1_f32<CB>((f2 << M::KR) | (f1 << M::P) | p) - t2;
    const uint32_t err2 = __builtin_bit_cast(uint32_t, __builtin_fmaf(d2, d2, (float)cost));
    const uint32_t best2 = wave_min<K>(err2);  // of the lane's group
    const half_t between = (half_t)__builtin_fminf(kCostInf, __builtin_bit_cast(float, best2));
    const float d1 = decode1_f32<CB>((f1 << M::KR) | edge) - t1;
    const uint32_t err1 = __builtin_bit_cast(uint32_t, __builtin_fmaf(d1, d1, (float)between));
    const uint32_t best1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)groups_min<K>(err1));
    if (best1 >= bound) {
        const half_t c[1] = {fetch()};
        edge = search_predecessor<K, CB>(c, 0u, t2, lane);
        return 0u;
    }
    // lowest f1 and, in its group, lowest f2 that attain the minima
    const int first = (int)__builtin_ctzll(__ballot(err1 == best1)) & ~(int)(KK - 1);
    const uint32_t mid = ((uint32_t)(first >> K) << M::P) | p;
    const uint32_t best = (uint32_t)__builtin_amdgcn_readlane((int)best2, first);
    const unsigned long long hit = __ballot(err2 == best) >> first;
    edge = best < bound ? ((uint32_t)__builtin_ctzll(hit) << M::P) | (mid >> K) : 0u;
    return mid;
}

// Workgroup b walks over tiles b, b + gridDim.x, .. in phases of 256 steps. With two
// cost-history slots (b + gridDim.x < n_slots) phase n runs the forward steps of slot n & 1
// (warm-up pass, two phases later the pinned pass) and the backtrack of what slot ~n & 1 did
// in phase n - 1; with one slot the odd phases only backtrack. (A tile
// alone on its CU takes 0.80 ms, of which the forward steps are 0.70.)
//
// The kernel is bound by VALU issue: 64 subtractions, 64 fmas and 32 v_min3 per lane and step, plus
// rounding and storing the 64 / NF results; the lane's 64 decoded values stay in registers as fp32 for
// the whole phase. Add and fma on plain registers run at 2.5 cycles per wave and SIMD where waves
// meet in runs of them, everything else (minima, conversions, the mixed fma) at 4; fp32 matrix
// instructions occupy the same units (16x16x1: 32 cycles for 16 differences), which pays against the
// subtraction only beside the mixed fma. 16 waves of at most 128 registers fill the CU, so the
// whole of a step hides its own LDS latency; one barrier per step. The wave that backtracks (0) waits for
// its loads of a step before it stores, and in the forms that copy finished rows it stores nothing.
// Measured, 4096 tiles (MCG), ms, before the four (mixed fma, fp16 rows, every row kept and copied, subtractions) and with
// all of them: K = 2 13.3 -> 10.6, 3 11.4 -> 9.05, 4 11.1 -> 8.5, 5 11.1 -> 8.0, 6 11.2 -> 9.9, 7 11.8 -> 10.7, 8 11.8
// -> 10.7; up to 256 tiles at once 0.84 -> 0.73, 0.81 -> 0.63, 0.81 -> 0.61, 0.82 -> 0.61, 0.79 -> 0.70, 0.83 -> 0.76, 0.87
// -> 0.78. What each gives by itself is beside it (SearchMap, and the differences below).
template <int K, int CB>
__global__ __launch_bounds__(kSearchThreads, 1) void quantize_tiles_kernel(
    const float* __restrict__ tiles, float* __restrict__ q_tiles, uint16_t* __restrict__ indices,
    unsigned char* history, int n_tiles, int n_slots) {
    using M = SearchMap<K>;
    constexpr int EDGES = M::EDGES, KK = M::KK, NG = M::NG, NS = M::NS, NF = M::NF, FS = M::FS;
    constexpr int NB = K > 6 ? 1 << (K - 6) : 1;
    constexpr size_t kSlotBytes = (size_t)256 * M::HIST_BYTES;
    using cost_t = typename M::cost_t;
    extern __shared__ __attribute__((aligned(16))) unsigned char rows_s[];  // [2][ROW_BYTES]
    __shared__ float target_s[2][256];
    __shared__ uint16_t state_s[256];
    __shared__ uint32_t red_key[16];
    __shared__ uint32_t pin_s[2];
    uint32_t tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane((int)(tid >> 6));

    const bool two = (int)(blockIdx.x + gridDim.x) < n_slots;
    auto phase_tile = [&](int n) -> long long {  // tile of forward phase n, -1 if it has none
        if (n < 0 || (!two && (n & 1))) return -1;
        const int j = two ? 2 * (n >> 2) + (n & 1) : n >> 2;
        const long long t = blockIdx.x + (long long)gridDim.x * j;
        return t < n_tiles ? t : -1;
    };
    uint32_t back_edge = 0;  // state the pending backtrack starts from
    for (int n = 0;; n++) {
        const long long tile = phase_tile(n), back_tile = phase_tile(n - 1);
        if (tile < 0 && back_tile < 0 && phase_tile(n + 1) < 0 && phase_tile(n + 2) < 0 &&
            phase_tile(n + 3) < 0)
            break;
        // the lane's addresses are derived anew in every phase: held across the phases
        // they would take registers that the step loop needs
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63;
        const int slot = n & 1, pass = (n >> 1) & 1, back_pass = ((n - 1) >> 1) & 1;
        unsigned char* hist = history + kSlotBytes * (blockIdx.x + (size_t)slot * gridDim.x);
        const unsigned char* back_hist = history + kSlotBytes * (blockIdx.x + (size_t)(slot ^ 1) * gridDim.x);
        // the warm-up pass starts at position 128 and is walked back to position 0 only
        const int roll = pass == 0 ? 128 : 0, back_roll = back_pass == 0 ? 128 : 0;
        const int back_end = back_pass == 0 ? 128 : 0;
        const bool backs = back_tile >= 0 && wave == 0;
        const uint32_t back_pin = back_pass == 1 ? pin_s[slot ^ 1] : 0;
        uint32_t edge = __builtin_amdgcn_readfirstlane((int)back_edge);

        // one move of the pending backtrack (one step, two up to K = 3) in two halves: request the costs in
        // front of it, later pick the predecessor. Costs of source (f, p) after step s (-1: in front of
        // the pinned pass, nothing but the pin):
        auto back_cost = [&](int s, uint32_t p, uint32_t f) {
            if (s < 0) return ((f << M::P) | p) == back_pin ? (half_t)0.0f : bits_to_half(0x7C00);
            return *reinterpret_cast<const half_t*>(back_hist + (size_t)(s / M::BACK) * M::HIST_BYTES + M::hist_at(p, f));
        };
        half_t cost[NB];
        auto back_request = [&](int step) {
            if constexpr (M::BACK == 2) {
                const uint32_t f1 = ((uint32_t)lane >> K) & (KK - 1);
                cost[0] = back_cost(step - 2, ((f1 << M::P) | (edge >> K)) >> K, lane & (KK - 1));
            } else {
#pragma unroll
                for (int j = 0; j < NB; j++) cost[j] = back_cost(step - 1, edge >> K, (uint32_t)(lane + 64 * j) & (KK - 1));
            }
        };
        auto back_take = [&](int step) {
            const int ri = (step + back_roll) & 255;
            if constexpr (M::BACK == 2) {
                const int rj = (step - 1 + back_roll) & 255;
                const uint32_t last = edge;
                const uint32_t mid = search_two_back<K, CB>(cost[0], edge, target_s[slot ^ 1][ri], target_s[slot ^ 1][rj],
                                                            lane, [&] { return back_cost(step - 2, 0u, lane & (KK - 1)); });
                if (lane == 0) {
                    state_s[ri] = (uint16_t)((mid << K) | last);
                    state_s[rj] = (uint16_t)((edge << K) | mid);
                }
            } else {
                const uint32_t prev = search_predecessor<K, CB>(cost, edge, target_s[slot ^ 1][ri], lane);
                if (lane == 0) state_s[ri] = (uint16_t)((prev << K) | edge);
                edge = prev;
            }
        };

        if (tile < 0) {
            if (backs)
                for (int step = 255; step >= back_end; step -= M::BACK) {
                    back_request(step);
                    back_take(step);
                }
        } else {
            const uint32_t pin = pin_s[slot];  // (pass 0: not used)
            if (pass == 0 && tid < 256) target_s[slot][tid] = tiles[(size_t)tile * 256 + tid];
            // Step 0 has no predecessor costs: a row of zeros stands in for them
            // (fma(dh, dh, 0) is the rounded square), and in the pinned pass +inf
            // everywhere but at the pin keeps every other predecessor from winning.
#pragma unroll 1
            for (uint32_t e = tid; e < (uint32_t)EDGES; e += kSearchThreads) {
                const cost_t open = pass == 0 ? (cost_t)0.0f : (cost_t)__builtin_inff();
                *reinterpret_cast<cost_t*>(rows_s + M::ROW_BYTES + M::at(e & ((1u << M::P) - 1), e >> M::P)) =
                    pass == 1 && e == pin ? (cost_t)0.0f : open;
            }
            // decoded values of the lane's codewords (f, p, l), f << KR | p << K | l, for the
            // steps of this phase (kept across phases they would be live next to the
            // backtrack's own code and spill)
            float16_t val[4];  // [group][target][fresh], flat
#pragma unroll
            for (int g = 0; g < NG; g++)
#pragma unroll
                for (int s = 0; s < NS; s++) {
                    const uint32_t e = (M::lane_p(tid, g) << K) | M::lane_l(tid, s);
#pragma unroll
                    for (int f = 0; f < NF; f += 4) {
                        const uint32_t c = ((M::lane_f(tid) + f) << M::KR) | e;
                        float v[4];
                        decode4_f32<CB>(c, c + EDGES, c + 2 * EDGES, c + 3 * EDGES, v);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            asm volatile("" : "+v"(v[i]));  // decoded here, not again in every step
                            val[((g * NS + s) * NF + f) / 16][((g * NS + s) * NF + f) % 16 + i] = v[i];
                        }
                    }
                }
            __syncthreads();
#pragma unroll 1
            for (int step = 0; step < 256; step++) {
                const unsigned char* prev_row = rows_s + ((step & 1) ^ 1) * M::ROW_BYTES;
                unsigned char* row = rows_s + (step & 1) * M::ROW_BYTES;
                const float target = target_s[slot][(step + roll) & 255];
                // (a move of two steps is requested in one forward step and made in the next)
                const int back_step = 255 - step / M::BACK * M::BACK;
                const bool back_now = backs && back_step >= back_end;
                if (back_now && step % M::BACK == 0) back_request(back_step);
                // the row before this one goes to the history (what the backtrack never reads is
                // left out: up to K = 3 every other row, in the warm-up pass those of the first half)
                if (!M::DIRECT && step > (pass == 0 ? 127 : 0) && step % M::BACK == 0) {
                    unsigned char* dst = hist + (size_t)((step - 1) / M::BACK) * M::HIST_BYTES;
                    if (tid >= kSearchThreads / 2)
                        for (uint32_t i = tid - kSearchThreads / 2; i < (uint32_t)M::HIST_BYTES / 16;
                             i += kSearchThreads / 2)
                            *reinterpret_cast<uint4_t*>(dst + 16 * i) = M::hist_piece(prev_row, i);
                }
                half_t out[NG][NS];
                const float minus_target = -target;
                auto differences = [&](int j) {
                    return __builtin_amdgcn_mfma_f32_16x16x1f32(1.0f, minus_target, val[j], 0, 0, 0);
                };
                float16_t diff, diff_next;
                if constexpr (!M::PLAIN_FMA) diff_next = differences(0);
#pragma unroll
                for (int g = 0; g < NG; g++) {
                    const uint32_t p = M::lane_p(tid, g), f0 = M::lane_f(tid);
                    float best[NS];
#pragma unroll
                    for (int s = 0; s < NS; s++) best[s] = kCostInf;
#pragma unroll
                    for (int fc = 0; fc < NF; fc += 8) {
                        constexpr int CH = NF < 8 ? NF : 8;
                        float pc[CH];
                        if constexpr (M::WIDE) {
#pragma unroll
                            for (int i = 0; i < CH; i += 4) {
                                const float4_t q = *reinterpret_cast<const float4_t*>(prev_row + M::at(p, f0 + fc + i));
#pragma unroll
                                for (int c = 0; c < 4; c++) pc[i + c] = q[c];
                            }
                        } else if constexpr (CH == 4) {
                            const half4_t q = *reinterpret_cast<const half4_t*>(prev_row + M::at(p, f0 + fc));
#pragma unroll
                            for (int c = 0; c < 4; c++) {
                                pc[c] = (float)q[c];
                                asm("" : "+v"(pc[c]));  // converted here, not in every fma
                            }
                        } else {
                            const uint4_t q = *reinterpret_cast<const uint4_t*>(prev_row + M::at(p, f0 + fc));
                            halfs_to_floats(q, pc);  // folded into the fma
                        }
                        // From K = 6 on sixteen differences at a time come from the matrix pipe (-target times one
                        // on top of the values: one rounding, as the subtraction), a batch ahead. With the
                        // subtraction, ms at 4096 / 64 tiles: K = 6 10.4 / 0.72 against 10.0 / 0.69, 7 11.1 / 0.77
                        // against 10.7 / 0.75, 8 11.65 / 0.85 against 10.9 / 0.76.
                        if constexpr (!M::PLAIN_FMA) {
                            if (fc % 16 == 0) {
                                diff = diff_next;
                                if (fc + 16 < NF) diff_next = differences(fc / 16 + 1);
                            }
                        }
                        // differences, fmas and minima in runs: the simple operations run at their higher
                        // rate where waves meet in them
                        float d[NS][CH];
                        if constexpr (M::PLAIN_FMA) {
#pragma unroll
                            for (int s = 0; s < NS; s++)
#pragma unroll
                                for (int i = 0; i < CH; i++) d[s][i] = val[((g * NS + s) * NF + fc) / 16][((g * NS + s) * NF + fc) % 16 + i] - target;
                            __builtin_amdgcn_sched_barrier(0);
                        } else {
#pragma unroll
                            for (int i = 0; i < CH; i++) d[0][i] = diff[fc % 16 + i];
                        }
#pragma unroll
                        for (int s = 0; s < NS; s++)
#pragma unroll
                            for (int i = 0; i < CH; i++) d[s][i] = __builtin_fmaf(d[s][i], d[s][i], pc[i]);
                        if constexpr (M::PLAIN_FMA) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int s = 0; s < NS; s++)
#pragma unroll
                            for (int i = 0; i < CH; i += 2)
                                // an error at or above the bound never wins, which is all the
                                // reference's clamp to 65504 achieves
                                best[s] = __builtin_fminf(__builtin_fminf(best[s], d[s][i]), d[s][i + 1]);
                    }
#pragma unroll
                    for (int s = 0; s < NS; s++) {
                        if constexpr (FS >= 2) best[s] = __builtin_fminf(best[s], dpp_move<0xB1>(best[s]));
                        if constexpr (FS >= 4) best[s] = __builtin_fminf(best[s], dpp_move<0x4E>(best[s]));
                        out[g][s] = (half_t)best[s];
                    }
                }
#pragma unroll
                for (int s = 0; s < NS; s++) {
                    const uint32_t e = (M::lane_p(tid, 0) << K) | M::lane_l(tid, s);
                    unsigned char* dst = row + M::at(e & ((1u << M::P) - 1), e >> M::P);
                    if constexpr (NG == 4 && !M::WIDE) {
                        *reinterpret_cast<half4_t*>(dst) = half4_t{out[0][s], out[1][s], out[2][s], out[3][s]};
                    } else if constexpr (NG == 4) {
                        *reinterpret_cast<float4_t*>(dst) =
                            float4_t{(float)out[0][s], (float)out[1][s], (float)out[2][s], (float)out[3][s]};
                    } else if constexpr (NG == 2) {
                        *reinterpret_cast<float2_t*>(dst) = float2_t{(float)out[0][s], (float)out[1][s]};
                    } else {
                        if (FS == 1 || (tid & (FS - 1)) == 0) *reinterpret_cast<cost_t*>(dst) = (cost_t)out[0][s];
                    }
                }
                if (back_now && step % M::BACK == M::BACK - 1) back_take(back_step);
                if constexpr (M::DIRECT) {
                    if (step % M::BACK == M::BACK - 1 && step >= (pass == 0 ? 127 : 0)) {
                        typedef half_t piece_t __attribute__((ext_vector_type(NG * NS < 8 ? NG * NS : 8)));
                        constexpr int N = sizeof(piece_t) / 2;
#pragma unroll
                        for (int j = 0; j < NG * NS; j += N) {
                            piece_t h;
#pragma unroll
                            for (int i = 0; i < N; i++) h[i] = out[(i + j) % NG][(i + j) / NG];
                            *reinterpret_cast<piece_t*>(hist + (size_t)(step / M::BACK) * M::HIST_BYTES + (NG * NS * tid + j) * 2) = h;
                        }
                    }
                }
                __syncthreads();
            }
        }
        if (backs && lane == 0 && back_pass == 0) pin_s[slot ^ 1] = edge;  // state in front of position 0
        if (tile >= 0 && pass == 0) {
            // first minimum of the final costs: key = cost bits : state (step 255 wrote row 1)
            uint32_t key = 0xFFFFFFFFu;
#pragma unroll 1
            for (uint32_t e = tid; e < (uint32_t)EDGES; e += kSearchThreads) {
                const uint32_t bits = half_to_bits((half_t) * reinterpret_cast<const cost_t*>(
                    rows_s + M::ROW_BYTES + M::at(e & ((1u << M::P) - 1), e >> M::P)));
                const uint32_t cand = (bits << 16) | e;
                key = cand < key ? cand : key;
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                const uint32_t o = (uint32_t)__shfl_xor((int)key, off, kWave);
                key = o < key ? o : key;
            }
            if (lane == 0) red_key[wave] = key;
        }
        __syncthreads();
        if (back_tile >= 0 && back_pass == 1 && tid < 256) {
            const uint32_t state = state_s[tid];
            indices[(size_t)back_tile * 256 + tid] = (uint16_t)state;
            q_tiles[(size_t)back_tile * 256 + tid] = decode1_f32<CB>(state);
        }
        if (tile >= 0 && pass == 0) {
            uint32_t key = red_key[0];
            for (int w = 1; w < 16; w++) key = red_key[w] < key ? red_key[w] : key;
            // a cost that never dropped below the bound selects state 0
            back_edge = (key >> 16) >= 0x7BFFu ? 0u : (key & 0xFFFFu);
        } else {
            back_edge = pin_s[slot];  // the pinned pass has to end where it began
        }
        __syncthreads();
    }
}

// K-bit symbols -> packed tile (ponyexl3/ref/trellis.py:13-49, mlx_trellis.py:66-84).
// Symbol c occupies stream bits [c*K, (c+1)*K), MSB first inside each 32-bit
// word; one lane assembles one word.
__global__ __launch_bounds__(256) void pack_trellis_kernel(const uint16_t* __restrict__ encoded,
                                                           uint32_t* __restrict__ packed,
                                                           long long n_words, int K) {
    const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
    if (gid >= n_words) return;
    const int words_per_tile = 8 * K;
    const long long tile = gid / words_per_tile;
    const int d = (int)(gid % words_per_tile);
    const uint16_t* src = encoded + tile * 256;
    const uint32_t mask = (1u << K) - 1u;
    const int first = (32 * d) / K, last = (32 * d + 31) / K;
    uint32_t word = 0;
    for (int c = first; c <= last; c++) {
        const int off = c * K - 32 * d;  // may be negative: the symbol began in the previous word
        const uint64_t v = (uint64_t)(src[c] & mask) << 32;
        word |= (uint32_t)(v >> (off + K));
    }
    packed[gid] = word;
}

static int quantize_cus() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
    return cus;
}

// Cost-history slots worth having: two tiles in flight on every CU.
static int quantize_slots_wanted() { return 2 * quantize_cus(); }

}  // namespace exl3

EXL3_EXPORT size_t exl3_quantize_slot_bytes(int K) {
    if (K < 2 || K > 8) return 0;
    return (size_t)256 * sizeof(uint16_t) << (16 - K);
}

EXL3_EXPORT size_t exl3_quantize_workspace_bytes(int n_tiles, int K) {
    if (K < 2 || K > 8 || n_tiles < 1) return 0;
    const int want = exl3::quantize_slots_wanted();
    return exl3_quantize_slot_bytes(K) * (size_t)(n_tiles < want ? n_tiles : want);
}

EXL3_EXPORT int exl3_quantize_tiles(const float* tiles, int n_tiles, int K, int cb, float* q_tiles,
                                    uint16_t* indices, void* workspace, size_t workspace_bytes,
                                    void* stream) {
    using namespace exl3;
    if (K < 2 || K > 8) return EXL3_E_BAD_K;  // K = 1 is not supported by the reference either
    if (int rc = check_k_cb(K, cb)) return rc;
    if (n_tiles < 0) return EXL3_E_BAD_SHAPE;
    if (n_tiles == 0) return EXL3_OK;
    if (!tiles || !q_tiles || !indices || !workspace) return EXL3_E_NULL_POINTER;
    const size_t slot = exl3_quantize_slot_bytes(K);
    size_t slots = workspace_bytes / slot;
    if (slots < 1) return EXL3_E_WORKSPACE;
    const size_t want = (size_t)quantize_slots_wanted();
    if (slots > want) slots = want;
    if (slots > (size_t)n_tiles) slots = (size_t)n_tiles;
    // one workgroup per CU; slots beyond the grid are the workgroups' second ones
    const size_t cus = (size_t)quantize_cus();
    const size_t grid = slots < cus ? slots : cus;
    return dispatch_k_cb(K, cb, [&](auto k, auto c) {
        if constexpr (k.value < 2) {
            return (int)EXL3_E_BAD_K;
        } else {
            constexpr size_t lds = 2 * (size_t)SearchMap<k.value>::ROW_BYTES;  // two cost rows
            if (hipFuncSetAttribute(
                    reinterpret_cast<const void*>(quantize_tiles_kernel<k.value, c.value>),
                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
                return (int)EXL3_E_LAUNCH;
            quantize_tiles_kernel<k.value, c.value>
                <<<dim3((unsigned)grid), dim3(kSearchThreads), lds, as_stream(stream)>>>(
                    tiles, q_tiles, indices, reinterpret_cast<unsigned char*>(workspace), n_tiles,
                    (int)slots);
            return launch_status();
        }
    });
}

EXL3_EXPORT int exl3_pack_trellis(const uint16_t* encoded, long long n_tiles, int K,
                                  uint16_t* packed, void* stream) {
    using namespace exl3;
    if (K < 1 || K > 8) return EXL3_E_BAD_K;
    if (n_tiles < 0) return EXL3_E_BAD_SHAPE;
    if (n_tiles == 0) return EXL3_OK;
    if (!encoded || !packed) return EXL3_E_NULL_POINTER;
    if (reinterpret_cast<uintptr_t>(packed) & 3) return EXL3_E_BAD_SHAPE;
    const long long n_words = n_tiles * 8 * K;
    const long long grid = (n_words + 255) / 256;
    if (grid > 0x7FFFFFFFLL) return EXL3_E_BAD_SHAPE;
    pack_trellis_kernel<<<dim3((unsigned)grid), dim3(256), 0, as_stream(stream)>>>(
        encoded, reinterpret_cast<uint32_t*>(packed), n_words, K);
    return launch_status();
}
