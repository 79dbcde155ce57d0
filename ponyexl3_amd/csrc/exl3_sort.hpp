// (token, slot) pairs sorted by expert and the row-block table of the prefill kernels, by the workgroups of one
// launch: a kernel of its own, or together with the rotation of the pairs' rows.
#pragma once

#include "exl3_device.hpp"

namespace exl3 {

constexpr int kSortMaxExperts = 1024;
constexpr int kSortMaxGroups = 32;

// Routing indices come from the caller's device memory; an out-of-range value is
// clamped so that it can never turn into an out-of-bounds read.
__device__ __forceinline__ int clamp_expert(int e, int E) { return e < 0 ? 0 : (e >= E ? E - 1 : e); }

struct SortArgs {
    const int* indices;
    int n_pairs, top_k, E, block_rows;
    int *order, *tok, *sidx;
    int4* table;
    int table_len, groups, staged;
};

// Ints of LDS that a workgroup of `threads` needs.
__host__ __device__ constexpr size_t sort_lds_ints(int threads, const SortArgs& a) {
    return (size_t)(threads / 64 + 2) * a.E + (a.staged ? a.n_pairs : 0);
}

// Stable counting sort by expert id. Outputs, all indexed by sorted position:
//   order[pos] = pair index (token * top_k + slot), tok[pos] = token,
//   sidx[pos] = expert (tok and sidx may be NULL); table[b] = {expert, first row, end row of
//   the expert, 0} for every block of block_rows rows, unused entries {E-1, N, N, 0} (empty).
// With `staged` the order is put together in LDS and written out in order: one CU's scattered
// 4-byte stores (64 lines per instruction) are what this kernel is otherwise bound by.
//
// Every workgroup owns a contiguous part of the pairs, each of its waves a segment of that and a
// cursor per expert in LDS: count, one scan over (expert, wave), then every wave places its segment 64
// pairs at a time without meeting the others. A pair's rank among equal experts of its 64 comes from
// ballots over the bits of the expert id. Where a part begins is known without an exchange:
// every workgroup counts all pairs, those before and behind its own part in two counters per expert (13 833
// pairs: 14 loads and LDS additions per lane). There one workgroup takes 21.5 us, 14 take 8.3; 6972 pairs
// 12.3 and 7.3.
__host__ __device__ constexpr int sort_pairs_per_wave(int n_pairs, int groups, int threads) {
    const long long waves = (long long)groups * (threads / 64);
    return (int)((n_pairs + 64 * waves - 1) / (64 * waves) * 64);
}

template <int THREADS>
__device__ __forceinline__ void sort_pairs(const SortArgs& a, int group, int* cursor) {
    constexpr int kWaves = THREADS / 64, kPer = kSortMaxExperts / THREADS;  // experts of a thread in the scan
    // cursor: [kWaves][E], pairs before [E], behind [E], staging
    __shared__ int scan_tmp[2][kWaves];
    const int* const indices = a.indices;
    const int n_pairs = a.n_pairs, E = a.E, block_rows = a.block_rows, groups = a.groups;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int* const before = cursor + kWaves * E;
    int* const behind = before + E;
    int* const stage = behind + E;
    for (int i = tid; i < (kWaves + 2) * E; i += THREADS) cursor[i] = 0;
    __syncthreads();
    const int per_wave = sort_pairs_per_wave(n_pairs, groups, THREADS);
    const int part = group * kWaves * per_wave;
    const int begin = min(part + wave * per_wave, n_pairs), end = min(begin + per_wave, n_pairs);
    int* mine = cursor + wave * E;
    // eight loads in flight
    for (int i0 = begin + lane; groups == 1 && i0 < end; i0 += 8 * 64) {
        int e[8];
#pragma unroll
        for (int j = 0; j < 8; j++) e[j] = indices[min(i0 + j * 64, n_pairs - 1)];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (i0 + j * 64 < end) atomicAdd(&mine[clamp_expert(e[j], E)], 1);
    }
    for (int i0 = wave * 64; groups > 1 && i0 < n_pairs; i0 += 8 * THREADS) {
        int e[8];
#pragma unroll
        for (int j = 0; j < 8; j++) e[j] = indices[min(i0 + j * THREADS + lane, n_pairs - 1)];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int i = i0 + j * THREADS;  // 64 pairs of one segment
            int* const count = i < part ? before
                               : i >= part + kWaves * per_wave ? behind : cursor + (i - part) / per_wave * E;
            if (i + lane < n_pairs) atomicAdd(&count[clamp_expert(e[j], E)], 1);
        }
    }
    __syncthreads();

    // exclusive scans over the experts (kPer to a thread): rows and blocks
    int c[kPer], inc_rows = 0, inc_blk = 0;
#pragma unroll
    for (int p = 0; p < kPer; p++) {
        const int e = tid * kPer + p;
        c[p] = 0;
        if (e < E) {
#pragma unroll
            for (int w = 0; w < kWaves + 2; w++) c[p] += cursor[w * E + e];
        }
        inc_rows += c[p];
        inc_blk += (c[p] + block_rows - 1) / block_rows;
    }
    const int own_rows = inc_rows, own_blk = inc_blk;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int r = __shfl_up(inc_rows, off, kWave), b = __shfl_up(inc_blk, off, kWave);
        if (lane >= off) {
            inc_rows += r;
            inc_blk += b;
        }
    }
    if (lane == 63) {
        scan_tmp[0][wave] = inc_rows;
        scan_tmp[1][wave] = inc_blk;
    }
    __syncthreads();
    int base_rows = 0, base_blk = 0, total_blk = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
        if (w < wave) {
            base_rows += scan_tmp[0][w];
            base_blk += scan_tmp[1][w];
        }
        total_blk += scan_tmp[1][w];
    }
    int row0 = base_rows + inc_rows - own_rows;  // first sorted row and block of the thread's first expert
    int blk0 = base_blk + inc_blk - own_blk;
#pragma unroll
    for (int p = 0; p < kPer; p++) {
        const int e = tid * kPer + p;
        if (e >= E) break;
        int at = row0 + before[e];
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const int n = cursor[w * E + e];
            cursor[w * E + e] = at;
            at += n;
        }
        const int nb = (c[p] + block_rows - 1) / block_rows;
        if (group == 0)
            for (int b = 0; b < nb && blk0 + b < a.table_len; b++)
                a.table[blk0 + b] = int4{e, row0 + b * block_rows, row0 + c[p], 0};
        row0 += c[p];
        blk0 += nb;
    }
    for (int b = total_blk + tid + group * THREADS; b < a.table_len; b += THREADS * groups)
        a.table[b] = int4{E - 1, n_pairs, n_pairs, 0};
    __syncthreads();

    int ebits = 0;
    while ((1 << ebits) < E) ebits++;
    for (int i0 = begin; i0 < end; i0 += 8 * 64) {
        int ids[8];
#pragma unroll
        for (int j = 0; j < 8; j++) ids[j] = indices[min(i0 + j * 64 + lane, n_pairs - 1)];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int i = i0 + j * 64 + lane;
            const bool valid = i < end;
            const int e = valid ? clamp_expert(ids[j], E) : 0;
            unsigned long long same = __ballot(valid);
            if (!same) break;
            for (int b = 0; b < ebits; b++) {
                const unsigned long long m = __ballot((e >> b) & 1);
                same &= ((e >> b) & 1) ? m : ~m;
            }
            const int rank = __popcll(same & ((1ull << lane) - 1ull));
            // every lane reads its expert's cursor before the first of the equal ones moves it,
            // and the next 64 pairs read behind that (e is 0 where there is no pair)
            const int first = mine[e];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (valid && rank == 0) mine[e] = first + __popcll(same);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (valid) {
                const int pos = first + rank;
                if (a.staged) stage[pos] = i;
                else a.order[pos] = i;
                if (a.tok) a.tok[pos] = i / a.top_k;
                if (a.sidx) a.sidx[pos] = e;
            }
        }
    }
    if (!a.staged) return;
    __syncthreads();
    for (int i = tid; i < n_pairs; i += THREADS) a.order[i] = stage[i];
}

}  // namespace exl3
