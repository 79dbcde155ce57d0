// Slots of a routing table grouped by expert, up to four to a group: what the grouped expert kernels
// (moe.hip) work through. A list of 16-byte entries; entry 0 holds the number of groups, entry 1 + i
//   {expert, rows, slot 0 | slot 1 << 16, slot 2 | slot 3 << 16}.
//
// One workgroup makes the list, once per call: behind the router's table in the router's own launch
// (its last workgroup), or in a launch of its own. Before, every wave of the expert kernels searched the
// whole table for the slots of its expert (about 100 VALU and 500 scalar instructions a wave), and the
// workgroups of slots that another one carries loaded their first weights for nothing: 24 tokens of 9 slots over
// 257 experts of 2048 x 512, gate/up 58.8 -> 52.5 us, down 32.1 -> 26.0, the block 94.9 -> 85.
#pragma once

#include "exl3_device.hpp"

namespace exl3 {

constexpr int kGroupRows = 4;          // batch rows one workgroup carries
constexpr int kGroupMaxSlots = 1024;   // slots of a list
constexpr int kGroupMaxExperts = 1024;
constexpr int kGroupThreads = 256;     // of the workgroup that makes the list

struct GroupScratch {  // in LDS
    int count[kGroupMaxExperts];
    int first[kGroupMaxExperts];
    int wave_total[kGroupThreads / kWave];
};

// Called by all kGroupThreads threads of a workgroup; expert_of(s), in [0, E), is the expert of slot s.
// Experts in falling order: a shared expert, the last of all and the one with the fullest groups, is
// started first. Which four of an expert's slots meet in a group depends on the order of the LDS
// additions and changes no result: the rows of a group never meet in a sum.
template <class ExpertOf>
__device__ __forceinline__ void make_slot_groups(ExpertOf&& expert_of, int slots, int E, int4* list, GroupScratch& g) {
    constexpr int kSlots = kGroupMaxSlots / kGroupThreads, kExperts = kGroupMaxExperts / kGroupThreads;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < E; i += kGroupThreads) g.count[i] = 0;
    __syncthreads();
    int e[kSlots], rank[kSlots];
#pragma unroll
    for (int j = 0; j < kSlots; j++) {
        const int s = tid + j * kGroupThreads;
        if (s < slots) {
            e[j] = expert_of(s);
            rank[j] = atomicAdd(&g.count[e[j]], 1);
        }
    }
    __syncthreads();
    int before[kExperts], mine = 0;
#pragma unroll
    for (int j = 0; j < kExperts; j++) {
        const int i = tid * kExperts + j;
        before[j] = mine;
        if (i < E) mine += (g.count[E - 1 - i] + kGroupRows - 1) / kGroupRows;
    }
    int upto = mine;  // groups of this thread's experts and all before them in the wave
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int v = __shfl_up(upto, off, kWave);
        if (lane >= off) upto += v;
    }
    if (lane == kWave - 1) g.wave_total[wave] = upto;
    __syncthreads();
    int base = 0;
#pragma unroll
    for (int w = 0; w < kGroupThreads / kWave; w++)
        if (w < wave) base += g.wave_total[w];
    if (tid == kGroupThreads - 1) list[0] = int4{base + upto, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < kExperts; j++) {
        const int i = tid * kExperts + j;
        if (i < E) g.first[E - 1 - i] = base + upto - mine + before[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSlots; j++) {
        const int s = tid + j * kGroupThreads;
        if (s < slots) {
            int4* at = list + 1 + g.first[e[j]] + rank[j] / kGroupRows;
            reinterpret_cast<uint16_t*>(at)[4 + rank[j] % kGroupRows] = (uint16_t)s;
            if (rank[j] % kGroupRows == 0) {
                at->x = e[j];
                at->y = min(kGroupRows, g.count[e[j]] - rank[j]);
            }
        }
    }
}

}  // namespace exl3
