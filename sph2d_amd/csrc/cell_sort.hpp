// Counting sort of the slots by cell for list builds: the order of
// radix_sort.hpp's stable sort (cell, then slot) in four kernels and the
// build's reorder, where the radix sort takes three kernels for each 8 bits
// of the cell index, and the cell-start table comes with it.
//
//   cell_count_kernel    the slots of each cell, and each slot's place in its
//                        cell in the order the atomics gave it; the slots of the
//                        last build are nearly in order, so a run of equal
//                        cells within a wave is one atomic
//   cell_sums_kernel, cell_starts_kernel   the counts' exclusive scan (the
//                        cell-start table LB); the counts are left zero
//   cell_scatter_kernel  slots and cells to LB + place
//   cell_place           in the reorder: a slot's place by its number among
//                        its cell's, which makes the order that of the stable
//                        sort whatever the atomics gave (dead particles, whose
//                        order nothing depends on, stay where they are)
// The kernels are a few us each, most of it latency.  A build's sort, radix
// and now (each kernel's time, without the gaps between 9 and 4 launches):
// 6,923 particles 34 and 16 us, 188,656 58 and 17, 1,020,263 74 and 23; in 3D
// at 6.6M, where the reorder compares 30 slots a cell, 172 and 136 with it.
#pragma once

#include "device_common.hpp"

namespace rrsph {

constexpr uint32_t kScanItems = 16, kScanCells = kBlock * kScanItems;  // cells of a scan block
__host__ __device__ inline uint32_t scan_blocks(uint32_t ncells) { return (ncells + 2 + kScanCells - 1) / kScanCells; }

__global__ void __launch_bounds__(kBlock) cell_count_kernel(StepParams P, const uint32_t* __restrict__ keys,
                                                            uint32_t* __restrict__ place,
                                                            uint32_t* __restrict__ count,
                                                            const Ctrl* __restrict__ ctrl) {
    if (ctrl->halted) return;
    const uint32_t lb = xcd_block(P.blocks_per_xcd);
    if (lb >= P.nblocks) return;
    const uint32_t s = lb * kBlock + threadIdx.x, lane = __lane_id();
    const bool valid = s < P.n;
    const uint32_t key = valid ? keys[s] : 0xffffffffu;
    const uint32_t left = (uint32_t)__shfl_up((int)key, 1);
    const bool head = lane == 0 || left != key;
    const unsigned long long heads = __ballot(head);
    const unsigned long long upto = heads & (~0ull >> (kWave - 1 - lane));  // this lane's run begins at the last of these
    const unsigned long long after = lane == kWave - 1 ? 0ull : heads >> (lane + 1);
    const uint32_t first = kWave - 1 - (uint32_t)__clzll((long long)upto);
    uint32_t base = 0;
    if (head && valid) base = atomicAdd(&count[key], after ? (uint32_t)__ffsll((long long)after) : kWave - lane);
    base = (uint32_t)__shfl((int)base, (int)first);
    if (valid) place[s] = base + lane - first;
}

// The inclusive scan of v over the block; s_w: kBlock / kWave words.
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* s_w) {
    const uint32_t lane = __lane_id(), wave = threadIdx.x / kWave;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)v, off);
        if ((int)lane >= off) v += y;
    }
    if (lane == kWave - 1) s_w[wave] = v;
    __syncthreads();
    for (uint32_t w = 0; w < wave; ++w) v += s_w[w];
    return v;
}

// The counts of each kScanCells cells (count holds whole blocks, zero past the last cell).
__global__ void __launch_bounds__(kBlock) cell_sums_kernel(const uint32_t* __restrict__ count,
                                                           uint32_t* __restrict__ sums,
                                                           const Ctrl* __restrict__ ctrl) {
    if (ctrl->halted) return;
    __shared__ uint32_t s_w[kBlock / kWave];
    const uint4* c = (const uint4*)(count + (size_t)blockIdx.x * kScanCells);
    uint32_t v = 0;
#pragma unroll
    for (uint32_t k = 0; k < kScanItems / 4; ++k) {
        const uint4 q = c[k * kBlock + threadIdx.x];
        v += q.x + q.y + q.z + q.w;
    }
    v = block_scan(v, s_w);
    if (threadIdx.x == kBlock - 1) sums[blockIdx.x] = v;
}

// LB[c], c <= ncells + 1: slots in cells before c.
__global__ void __launch_bounds__(kBlock) cell_starts_kernel(uint32_t ncells, uint32_t* __restrict__ count,
                                                             const uint32_t* __restrict__ sums,
                                                             uint32_t* __restrict__ LB,
                                                             const Ctrl* __restrict__ ctrl) {
    if (ctrl->halted) return;
    __shared__ uint32_t s_w[kBlock / kWave], s_w2[kBlock / kWave], s_before;
    uint32_t before = 0;
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kBlock) before += sums[b];
    before = block_scan(before, s_w);
    if (threadIdx.x == kBlock - 1) s_before = before;
    uint4* mine = (uint4*)(count + (size_t)blockIdx.x * kScanCells + threadIdx.x * kScanItems);
    uint32_t v[kScanItems], sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < kScanItems / 4; ++k) {
        const uint4 q = mine[k];
        v[4 * k] = q.x;
        v[4 * k + 1] = q.y;
        v[4 * k + 2] = q.z;
        v[4 * k + 3] = q.w;
        mine[k] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (uint32_t k = 0; k < kScanItems; ++k) sum += v[k];
    const uint32_t incl = block_scan(sum, s_w2);  // (its barrier orders s_before too)
    uint32_t at = s_before + incl - sum;
    const uint32_t c0 = blockIdx.x * kScanCells + threadIdx.x * kScanItems;
#pragma unroll
    for (uint32_t k = 0; k < kScanItems; ++k) {
        if (c0 + k < ncells + 2) LB[c0 + k] = at;
        at += v[k];
    }
}

__global__ void __launch_bounds__(kBlock) cell_scatter_kernel(StepParams P, const uint32_t* __restrict__ keys,
                                                              const uint32_t* __restrict__ place,
                                                              const uint32_t* __restrict__ LB,
                                                              uint32_t* __restrict__ skey,
                                                              uint32_t* __restrict__ slots,
                                                              const Ctrl* __restrict__ ctrl) {
    if (ctrl->halted) return;
    const uint32_t lb = xcd_block(P.blocks_per_xcd);
    const uint32_t s = lb * kBlock + threadIdx.x;
    if (lb >= P.nblocks || s >= P.n) return;
    const uint32_t key = keys[s], to = LB[key] + place[s];
    skey[to] = key;
    slots[to] = s;
}

// Where the slot that the scatter left at s (of cell k) goes.
__device__ __forceinline__ uint32_t cell_place(const StepParams& P, const uint32_t* __restrict__ LB,
                                               const uint32_t* __restrict__ slots, uint32_t s, uint32_t k) {
    if (k >= P.ncells) return s;
    const uint32_t b = LB[k], e = LB[k + 1], mine = slots[s];
    uint32_t to = b;
    for (uint32_t i = b; i < e; ++i) to += slots[i] < mine ? 1u : 0u;
    return to;
}

}  // namespace rrsph
