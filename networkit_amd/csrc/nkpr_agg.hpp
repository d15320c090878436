// Sums per key over a stream of (key, weight) pairs whose keys repeat very unevenly: the out-degrees
// of a graph's arcs.  On a power-law graph most arcs name a few thousand sources, and an atomic per
// arc on their counters queues (2.4 ms for the counts and weights of 1.5e7 R-MAT arcs).  A block
// therefore keeps a direct-mapped table in LDS: the first key to reach a slot owns it and is summed
// there, others go to memory at once; the table is added to memory at the end, so a hub costs an
// atomic per block.  Frequent keys reach their slot early and own most of what repeats.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nkpr {

constexpr uint32_t kAggSlots = 2048;   // 32 KB: four blocks of kAggThreads a CU
constexpr int kAggThreads = 512;
constexpr unsigned kAggBlocks = 1024;  // persistent: a table serves m / kAggBlocks arcs
constexpr uint32_t kAggEmpty = 0xFFFFFFFFu;

struct AggTable {
    uint32_t key[kAggSlots];
    uint32_t count[kAggSlots];
    double sum[kAggSlots];

    __device__ __forceinline__ void clear() {
        for (uint32_t i = threadIdx.x; i < kAggSlots; i += kAggThreads) {
            key[i] = kAggEmpty;
            count[i] = 0u;
            sum[i] = 0.0;
        }
        __syncthreads();
    }
    // counts and sums may be nullptr (not wanted); keys lie below 2^31
    __device__ __forceinline__ void add(uint32_t v, double w, uint32_t *counts, double *sums) {
        const uint32_t slot = (v * 2654435761u) >> 21;
        uint32_t k = key[slot];
        if (k == kAggEmpty) {
            k = atomicCAS(&key[slot], kAggEmpty, v);
            if (k == kAggEmpty) k = v;
        }
        if (k == v) {
            if (counts) atomicAdd(&count[slot], 1u);
            if (sums) unsafeAtomicAdd(&sum[slot], w);
        } else {
            if (counts) atomicAdd(&counts[v], 1u);
            if (sums) unsafeAtomicAdd(&sums[v], w);
        }
    }
    __device__ __forceinline__ void flush(uint32_t *counts, double *sums) {
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < kAggSlots; i += kAggThreads) {
            const uint32_t v = key[i];
            if (v == kAggEmpty) continue;
            if (counts) atomicAdd(&counts[v], count[i]);
            if (sums) unsafeAtomicAdd(&sums[v], sum[i]);
        }
    }
};
static_assert(kAggSlots == 1u << (32 - 21), "the hash keeps the top 11 bits");

inline unsigned agg_blocks(uint64_t m) {
    const uint64_t b = (m + kAggThreads - 1) / kAggThreads;
    return (unsigned)(b < 1 ? 1 : (b < kAggBlocks ? b : kAggBlocks));
}

}  // namespace nkpr
