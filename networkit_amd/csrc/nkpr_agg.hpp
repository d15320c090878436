// Sums per key over a stream of (key, weight) pairs whose keys may repeat very unevenly: the
// out-degrees of a graph's arcs.  Atomics on one address queue: with an atomic per arc, half of
// 1.7e7 arcs leaving one source took 103 ms, and 90% of them leaving 100 sources 3.9 ms.  A block
// therefore keeps a direct-mapped table in LDS: the first key to reach a slot owns it and is summed
// there, others go to memory at once; the table is added to memory at the end, so a hub costs an
// atomic per block: 0.7 and 0.2 ms for these two.
//
// What the table does not do is save atomics where hubs are many: of the arcs of an R-MAT graph four
// in five name a source that owns no slot, and the kernel takes what the atomics take, about
// 1.1e10 a second (counts and weights of 1.5e7 arcs: 2.5 to 3.2 ms with an atomic per arc, 2.4
// now; of 5e8 arcs 71 and 74 ms; uniform sources 1.33 both).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace nkpr {

constexpr uint32_t kAggSlots = 2048;   // 32 KB: four blocks of kAggThreads a CU
constexpr int kAggThreads = 512;
constexpr unsigned kAggBlocks = 1024;  // persistent, at most (see agg_blocks)
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

// Blocks for m arcs.  A table is emptied into memory at the end, up to kAggSlots atomics a block, so few
// arcs a block cost more than an atomic per arc; a block per CU comes before that.  Weights of R-MAT
// graphs in us, atomic per arc / blocks of 512 arcs / this rule: 1.4e5 arcs 38 / 43 / 27, 5.8e5
// 115 / 142 / 74, 1.7e6 273 / 231 / 180.
constexpr uint64_t kAggFewArcs = 1024, kAggArcs = 4096;
constexpr uint64_t kAggFewBlocks = 256;
inline unsigned agg_blocks(uint64_t m) {
    uint64_t b = (m + kAggFewArcs - 1) / kAggFewArcs;
    if (b > kAggFewBlocks) b = std::max(kAggFewBlocks, (m + kAggArcs - 1) / kAggArcs);
    return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(b, kAggBlocks));
}

}  // namespace nkpr
