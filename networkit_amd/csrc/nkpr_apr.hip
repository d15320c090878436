// Approximate personalised PageRank by residual pushes (ACL), the kernel of NetworKit's
// ApproximatePageRank (networkit/cpp/scd/ApproximatePageRank.cpp:18-61) and PageRankNibble.
//
// The reference keeps a FIFO queue and pushes one node at a time:
//   push(u): res = r[u]; vol = weightedDegree(u, countSelfLoopsTwice = true);
//            every neighbour v (out-list order) gets mass = (1 - alpha) res w / (2 vol) and is
//            queued when its residual crosses eps vol(v); p[u] += alpha res;
//            r[u] = (1 - alpha) res / 2, queued again when r[u] / vol >= eps.
// Here all queued nodes push at once, round after round (a frontier):
//   first every frontier node's residual is taken (so that mass arriving during the
//   round stays for the next one, whatever the schedule), adding alpha res to p and keeping
//   (1 - alpha) res / 2; then a lane group per node sends the masses with atomic adds; a node whose
//   residual crosses its threshold through an add is appended to the next frontier once (a
//   flag bit per node).
// Residuals are 64-bit fixed point (2^-62 units; the total mass is at most 1), so the atomic
// sums are exact and independent of their order: the frontier of every round, p and r are the
// same on every run, bit for bit (only the order of a frontier's entries varies).  Each sent
// and kept mass is rounded to the nearest unit (at most 2^-63 off, the errors of a run add up
// like a random walk, about sqrt(edge pushes) 2^-63); thresholds are ceil(eps vol 2^62), so
// r < eps vol holds exactly for every residual below 2^-9.
// Every push moves mass as the reference's does, so the ACL identity
// p + pr_alpha(r) = pr_alpha(seeds) and the stopping rule (every residual below eps vol when the
// frontier is empty) hold as in the reference; the push order differs, so p differs from the
// reference's within the bound that rule gives.  The share a self-loop sends back to u is
// dropped, as in the reference (its r[u] = (1 - alpha) res / 2 is an assignment after the
// loop), so on graphs with self-loops the identity holds for the walk without them,
// (I + D^-1 A_offdiag) / 2 with D counting each self-loop twice.
//
// Layout: the graph's out-lists (forNeighborsOf order) as CSR with int32 ids and optional FP64
// weights, vol[z] computed once; p[z] (FP64), r[z] (fixed point), flags[z] (bit 0 touched, bit 1
// queued), two frontier arrays and what each frontier node pushes.  Only the touched entries are cleared
// after a run, so a run costs O(z) only for the scan that lists the touched nodes.
// Algorithmic bytes per push: 4 + 8 (id, weight) and one 8-byte atomic per out-edge, 8 + 8 + 8
// per pushed node.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "nkpr_internal.hpp"

struct nkpr_apr {
    int device = 0;
    hipStream_t stream = nullptr;
    uint64_t z = 0, m = 0;
    nkpr::DevBuf ptr, dst, w, vol;
    nkpr::DevBuf p, r, flags, f0, f1, push, chunks, cnt, out_ids, out_p, out_r, out_cnt, seeds;
    uint64_t chunk_cap = 0;  // entries per heavy chunk list (two lists)
    bool dirty = true;  // p, r, flags hold a run that was not cleared
    uint32_t apart = 0;  // runs still to be made with a launch per part (a wait of the grid expired)
    ~nkpr_apr() {
        nkpr::stream_put(stream, device);
    }
};

namespace nkpr {
namespace {

constexpr uint32_t kTouched = 1, kQueued = 2;
// 512 threads: the grids of four runs (a process has four hardware queues) fit the device together, so
// that none waits for blocks which another keeps out.  1024 took the same time alone (3.29 and 3.35 ms
// a run); four threads share the device at 0.87 ms a run, 1.17 with two launches a round.  More grids
// than four (several processes) may keep each other's blocks out: see kMissing.
constexpr int kPushThreads = 512;
constexpr uint32_t kPushLanes = 32;  // lanes that push one frontier node
// Rounds after which the host looks whether the frontier is empty: of one launch, and of launches
// apart (NKPR_APR_BATCH, 1 to 256, overrides both).
constexpr uint32_t kTogetherRounds = 4096, kApartRounds = 16;
// A wait of the grid for a block that cannot start ends after kMissing (2 s, in units of 10 ns).  The
// run, and the next kApartRuns of the handle, then launch the parts of a round apart, where no block
// waits for another and the device stays full.
constexpr uint64_t kMissing = 200000000;
constexpr uint32_t kApartRuns = 64;
constexpr double kUnit = 4611686018427387904.0;  // 2^62 fixed-point units per unit of mass

// ceil(eps vol 2^62): r < thr  <=>  r 2^-62 < eps vol (the product rounded as the reference's).
// A node without out-edges (vol 0) follows the reference's two tests: a neighbour's add never
// queues it (r[v] < vol eps is false), and as a pushed node (only a seed can be one) it is
// pushed again while any residual is left (r / vol >= eps holds for every r > 0).
__device__ __forceinline__ uint64_t threshold_of(double eps, double vol, bool self) {
    const double t = eps * vol * kUnit;
    if (!(t > 0.0)) return self ? 1ull : ~0ull;
    return t >= 1.8e19 ? ~0ull : (uint64_t)ceil(t);
}

// offsets rising from 0 (ptr[z] = m by construction): bad[0] counts the others
__global__ void apr_check_kernel(const uint64_t *ptr, uint64_t z, uint32_t *bad) {
    for (uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; u < z;
         u += (uint64_t)gridDim.x * blockDim.x)
        if (ptr[u] > ptr[u + 1] || (u == 0 && ptr[0] != 0)) atomicAdd(bad, 1u);
}

__global__ void apr_vol_kernel(const uint64_t *ptr, const int32_t *dst, const double *w,
                               uint64_t z, double *vol, uint32_t *bad) {
    // Graph::weightedDegree(u, countSelfLoopsTwice = true): a wave per node; bad[0] counts
    // weights that are negative or not numbers and ids outside [0, z)
    const int lane = threadIdx.x & 63;
    const uint64_t nw = ((uint64_t)gridDim.x * blockDim.x) >> 6;
    for (uint64_t u = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6; u < z; u += nw) {
        double s = 0.0;
        for (uint64_t e = ptr[u] + lane; e < ptr[u + 1]; e += 64) {
            const double x = w ? w[e] : 1.0;
            const int32_t v = dst[e];
            if (!(x >= 0.0) || v < 0 || (uint64_t)v >= z) atomicAdd(bad, 1u);
            s += (uint64_t)v == u ? 2.0 * x : x;
        }
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) vol[u] = s;
    }
}

__global__ void apr_clear_kernel(double *p, uint64_t *r, uint32_t *flags, uint64_t z) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < z;
         i += (uint64_t)gridDim.x * blockDim.x) {
        p[i] = 0.0;
        r[i] = 0ull;
        flags[i] = 0u;
    }
}

// after a run: clear the entries it touched (listed by the compaction)
__global__ void apr_reset_kernel(const uint32_t *ids, const uint32_t *count, double *p,
                                 uint64_t *r, uint32_t *flags) {
    const uint32_t k = count[0];
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < k; i += gridDim.x * blockDim.x) {
        const uint32_t u = ids[i];
        p[u] = 0.0;
        r[u] = 0ull;
        flags[u] = 0u;
    }
}

// Counters (cnt, a device buffer of uint32).  Round k pushes frontier k & 1 (size cnt[k % 3]) and
// appends to the other frontier array (size cnt[(k + 1) % 3]); its take clears cnt[(k + 2) % 3],
// the size round k - 1 pushed, for round k + 1's appends.  The heavy chunk lists alternate the
// same way (sizes cnt[kCntChunks + (k & 1)]).  [4..5] the out-edges of the pushed nodes, [6..7]
// the pushes, [8] the rounds with a non-empty frontier, [12] set when a wait of the grid barrier
// took too long; from kCntBarrier on the barrier's arrivals, a line per counter.
constexpr int kCntEdges = 4, kCntPushes = 6, kCntRounds = 8, kCntChunks = 10, kCntAbort = 12;
constexpr int kCntBarrier = 32, kBarGroups = 16, kBarStride = 32;
constexpr int kCntWords = kCntBarrier + (kBarGroups + 1) * kBarStride;
// A node with more out-edges than kPushChunk is pushed by several lane groups, kPushChunk edges each.
constexpr uint32_t kPushChunk = 64;

// What the push of a frontier node needs, gathered by the take: the push then starts its
// edge loads after one read instead of three dependent ones.
struct Push {
    uint64_t first;       // its out-edges [first, first + count)
    uint64_t count_node;  // count << 32 | node
    double share;         // (1 - alpha) res / (2 vol): the mass per unit of weight
};

// Accesses to what other blocks of the launch write: coherent between the XCDs' L2 caches.
template <typename T> __device__ __forceinline__ T ld_agent(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ __forceinline__ void st_agent(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Every block arrives before any goes on; `turn` counts the barriers since the counters were
// cleared.  Every thread waits for its own stores first.  Blocks count in kBarGroups groups, whose
// last ones count at the top: 256 adds to one address would queue for longer than the rounds' own
// work.  The grid has a block per CU, all of which are resident once the kernels ahead of them
// have ended; should one still be missing after `ticks` (of 10 ns), the wait ends, every block leaves
// (false) and the run is done again with the parts apart.
__device__ __forceinline__ bool grid_barrier(uint32_t *cnt, uint32_t turn, uint64_t ticks, uint32_t *ok) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t *bar = cnt + kCntBarrier;
        const uint32_t grp = blockIdx.x % kBarGroups;
        const uint32_t members = (gridDim.x - grp + kBarGroups - 1) / kBarGroups;
        const uint32_t all = min(gridDim.x, (uint32_t)kBarGroups) * (turn + 1);
        if (atomicAdd(bar + kBarStride * (1 + grp), 1u) + 1 == members * (turn + 1)) atomicAdd(bar, 1u);
        const uint64_t t0 = wall_clock64();
        uint32_t fine = 1;
        for (uint32_t i = 1; (int32_t)(ld_agent(bar) - all) < 0; ++i) {
            if ((i % 64 == 0 || ticks == 0) && (ld_agent(cnt + kCntAbort) || wall_clock64() - t0 > ticks)) {
                st_agent(cnt + kCntAbort, 1u);
                fine = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        *ok = fine;
    }
    __syncthreads();
    return *ok != 0;
}

// the seeds: residual 1/|seeds|, touched, queued, in frontier 0 (ids ascending)
__global__ void apr_seed_kernel(const uint32_t *seeds, uint32_t k, uint64_t *r, uint32_t *flags,
                                uint32_t *front, uint32_t *cnt) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < k; i += gridDim.x * blockDim.x) {
        const uint32_t s = seeds[i];
        r[s] = (uint64_t)(kUnit / (double)k);
        flags[s] = kTouched | kQueued;
        front[i] = s;
    }
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < kCntWords; i += blockDim.x) cnt[i] = i == 0 ? k : 0u;
}

// Rounds first .. first + rounds - 1, or until a frontier is empty.  A round has two parts with a grid
// barrier after each; with PARTS one of the two, the launch is that part of round `first`.
//
// Take: a thread per frontier node u takes its residual res, adds alpha res to p[u] and leaves
// (1 - alpha) res / 2 in r[u], queueing u again when that alone reaches its threshold; a node with
// more than kPushChunk out-edges lists its chunks.
//
// Push: a lane group per frontier node with at most kPushChunk out-edges and one per chunk of the
// others sends the masses (1 - alpha) res w / (2 vol).  At the start of the push every residual
// lies below its threshold unless its node is already queued, and all adds are positive, so the
// add that crosses a threshold is the one that finds the residual below it and leaves it at or
// above it; that add sets the node's queued bit.  Only an add that finds no residual marks the
// node touched (one that holds some was marked by an earlier add).
//
// Bound by latency: a round is a few thousand edges, some ten dependent accesses of about 1 us
// each.  Two launches a round put some 7 us between every two kernels beside that; the rounds
// therefore share one launch, a block per CU.  The returning add is issued
// before the threshold is formed, so that it and the load of vol[v] are in flight together; a
// block collects what it queues in LDS and takes its places in the next frontier with one add.
// Hyperbolic graph of 2e6 nodes, eps 1e-8, three seeds: 3.76, 2.96 and 2.73 ms a run with two launches a
// round, 3.24, 2.46 and 2.49 now; 64 seeds on 6e6 nodes, eps 1e-9: 18.6 and 16.3 ms (1.1e10 adds
// a second, what the atomics give).
constexpr int kTake = 1, kPush = 2, kRound = kTake | kPush;
template <int PARTS>
__global__ __launch_bounds__(kPushThreads) void apr_rounds_kernel(
    const uint64_t *ptr, const int32_t *dst, const double *w, const double *vol, double alpha, double eps,
    uint32_t *f0, uint32_t *f1, uint32_t *cnt, uint32_t first, uint32_t rounds, double *p, uint64_t *r, uint32_t *flags, Push *push,
    uint64_t *chunks, uint64_t chunk_cap, uint64_t ticks) {
    constexpr uint32_t kGroups = kPushThreads / kPushLanes;
    __shared__ uint32_t list[kPushThreads + kGroups * kPushChunk];
    __shared__ uint32_t n_list, base, ok;
    __shared__ unsigned long long edges;
    // Set already: this block came too late.  One thread asks for the whole block: the word may be set
    // between two waves' reads, and waves that went on without the first one would find n_list, base
    // and edges unset and pass the barriers, which do not count waves that have ended.
    if (threadIdx.x == 0) {
        edges = 0;
        n_list = base = 0;
        ok = ld_agent(cnt + kCntAbort) == 0u;
    }
    __syncthreads();
    if (!ok) return;
    const uint32_t lane = threadIdx.x % kPushLanes;
    // consecutive entries go to different blocks, so that a small frontier uses every CU
    const uint32_t group = threadIdx.x / kPushLanes * gridDim.x + blockIdx.x, ngroups = gridDim.x * kGroups;
    const uint32_t thread = threadIdx.x * gridDim.x + blockIdx.x, nthreads = gridDim.x * kPushThreads;
    // the block's list into the next frontier (every thread calls it)
    auto flush = [&](uint32_t *next, uint32_t *ncnt) {
        __syncthreads();
        const uint32_t k = n_list;
        if (k) {
            if (threadIdx.x == 0) base = atomicAdd(ncnt, k);
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < k; i += kPushThreads) st_agent(next + base + i, list[i]);
            if (threadIdx.x == 0) n_list = 0;
        }
        __syncthreads();
    };
    for (uint32_t round = first; round - first < rounds; ++round) {
        const uint32_t k2 = round & 1, k3 = round % 3;
        const uint32_t *front = k2 ? f1 : f0;
        uint32_t *next = k2 ? f0 : f1, *ncnt = cnt + (k3 + 1) % 3, *hcnt = cnt + kCntChunks + k2;
        uint64_t *chunk = chunks + (k2 ? chunk_cap : 0);
        const uint32_t nf = ld_agent(cnt + k3);
        if constexpr (PARTS & kTake) {
            // (after the last round too: launches apart go on to the end of their batch)
            if (blockIdx.x == 0 && threadIdx.x == 0) {
                st_agent(cnt + (k3 + 2) % 3, 0u);
                st_agent(cnt + kCntChunks + (k2 ^ 1), 0u);
                if (nf) {
                    *reinterpret_cast<unsigned long long *>(cnt + kCntPushes) += nf;
                    cnt[kCntRounds] += 1u;
                }
            }
        }
        if (nf == 0) break;
        if constexpr (PARTS & kTake) {
            for (uint32_t i0 = 0; i0 < nf; i0 += nthreads) {
                const uint32_t i = i0 + thread;
                if (i < nf) {
                    const uint32_t u = ld_agent(front + i);
                    const uint64_t res = ld_agent(r + u), b = ptr[u], deg = ptr[u + 1] - b;
                    const double vu = vol[u], pu = ld_agent(p + u);
                    const double dres = (double)res;
                    const uint64_t keep = __double2ull_rn((1.0 - alpha) * dres / 2);
                    const bool again = keep >= threshold_of(eps, vu, true);
                    st_agent(p + u, pu + alpha * dres / kUnit);
                    st_agent(r + u, keep);
                    st_agent(flags + u, again ? (kTouched | kQueued) : kTouched);
                    Push *o = push + i;
                    st_agent(&o->first, b);
                    st_agent(&o->count_node, deg << 32 | u);
                    st_agent(&o->share, vu > 0.0 ? (1.0 - alpha) * dres / (2.0 * vu) : 0.0);
                    atomicAdd(&edges, (unsigned long long)deg);
                    if (deg > kPushChunk) {
                        const uint32_t nc = (uint32_t)((deg + kPushChunk - 1) / kPushChunk);
                        const uint32_t at = atomicAdd(hcnt, nc);
                        for (uint32_t c = 0; c < nc; ++c) st_agent(chunk + at + c, (uint64_t)c << 32 | i);
                    }
                    if (again) list[atomicAdd(&n_list, 1u)] = u;
                }
                // (the last turn's nodes wait for those of the push)
                if (PARTS == kTake || nf - i0 > nthreads) flush(next, ncnt);
            }
        }
        if constexpr (PARTS == kTake) break;
        if constexpr (PARTS == kRound)
            if (!grid_barrier(cnt, 2 * round, ticks, &ok)) break;
        // the first turn's items are on their way beside the number of chunks
        const uint32_t nh = ld_agent(hcnt);
        uint64_t from = 0, cn = 0;
        double share = 0.0;
        auto load = [&](uint32_t i) {
            from = ld_agent(&push[i].first);
            cn = ld_agent(&push[i].count_node);
            share = ld_agent(&push[i].share);
        };
        if (group < nf) load(group);
        for (uint32_t t0 = 0; t0 < nf + nh; t0 += ngroups) {
            const uint32_t t = t0 + group;
            uint64_t b = 0, end = 0;
            if (t < nf) {
                if (t0) load(t);
                b = from;
                end = cn >> 32 > kPushChunk ? b : b + (cn >> 32);  // the others are pushed by their chunks
            } else if (t < nf + nh) {
                const uint64_t c = ld_agent(chunk + (t - nf));
                load((uint32_t)c);
                b = from + (c >> 32) * kPushChunk;
                end = std::min<uint64_t>(from + (cn >> 32), b + kPushChunk);
            }
            const uint32_t u = (uint32_t)cn;
            for (uint64_t e = b + lane; e < end; e += kPushLanes) {
                const uint32_t v = (uint32_t)dst[e];
                // a self-loop sends nothing: the reference overwrites r[u] after its loop
                if (v == u) continue;
                const uint64_t mass = __double2ull_rn(share * (w ? w[e] : 1.0));
                const uint64_t old = atomicAdd(reinterpret_cast<unsigned long long *>(&r[v]),
                                               (unsigned long long)mass);
                const uint64_t thr = threshold_of(eps, vol[v], false);
                if (old < thr && old + mass >= thr) {
                    if (!(atomicOr(&flags[v], kQueued | kTouched) & kQueued)) list[atomicAdd(&n_list, 1u)] = v;
                } else if (old == 0) {
                    atomicOr(&flags[v], kTouched);
                }
            }
            flush(next, ncnt);
        }
        if constexpr (PARTS == kPush) break;
        if constexpr (PARTS == kRound)
            if (!grid_barrier(cnt, 2 * round + 1, ticks, &ok)) break;
    }
    __syncthreads();
    if (threadIdx.x == 0 && edges)
        atomicAdd(reinterpret_cast<unsigned long long *>(cnt + kCntEdges), edges);
}

// touched nodes in ascending id order: per-block counts, then a one-block scan, then writes
__global__ void apr_count_kernel(const uint32_t *flags, uint64_t z, uint32_t *bc) {
    __shared__ uint32_t s[256];
    const uint64_t per = (z + gridDim.x - 1) / gridDim.x;
    const uint64_t b = (uint64_t)blockIdx.x * per, e = std::min<uint64_t>(z, b + per);
    uint32_t c = 0;
    for (uint64_t i = b + threadIdx.x; i < e; i += blockDim.x) c += (flags[i] & kTouched) ? 1u : 0u;
    s[threadIdx.x] = c;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) s[threadIdx.x] += s[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) bc[blockIdx.x] = s[0];
}

// exclusive sums of the nb (= blockDim.x, a multiple of 64) block counts, one thread each
__global__ void apr_scan_kernel(uint32_t *bc, uint32_t nb, uint32_t *total) {
    __shared__ uint32_t wsum[16];
    const uint32_t t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const uint32_t c = t < nb ? bc[t] : 0u;
    uint32_t x = c;  // inclusive scan inside the wave
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if ((int)lane >= o) x += y;
    }
    if (lane == 63) wsum[wv] = x;
    __syncthreads();
    if (t == 0) {
        uint32_t acc = 0;
        for (uint32_t i = 0; i < blockDim.x / 64; ++i) {
            const uint32_t v = wsum[i];
            wsum[i] = acc;
            acc += v;
        }
        total[0] = acc;
    }
    __syncthreads();
    if (t < nb) bc[t] = wsum[wv] + x - c;
}

__global__ void apr_compact_kernel(const uint32_t *flags, const double *p, const uint64_t *r,
                                   uint64_t z, const uint32_t *bc, uint32_t *ids, double *op,
                                   double *orr) {
    // one block per range; the range is walked in order 256 slots at a time
    __shared__ uint32_t s[256];
    __shared__ uint32_t base;
    const uint64_t per = (z + gridDim.x - 1) / gridDim.x;
    const uint64_t b = (uint64_t)blockIdx.x * per, e = std::min<uint64_t>(z, b + per);
    if (threadIdx.x == 0) base = bc[blockIdx.x];
    __syncthreads();
    for (uint64_t c0 = b; c0 < e; c0 += blockDim.x) {
        const uint64_t i = c0 + threadIdx.x;
        const uint32_t t = (i < e && (flags[i] & kTouched)) ? 1u : 0u;
        s[threadIdx.x] = t;
        __syncthreads();
        // inclusive scan in LDS (Hillis-Steele)
        for (int o = 1; o < 256; o <<= 1) {
            const uint32_t add = (int)threadIdx.x >= o ? s[threadIdx.x - o] : 0u;
            __syncthreads();
            s[threadIdx.x] += add;
            __syncthreads();
        }
        if (t) {
            const uint32_t at = base + s[threadIdx.x] - 1;
            ids[at] = (uint32_t)i;
            op[at] = p[i];
            orr[at] = (double)r[i] / kUnit;
        }
        __syncthreads();
        if (threadIdx.x == 0) base += s[255];
        __syncthreads();
    }
}

}  // namespace

void apr_create_impl(uint64_t z, const uint64_t *ptr, const int32_t *dst, const double *w,
                     int32_t device_ptrs, nkpr_apr **out) {
    NKPR_CHECK(out != nullptr, "out is NULL");
    NKPR_CHECK(z > 0 && z < 0x7FFFFFFFull, "the graph needs 1 .. 2^31 - 2 slots");
    NKPR_CHECK(ptr != nullptr, "ptr is NULL");
    std::unique_ptr<nkpr_apr> a(new nkpr_apr());
    NKPR_HIP(hipGetDevice(&a->device));
    a->stream = stream_get();
    const hipStream_t s = a->stream;
    const hipMemcpyKind kind = device_ptrs ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    uint64_t m = 0;
    if (device_ptrs) read_back(s, {{&m, ptr + z, 8}});
    else m = ptr[z];
    NKPR_CHECK(m == 0 || dst != nullptr, "dst is NULL");
    a->z = z;
    a->m = m;
    a->ptr.alloc(8 * (z + 1));
    a->dst.alloc(4 * std::max<uint64_t>(m, 1));
    NKPR_HIP(hipMemcpyAsync(a->ptr.p, ptr, 8 * (z + 1), kind, s));
    if (m) NKPR_HIP(hipMemcpyAsync(a->dst.p, dst, 4 * m, kind, s));
    if (w && m) {
        a->w.alloc(8 * m);
        NKPR_HIP(hipMemcpyAsync(a->w.p, w, 8 * m, kind, s));
    }
    a->vol.alloc(8 * z);
    a->p.alloc(8 * z);
    a->r.alloc(8 * z);
    a->flags.alloc(4 * z);
    a->f0.alloc(4 * z);
    a->f1.alloc(4 * z);
    a->push.alloc(sizeof(Push) * z);
    // chunks of the nodes with more than kPushChunk out-edges: at most 2 deg / kPushChunk per node
    a->chunk_cap = 2 * m / kPushChunk + 64;
    a->chunks.alloc(2 * 8 * a->chunk_cap);
    a->cnt.alloc(4 * kCntWords);
    a->out_cnt.alloc(4 * 1025);
    a->out_ids.alloc(4 * z);
    a->out_p.alloc(8 * z);
    a->out_r.alloc(8 * z);
    NKPR_HIP(hipMemsetAsync(a->cnt.p, 0, 64, s));
    hipLaunchKernelGGL(apr_check_kernel, dim3((unsigned)std::min<uint64_t>((z + 255) / 256, 65536)),
                       dim3(256), 0, s, a->ptr.as<uint64_t>(), z, a->cnt.as<uint32_t>());
    NKPR_HIP(hipGetLastError());
    uint32_t bad = 0;
    read_back(s, {{&bad, a->cnt.p, 4}});
    NKPR_CHECK(bad == 0, "offsets must rise from 0 to the number of entries");
    hipLaunchKernelGGL(apr_vol_kernel, dim3((unsigned)std::min<uint64_t>((z * 64 + 255) / 256, 65536)),
                       dim3(256), 0, s, a->ptr.as<uint64_t>(), a->dst.as<int32_t>(),
                       a->w.as<double>(), z, a->vol.as<double>(), a->cnt.as<uint32_t>());
    NKPR_HIP(hipGetLastError());
    // the host arrays may be released when this returns
    read_back(s, {{&bad, a->cnt.p, 4}});
    NKPR_CHECK(bad == 0, "neighbour ids must lie in [0, z) and weights must be non-negative");
    *out = a.release();
}

void apr_destroy_impl(nkpr_apr *a) { delete a; }

int apr_device(const nkpr_apr *a) { return a->device; }

void apr_run_impl(nkpr_apr *a, double alpha, double eps, const uint64_t *seeds, uint64_t nseeds,
                  uint64_t *count, int64_t *ids_out, double *p_out, double *r_out,
                  nkpr_apr_stats *st) {
    const auto t0 = std::chrono::steady_clock::now();
    NKPR_CHECK(a != nullptr, "handle is NULL");
    NKPR_CHECK(seeds != nullptr && nseeds > 0, "at least one seed is needed");
    NKPR_CHECK(count != nullptr, "count is NULL");
    NKPR_CHECK(alpha > 0.0 && alpha <= 1.0, "alpha must lie in (0, 1]");
    NKPR_CHECK(eps > 0.0, "epsilon must be > 0");
    // std::set<node>: ids ascending, no repeats
    std::vector<uint32_t> sd;
    sd.reserve(nseeds);
    for (uint64_t i = 0; i < nseeds; ++i) {
        NKPR_CHECK(seeds[i] < a->z, "seed id out of range");
        sd.push_back((uint32_t)seeds[i]);
    }
    std::sort(sd.begin(), sd.end());
    sd.erase(std::unique(sd.begin(), sd.end()), sd.end());
    const hipStream_t s = a->stream;
    const uint64_t z = a->z;
    a->seeds.alloc(4 * sd.size());
    NKPR_HIP(hipMemcpyAsync(a->seeds.p, sd.data(), 4 * sd.size(), hipMemcpyHostToDevice, s));
    // The rounds of a launch end by themselves when a frontier is empty.  Its blocks wait for each
    // other, one per CU.
    uint64_t ticks = kMissing;
    // test hook: 0 ends a wait that is not over at once
    if (const char *e = std::getenv("NKPR_TEST_APR_WAIT"); e && *e) ticks = std::strtoull(e, nullptr, 10);
    uint32_t together = kTogetherRounds, batch = kApartRounds;
    if (const char *e = std::getenv("NKPR_APR_BATCH"))
        together = batch = (uint32_t)std::max(1, std::min(256, std::atoi(e)));
    int cus = 0;
    NKPR_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, a->device));
    const unsigned grid = (unsigned)std::max(cus, 1);
    uint32_t host_cnt[16] = {0}, round = 0;
    auto start = [&] {
        if (a->dirty) {
            const unsigned gz = (unsigned)std::min<uint64_t>((z + 255) / 256, 65536);
            hipLaunchKernelGGL(apr_clear_kernel, dim3(gz), dim3(256), 0, s, a->p.as<double>(),
                               a->r.as<uint64_t>(), a->flags.as<uint32_t>(), z);
        }
        a->dirty = true;
        hipLaunchKernelGGL(apr_seed_kernel, dim3(1), dim3(256), 0, s, a->seeds.as<uint32_t>(),
                           (uint32_t)sd.size(), a->r.as<uint64_t>(), a->flags.as<uint32_t>(),
                           a->f0.as<uint32_t>(), a->cnt.as<uint32_t>());
        round = 0;
    };
    auto launch = [&](auto kernel, unsigned blocks, uint32_t rounds) {
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kPushThreads), 0, s, a->ptr.as<uint64_t>(),
                           a->dst.as<int32_t>(), a->w.as<double>(), a->vol.as<double>(), alpha, eps,
                           a->f0.as<uint32_t>(), a->f1.as<uint32_t>(), a->cnt.as<uint32_t>(), round, rounds,
                           a->p.as<double>(), a->r.as<uint64_t>(), a->flags.as<uint32_t>(), a->push.as<Push>(),
                           a->chunks.as<uint64_t>(), a->chunk_cap, ticks);
        NKPR_HIP(hipGetLastError());
    };
    start();
    bool apart = a->apart > 0;
    if (apart) --a->apart;
    for (;;) {
        if (apart) {
            for (uint32_t k = 0; k < batch; ++k, ++round) {
                launch(apr_rounds_kernel<kTake>, 4 * grid, 1);
                launch(apr_rounds_kernel<kPush>, 4 * grid, 1);
            }
        } else {
            launch(apr_rounds_kernel<kRound>, grid, together);
        }
        read_back(s, {{host_cnt, a->cnt.p, sizeof(host_cnt)}});
        if (host_cnt[kCntAbort]) {
            apart = true;
            a->apart = kApartRuns;
            start();
            continue;
        }
        if (!apart) round = host_cnt[kCntRounds];
        if (host_cnt[round % 3] == 0) break;  // the frontier of the next round is empty
    }
    uint64_t rounds = host_cnt[kCntRounds], pushes = 0;
    std::memcpy(&pushes, host_cnt + kCntPushes, 8);
    // the touched nodes, ascending
    const unsigned nbk = 1024;
    hipLaunchKernelGGL(apr_count_kernel, dim3(nbk), dim3(256), 0, s, a->flags.as<uint32_t>(), z,
                       a->out_cnt.as<uint32_t>());
    hipLaunchKernelGGL(apr_scan_kernel, dim3(1), dim3(nbk), 0, s, a->out_cnt.as<uint32_t>(), nbk,
                       a->out_cnt.as<uint32_t>() + nbk);
    hipLaunchKernelGGL(apr_compact_kernel, dim3(nbk), dim3(256), 0, s, a->flags.as<uint32_t>(),
                       a->p.as<double>(), a->r.as<uint64_t>(), z, a->out_cnt.as<uint32_t>(),
                       a->out_ids.as<uint32_t>(), a->out_p.as<double>(), a->out_r.as<double>());
    hipLaunchKernelGGL(apr_reset_kernel, dim3(1024), dim3(256), 0, s, a->out_ids.as<uint32_t>(),
                       a->out_cnt.as<uint32_t>() + nbk, a->p.as<double>(), a->r.as<uint64_t>(),
                       a->flags.as<uint32_t>());
    NKPR_HIP(hipGetLastError());
    uint32_t k = 0;
    read_back(s, {{&k, a->out_cnt.as<uint32_t>() + nbk, 4}});
    a->dirty = false;
    *count = k;
    if (ids_out || p_out || r_out) {
        std::vector<uint32_t> ids(k);
        read_back(s, {{ids.data(), a->out_ids.p, ids_out ? 4 * (size_t)k : 0},
                      {p_out, a->out_p.p, p_out ? 8 * (size_t)k : 0},
                      {r_out, a->out_r.p, r_out ? 8 * (size_t)k : 0}});
        if (ids_out)
            for (uint32_t i = 0; i < k; ++i) ids_out[i] = (int64_t)ids[i];
    }
    if (st) {
        uint64_t ep = 0;
        std::memcpy(&ep, host_cnt + kCntEdges, 8);
        st->edge_pushes = ep;
        st->rounds = rounds;
        st->pushes = pushes;
        st->touched = k;
        st->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    }
}

}  // namespace nkpr
