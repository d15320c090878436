// Graph upload and preprocessing: the device-side half of "export the Graph to CSC".
//
// Input: the in-lists NetworKit's PageRank iterates (Graph::forInEdgesOf,
// include/networkit/graph/Graph.hpp:1918-1938) as CSC, optional weights, optional exists[]
// and optional weighted out-degrees (Graph::weightedDegree, networkit/cpp/graph/Graph.cpp:
// 427-455,539).  Output layout in HBM (compact ids 0..n-1 over existing nodes):
//   - nodes relabelled by out-degree, descending (ties by slot id): the sources gathered most
//     often form a dense prefix of the gathered vector (cache reuse in L2 / Infinity Cache)
//     and the nodes without out-edges form the tail [sink_begin, n), so the sink mass is a
//     range sum and needs no per-node flag;
//   - colptr (uint64) over the relabelled rows, every in-list sorted by the new source id;
//   - weighted graphs: folded coefficients w_vu / deg_v in FP32 and FP64 (one stream per
//     edge instead of a weight stream plus a degree gather);
//   - unweighted graphs: 1/deg per node in FP32 and FP64 (the sweep prescales x instead);
//   - the sweep schedule (work items, see nkpr_internal.hpp).
#include <hip/hip_runtime.h>

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

#include "nkpr_agg.hpp"
#include "nkpr_internal.hpp"

namespace nkpr {
namespace {

inline unsigned blocks_for(uint64_t n, int t = 256) { return (unsigned)((n + t - 1) / t); }

// validation flags
constexpr uint32_t kBadSrc = 1, kBadPtr = 2, kBadExists = 4, kBadGroup = 8;
constexpr uint32_t kNotUnitDegree = 16;  // not an error: some node's given out-degree is not 1

// Sets kNotUnitDegree in *flags when deg[i] != 1 for an existing i < count (exists may be NULL).
__global__ void unit_degree_kernel(const double *deg, uint64_t count, const uint8_t *exists,
                                   uint32_t *flags) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (uint64_t)gridDim.x * blockDim.x)
        if ((!exists || exists[i]) && deg[i] != 1.0) atomicOr(flags, kNotUnitDegree);
}

__global__ void validate_ptr_kernel(const uint64_t *colptr, uint64_t z, uint64_t m,
                                    const uint8_t *exists, uint32_t *flags) {
    const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= z) return;
    const uint64_t b = colptr[u], e = colptr[u + 1];
    if (e < b || e > m) atomicOr(flags, kBadPtr);
    if (exists && !exists[u] && e != b) atomicOr(flags, kBadExists);
}

// Out-degrees and (wdeg given) weighted out-degrees of the arcs' sources.
__global__ __launch_bounds__(kAggThreads) void out_degree_kernel(const int32_t *src, uint64_t m, uint64_t z,
                                                                 const uint8_t *exists, const float *w,
                                                                 const double *w64, uint32_t *outcnt,
                                                                 double *wdeg, uint32_t *flags) {
    __shared__ AggTable agg;
    agg.clear();
    for (uint64_t e = (uint64_t)blockIdx.x * kAggThreads + threadIdx.x; e < m;
         e += (uint64_t)gridDim.x * kAggThreads) {
        const int32_t v = src[e];
        if (v < 0 || (uint64_t)v >= z || (exists && !exists[v])) {
            atomicOr(flags, kBadSrc);
            continue;
        }
        agg.add((uint32_t)v, wdeg ? (w64 ? w64[e] : (w ? (double)w[e] : 1.0)) : 0.0, outcnt, wdeg);
    }
    agg.flush(outcnt, wdeg);
}

__global__ void relabel_keys_kernel(const uint32_t *outcnt, const uint8_t *exists, uint64_t z,
                                    uint32_t *keys, int32_t *vals) {
    const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= z) return;
    const bool ex = !exists || exists[u];
    // ascending sort of keys == descending out-degree; deleted slots last
    keys[u] = ex ? (0xFFFFFFFEu - outcnt[u]) : 0xFFFFFFFFu;
    vals[u] = (int32_t)u;
}

// Graph of every slot of a batch: the group whose slot range [off[g], off[g+1]) holds it.
__global__ void group_id_kernel(const uint64_t *off, uint32_t groups, uint64_t z, uint32_t *gid) {
    const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= z) return;
    uint32_t lo = 0, hi = groups;  // last g with off[g] <= u
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (off[mid] <= u) lo = mid;
        else hi = mid;
    }
    gid[u] = lo;
}

// Batch relabelling: graph id first, then out-degree descending, deleted slots last.
__global__ void group_keys_kernel(const uint32_t *outcnt, const uint8_t *exists,
                                  const uint32_t *gid, uint32_t groups, uint64_t z,
                                  uint64_t *keys, int32_t *vals, uint32_t *cnt_exist,
                                  uint32_t *cnt_nonsink) {
    const uint64_t u = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= z) return;
    const bool ex = !exists || exists[u];
    keys[u] = ex ? (((uint64_t)gid[u] << 32) | (0xFFFFFFFEu - outcnt[u]))
                 : (((uint64_t)groups << 32) | 0xFFFFFFFFu);
    vals[u] = (int32_t)u;
    if (ex) {
        atomicAdd(&cnt_exist[gid[u]], 1u);
        if (outcnt[u] > 0) atomicAdd(&cnt_nonsink[gid[u]], 1u);
    }
}

// Every in-edge must stay inside its graph.
__global__ void group_edges_kernel(const uint64_t *colptr, const int32_t *src, const uint32_t *gid,
                                   uint64_t z, uint32_t *flags) {
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t nwaves = ((uint64_t)gridDim.x * blockDim.x) >> 6;
    for (uint64_t r = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6; r < z; r += nwaves) {
        const uint32_t g = gid[r];
        for (uint64_t i = colptr[r] + lane; i < colptr[r + 1]; i += 64)
            if (gid[src[i]] != g) atomicOr(flags, kBadGroup);
    }
}

// Existing nodes and those with out-edges: one atomic per block on either count.
__global__ __launch_bounds__(256) void count_kernel(const uint32_t *outcnt, const uint8_t *exists, uint64_t z,
                                                    unsigned long long *n_exist,
                                                    unsigned long long *n_nonsink) {
    __shared__ uint32_t s_cnt[2];
    if (threadIdx.x < 2) s_cnt[threadIdx.x] = 0;
    __syncthreads();
    uint32_t ne = 0, ns = 0;
    for (uint64_t u = (uint64_t)blockIdx.x * 256 + threadIdx.x; u < z; u += (uint64_t)gridDim.x * 256) {
        const bool ex = !exists || exists[u];
        ne += ex ? 1u : 0u;
        ns += ex && outcnt[u] > 0 ? 1u : 0u;
    }
    for (int off = 32; off > 0; off >>= 1) {
        ne += __shfl_xor(ne, off, 64);
        ns += __shfl_xor(ns, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&s_cnt[0], ne);
        atomicAdd(&s_cnt[1], ns);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicAdd(n_exist, (unsigned long long)s_cnt[0]);
        atomicAdd(n_nonsink, (unsigned long long)s_cnt[1]);
    }
}

// Edges from the first `count` relabelled sources (one block).
__global__ __launch_bounds__(1024) void hub_edges_kernel(const int32_t *perm, uint32_t count, const uint32_t *outcnt,
                                                         unsigned long long *sum) {
    unsigned long long mine = 0;
    for (uint32_t r = threadIdx.x; r < count; r += 1024) mine += outcnt[perm[r]];
    for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(sum, mine);
}

__global__ void iperm_kernel(const int32_t *perm, uint32_t n, int32_t *iperm) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n) iperm[perm[r]] = (int32_t)r;
}

__global__ void new_lengths_kernel(const int32_t *perm, uint32_t n, const uint64_t *colptr_in,
                                   uint64_t *len) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n) {
        const int32_t o = perm[r];
        len[r] = colptr_in[o + 1] - colptr_in[o];
    } else if (r == n) {
        len[r] = 0;
    }
}

// Slice of an in-edge of sliced row j from source v.  Sources ranked below `rep` (the most
// gathered ones; relabelled ids are out-degree ranks) are cached by every XCD and their edges
// are spread over the slices by row, which keeps the slices balanced and keeps the requests
// for the hottest lines off a single L2 channel; every other source belongs to one slice by
// its 32-id line group.
__device__ __forceinline__ uint32_t slice_of(uint32_t v, uint64_t j, uint32_t rep, uint32_t S) {
    return (v < rep) ? (uint32_t)(j % S) : ((v >> kSliceShift) % S);
}

// Place of every old row in the sweep's lists: its index, with kSlicedRow set for sliced rows.
constexpr uint32_t kSlicedRow = 0x80000000u;
__global__ void row_place_kernel(const int32_t *perm, const uint32_t *rows, uint32_t count, uint32_t flag,
                                 uint32_t *place) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < count) place[perm[rows[j]]] = j | flag;
}

// Sort key of every edge: (segment << vbits) | new source, value = old edge index.  A segment is a
// direct row, or a sliced row's part in one slice; they are numbered in the order of the sweep
// (direct rows, then slice by slice), so that one stable sort leaves the edges where the sweep reads
// them, by source within a segment.
//
// A block takes kKeyTile consecutive edges and looks its rows up in the offsets: a wave per row
// left most lanes without an edge (R-MAT, 1.5e7 arcs: 0.73 ms, and 2.8 ms more for a second
// pair of row-wise kernels that moved the sorted edges into slices; now 0.19 ms).
constexpr uint32_t kKeyTile = 2048;
__global__ __launch_bounds__(256) void edge_keys_kernel(const uint64_t *colptr_in, const int32_t *src_in, uint64_t m,
                                                        const int32_t *iperm, const uint32_t *place, uint64_t z,
                                                        uint32_t n_d, uint32_t n_s, uint32_t S, uint32_t rep,
                                                        int vbits, uint64_t *keys, uint32_t *vals) {
    __shared__ uint64_t s_row[2];
    const uint64_t e0 = (uint64_t)blockIdx.x * kKeyTile, e1 = std::min<uint64_t>(e0 + kKeyTile, m);
    if (threadIdx.x < 2) s_row[threadIdx.x] = row_of(colptr_in, 0, z, threadIdx.x ? e1 - 1 : e0);
    __syncthreads();
    const uint64_t r0 = s_row[0], r1 = s_row[1] + 1;
    for (uint64_t i = e0 + threadIdx.x; i < e1; i += 256) {
        const uint32_t v = (uint32_t)iperm[src_in[i]];
        const uint32_t at = place[row_of(colptr_in, r0, r1, i)], j = at & ~kSlicedRow;
        const uint64_t seg = (at & kSlicedRow) ? n_d + (uint64_t)slice_of(v, j, rep, S) * n_s + j : j;
        keys[i] = (seg << vbits) | v;
        vals[i] = (uint32_t)i;
    }
}

// First edge of every (slice, sliced row) segment, from the sorted keys; ptr[count] = m.
__global__ void segment_starts_kernel(const uint64_t *keys, uint64_t m, int vbits, uint64_t first, uint64_t count,
                                      uint32_t *ptr) {
    for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k <= count;
         k += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t key = (first + k) << vbits;
        uint64_t lo = 0, hi = k == count ? 0 : m;
        if (k == count) lo = m;
        while (lo < hi) {
            const uint64_t mid = (lo + hi) / 2;
            if (keys[mid] < key) lo = mid + 1;
            else hi = mid;
        }
        ptr[k] = (uint32_t)lo;
    }
}

// kCap entries of padding after the last edge
__global__ void pad_kernel(int32_t *src, float *c32, double *c64) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    src[i] = 0;
    if (c32) c32[i] = 0.0f;
    if (c64) c64[i] = 0.0;
}

__global__ void edge_output_kernel(const uint64_t *keys, const uint32_t *vals, uint64_t m, uint64_t vmask,
                                   const float *w_in, const double *w64_in, const int32_t *src_in,
                                   const double *wdeg, int32_t *src_out, float *coef32,
                                   double *coef64) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m;
         i += (uint64_t)gridDim.x * blockDim.x) {
        src_out[i] = (int32_t)(keys[i] & vmask);
        if (coef32) {
            const uint32_t o = vals[i];
            const double w = w64_in ? w64_in[o] : (double)w_in[o];
            const double c = w / wdeg[src_in[o]];
            coef64[i] = c;
            coef32[i] = (float)c;
        }
    }
}

__global__ void inv_degree_kernel(const int32_t *perm, uint32_t n, const uint32_t *outcnt,
                                  const double *wdeg, double *inv64, float *inv32, double *deg64) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const double d = wdeg[perm[r]], v = (outcnt[perm[r]] > 0) ? 1.0 / d : 0.0;
    inv64[r] = v;
    if (deg64) deg64[r] = d;
    if (inv32) inv32[r] = (float)v;
}

// flag = 1 when some FP64 weight is not the FP32 weight given beside it.  Each thread keeps its
// own result over a grid-stride loop; one atomic per block at most (the grid is capped by the
// launcher), so a graph whose weights all differ does not serialise on one address.
__global__ void fp32_exact_kernel(const float *w, const double *w64, uint64_t m, uint32_t *flag) {
    int diff = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m;
         i += (uint64_t)gridDim.x * blockDim.x)
        diff |= (double)w[i] != w64[i];
    if (__syncthreads_or(diff) && threadIdx.x == 0) atomicOr(flag, 1u);
}

// invw64[u] = 1 / deg[u] (compact order; 0 for nodes without out-weight)
__global__ void inv_of_kernel(const double *deg, uint32_t n, double *invw64) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n) invw64[r] = deg[r] > 0.0 ? 1.0 / deg[r] : 0.0;
}

// ---- schedule, on the device ----------------------------------------------------------------

struct DirectRow {  // rows of at most dmax in-edges (want), or the others
    const uint64_t *colptr;
    uint64_t dmax;
    bool want;
    __device__ bool operator()(uint32_t r) const { return (colptr[r + 1] - colptr[r] <= dmax) == want; }
};

__global__ void row_length_kernel(const uint64_t *colptr, const uint32_t *rows, uint32_t count, uint32_t *len) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < count) len[k] = (uint32_t)(colptr[rows[k] + 1] - colptr[rows[k]]);
    else if (k == count) len[k] = 0;
}

__global__ __launch_bounds__(256) void max_length_kernel(const uint64_t *colptr, uint32_t n, unsigned long long *most) {
    unsigned long long mine = 0;
    for (uint64_t r = (uint64_t)blockIdx.x * 256 + threadIdx.x; r < n; r += (uint64_t)gridDim.x * 256)
        mine = std::max<unsigned long long>(mine, colptr[r + 1] - colptr[r]);
    for (int off = 32; off > 0; off >>= 1) mine = std::max<unsigned long long>(mine, __shfl_xor(mine, off, 64));
    if ((threadIdx.x & 63) == 0 && mine) atomicMax(most, mine);
}

// Row segments of more than kCap in-edges, in no order: {index over all slices, first edge, length}.
__global__ void heavy_rows_kernel(const uint32_t *ptr, uint64_t count, uint32_t *n_heavy, uint4 *heavy) {
    for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < count;
         j += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t b = ptr[j], len = ptr[j + 1] - b;
        if (len > (uint32_t)kCap) heavy[atomicAdd(n_heavy, 1u)] = make_uint4((uint32_t)j, b, len, 0u);
    }
}

// Greedy work items over the rows of `lists` lists of nrows rows each (list q's in-edge offsets start
// at ptr[q nrows]): runs of consecutive rows with at most `cap` in-edges and kRowsMax rows (a row with
// more has an item of its own); rows longer than kCap are left out (see build_heavy).  A wave takes
// seg_rows rows of a list, 64 row ends at a time in its lanes, the next 64 on their way: cuts cost no
// memory access (a load per cut took 1.1 us, 0.29 ms for 256 rows that each fill an item).  Without
// `items` it only counts.
__global__ __launch_bounds__(256) void build_items_kernel(const uint32_t *ptr, uint32_t nrows, uint32_t lists,
                                                          uint32_t segs, uint32_t seg_rows, uint32_t cap,
                                                          uint32_t *counts, const uint32_t *first, uint4 *items) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t seg = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (seg >= lists * segs) return;
    const uint32_t *P = ptr + (uint64_t)(seg / segs) * nrows;
    const uint32_t begin = (seg % segs) * seg_rows, end = min(nrows, begin + seg_rows);
    const uint32_t at = items ? first[seg] : 0;
    uint32_t made = 0;
    auto put = [&](uint32_t r0, uint32_t r1, uint32_t p0, uint32_t p1) {
        if (items && lane == 0) items[at + made] = make_uint4(r0, r1, p0, p1 - p0);
        ++made;
    };
    // the item that grows: rows [r, ..) from edge p0 on; pw the first edge of the window
    uint32_t r = begin, p0 = P[begin], pw = p0, ahead = P[min(begin + lane + 1, end)];
    for (uint32_t w = begin; w < end; w += 64) {
        const uint32_t e = ahead, wend = min(w + 64, end);
        ahead = P[min(w + 64 + lane + 1, end)];
        while (r < wend) {
            const uint32_t j = w + lane, from = max(r, w);
            const uint32_t next =
                from + (uint32_t)__popcll(__ballot(j >= from && j < wend && e - p0 <= cap && j + 1 - r <= (uint32_t)kRowsMax));
            if (next == wend && wend < end) break;  // may grow into the next window
            if (next > r) {
                const uint32_t p1 = next == w ? pw : __shfl(e, next - 1 - w, 64);
                put(r, next, p0, p1);
                r = next;
                p0 = p1;
            } else {
                const uint32_t p1 = __shfl(e, r - w, 64);
                if (p1 - p0 <= (uint32_t)kCap) put(r, r + 1, p0, p1);
                ++r;
                p0 = p1;
            }
        }
        pw = __shfl(e, 63, 64);
    }
    if (!items && lane == 0) counts[seg] = made;
}

__global__ void split_flag_kernel(const uint32_t *rows, uint32_t count, uint8_t *flag) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) flag[rows[i]] = 1;
}

struct SplitRec {
    uint32_t first[kSlices];
    uint32_t count[kSlices];
};

// Items of the rows longer than kCap of one slice: vector items, and split chunks (recorded in
// `splits`) above kVectorMax; the chunks first.  rows: {row, first edge, length}, by row.
void build_heavy(const std::vector<uint4> &rows, uint32_t slice, std::vector<uint4> &out, uint32_t &split_slots,
                 std::map<uint32_t, SplitRec> &splits) {
    std::vector<uint4> vec;
    for (const uint4 &h : rows) {
        if (h.z <= kVectorMax) {
            vec.push_back(make_uint4(h.x, h.x + 1, h.y, h.z));
            continue;
        }
        const uint32_t chunks = (h.z + kChunk - 1) / kChunk;
        SplitRec &rec = splits[h.x];
        rec.first[slice] = split_slots;
        rec.count[slice] = chunks;
        for (uint32_t c = 0; c < chunks; ++c)
            out.push_back(make_uint4(h.x, split_slots++ | kSplitFlag, h.y + c * kChunk,
                                     std::min(kChunk, h.z - c * kChunk)));
    }
    out.insert(out.end(), vec.begin(), vec.end());
}

template <typename V> void upload(nkpr_graph *g, nkpr::DevBuf &b, const std::vector<V> &h) {
    b.alloc(sizeof(V) * std::max<size_t>(h.size(), 1));
    if (!h.empty())
        NKPR_HIP(hipMemcpyAsync(b.p, h.data(), sizeof(V) * h.size(), hipMemcpyHostToDevice,
                                g->stream));
}

uint32_t env_u32(const char *name, uint32_t dflt) {
    const char *v = std::getenv(name);
    if (!v || !*v) return dflt;
    return (uint32_t)std::strtoul(v, nullptr, 10);
}

// Splits the rows of g->colptr into direct and sliced ones, in the order in which a sweep takes
// them; the in-edges are then sorted into that order.  sel: 32 cleared bytes for the counts of direct
// and sliced rows and, 16 bytes on, the largest in-degree.  Reads hub_edges back along the way.
void schedule_rows(nkpr_graph *g, uint32_t *sel, const unsigned long long *hub_edges) {
    const hipStream_t s = g->stream;
    const uint32_t n = g->n;
    // slicing pays off once the gathered vector outgrows one L2; below that everything is
    // direct.  NKPR_SLICES (1 or 8) and NKPR_DIRECT_MAX_DEG override the defaults.
    // (the rows of a batch's graph gather from that graph's part of it alone: a union of 160
    // graphs, 1.3e6 nodes, takes 2.76 instead of 3.54 ms per solve unsliced)
    uint32_t reach = n;
    if (g->n_groups) {
        reach = 0;
        for (uint32_t q = 0; q < g->n_groups; ++q) reach = std::max(reach, g->goff[q + 1] - g->goff[q]);
    }
    uint32_t S = (reach >= (1u << 20)) ? (uint32_t)kSlices : 1u;
    S = env_u32("NKPR_SLICES", S);
    NKPR_CHECK(S == 1 || S == (uint32_t)kSlices, "NKPR_SLICES must be 1 or 8");
    uint32_t dmax = (S == 1) ? (uint32_t)kCap : kDefaultDirectMaxDeg;
    dmax = std::min<uint32_t>(env_u32("NKPR_DIRECT_MAX_DEG", dmax), (uint32_t)kCap);
    const uint32_t rep = env_u32("NKPR_SLICE_REPLICATE", kDefaultSliceReplicate);
    g->n_slices = S;
    g->direct_max_deg = dmax;

    // direct and sliced rows, the direct rows' offsets and the largest in-degree, without a row's
    // length leaving the device (loops over the rows on the host and the copies they needed took
    // half of the 18 ms of a handle over 1e6 nodes)
    {
        DevBuf rows, tmp, lens;
        rows.alloc(4 * std::max<size_t>(2 * (size_t)n, 1));
        uint32_t *dr = rows.as<uint32_t>(), *sr = dr + n;
        const hipcub::CountingInputIterator<uint32_t> ids(0);
        const DirectRow is_d{g->colptr.as<uint64_t>(), dmax, true}, is_s{g->colptr.as<uint64_t>(), dmax, false};
        size_t tb = 0;
        if (n) {
            NKPR_HIP(hipcub::DeviceSelect::If(nullptr, tb, ids, dr, sel, (int)n, is_d, s));
            tmp.alloc(tb);
            NKPR_HIP(hipcub::DeviceSelect::If(tmp.p, tb, ids, dr, sel, (int)n, is_d, s));
            NKPR_HIP(hipcub::DeviceSelect::If(tmp.p, tb, ids, sr, sel + 1, (int)n, is_s, s));
            hipLaunchKernelGGL(max_length_kernel, dim3((unsigned)std::min<uint64_t>(blocks_for(n), 1024)), dim3(256),
                               0, s, g->colptr.as<uint64_t>(), n, reinterpret_cast<unsigned long long *>(sel + 4));
            NKPR_HIP(hipGetLastError());
        }
        uint32_t got[6] = {0};
        unsigned long long hub = 0;
        read_back(s, {{got, sel, sizeof(got)}, {&hub, hub_edges, 8}});
        g->hub_edges = hub;
        g->n_d = got[0];
        g->n_s = got[1];
        g->max_in_degree = (uint64_t)got[4] | ((uint64_t)got[5] << 32);
        g->drow.alloc(4 * std::max<size_t>(g->n_d, 1));
        g->srow.alloc(4 * std::max<size_t>(g->n_s, 1));
        g->dptr.alloc(4 * ((size_t)g->n_d + 1));
        if (g->n_d) NKPR_HIP(hipMemcpyAsync(g->drow.p, dr, 4 * (size_t)g->n_d, hipMemcpyDeviceToDevice, s));
        if (g->n_s) NKPR_HIP(hipMemcpyAsync(g->srow.p, sr, 4 * (size_t)g->n_s, hipMemcpyDeviceToDevice, s));
        lens.alloc(4 * ((size_t)g->n_d + 1));
        hipLaunchKernelGGL(row_length_kernel, dim3(blocks_for((uint64_t)g->n_d + 1)), dim3(256), 0, s,
                           g->colptr.as<uint64_t>(), g->drow.as<uint32_t>(), g->n_d, lens.as<uint32_t>());
        NKPR_HIP(hipGetLastError());
        tb = 0;
        DevBuf tmp2;
        NKPR_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, lens.as<uint32_t>(), g->dptr.as<uint32_t>(),
                                                  (size_t)g->n_d + 1, s));
        tmp2.alloc(tb);
        NKPR_HIP(hipcub::DeviceScan::ExclusiveSum(tmp2.p, tb, lens.as<uint32_t>(), g->dptr.as<uint32_t>(),
                                                  (size_t)g->n_d + 1, s));
    }
    NKPR_CHECK((uint64_t)S * g->n_s + 1 < 0xFFFFFFFFull, "too many sliced rows");
}

// The work items over the rows of schedule_rows, once g->src / g->coef* and g->sptr stand.
void schedule_items(nkpr_graph *g) {
    const hipStream_t s = g->stream;
    const uint64_t m = g->m;
    const uint32_t S = g->n_slices, n_s = g->n_s;
    const uint64_t ns_tot = (uint64_t)S * n_s;
    // work items: the rows longer than kCap on the host (at most m / kCap), the runs of shorter rows
    // on the device, whose counts per segment give every run its place
    std::vector<uint4> heavy;
    if (n_s) {
        DevBuf hv, nhv;
        hv.alloc(sizeof(uint4) * (m / kCap + 1));
        nhv.alloc(4);
        NKPR_HIP(hipMemsetAsync(nhv.p, 0, 4, s));
        hipLaunchKernelGGL(heavy_rows_kernel, dim3((unsigned)std::min<uint64_t>(blocks_for(ns_tot), 4096)), dim3(256),
                           0, s, (const uint32_t *)g->sptr.as<uint32_t>(), ns_tot, nhv.as<uint32_t>(), hv.as<uint4>());
        NKPR_HIP(hipGetLastError());
        uint32_t nh = 0;
        read_back(s, {{&nh, nhv.p, 4}});
        heavy.resize(nh);
        read_back(s, {{heavy.data(), hv.p, sizeof(uint4) * (size_t)nh}});
        std::sort(heavy.begin(), heavy.end(), [](const uint4 &x, const uint4 &y) { return x.x < y.x; });
    }
    // Items of kCap in-edges leave most CUs idle below kItemsWanted of them: a graph of 20,000
    // nodes and 1.5e5 arcs ran on 40 blocks.  Such graphs take smaller items.
    uint32_t cap = kCap;
    while (S == 1 && cap > kCapMin && m < (uint64_t)cap * kItemsWanted) cap /= 2;
    // a segment of about 32 items
    const uint64_t per_item = (uint64_t)cap * (g->n_d + ns_tot) / std::max<uint64_t>(m, 1);
    uint32_t seg_rows = 256;
    while (seg_rows < 8192 && seg_rows < 32 * std::min<uint64_t>(per_item, kRowsMax)) seg_rows *= 2;
    const uint32_t dsegs = (g->n_d + seg_rows - 1) / seg_rows, ssegs = (n_s + seg_rows - 1) / seg_rows;
    const uint32_t nseg = dsegs + S * ssegs;
    DevBuf cnt_b, first_b;
    cnt_b.alloc(4 * std::max<size_t>(nseg, 1));
    first_b.alloc(4 * std::max<size_t>(nseg, 1));
    auto runs = [&](const uint32_t *first, uint4 *di, uint4 *si) {
        uint32_t *cnt = cnt_b.as<uint32_t>();
        if (dsegs)
            hipLaunchKernelGGL(build_items_kernel, dim3((dsegs + 3) / 4), dim3(256), 0, s,
                               (const uint32_t *)g->dptr.as<uint32_t>(), g->n_d, 1u, dsegs, seg_rows, cap, cnt, first, di);
        if (ssegs)
            hipLaunchKernelGGL(build_items_kernel, dim3((S * ssegs + 3) / 4), dim3(256), 0, s,
                               (const uint32_t *)g->sptr.as<uint32_t>(), n_s, S, ssegs, seg_rows, cap, cnt + dsegs,
                               first ? first + dsegs : nullptr, si);
        NKPR_HIP(hipGetLastError());
    };
    runs(nullptr, nullptr, nullptr);
    std::vector<uint32_t> cnt(nseg), first(nseg);
    read_back(s, {{cnt.data(), cnt_b.p, 4 * (size_t)nseg}});
    uint64_t at = 0;
    for (uint32_t i = 0; i < dsegs; ++i) {
        first[i] = (uint32_t)at;
        at += cnt[i];
    }
    g->n_ditems = (uint32_t)at;
    uint32_t split_slots = 0;
    std::map<uint32_t, SplitRec> splits;
    std::vector<std::vector<uint4>> hitems(S);
    at = 0;
    size_t h0 = 0;
    for (uint32_t q = 0; q < S; ++q) {
        std::vector<uint4> rows;
        for (; h0 < heavy.size() && heavy[h0].x < (uint64_t)(q + 1) * n_s; ++h0) {
            rows.push_back(heavy[h0]);
            rows.back().x -= q * n_s;
        }
        build_heavy(rows, q, hitems[q], split_slots, splits);
        g->sitem_off[q] = (uint32_t)at;
        at += hitems[q].size();
        for (uint32_t i = 0; i < ssegs; ++i) {
            first[dsegs + q * ssegs + i] = (uint32_t)at;
            at += cnt[dsegs + q * ssegs + i];
        }
    }
    for (uint32_t q = S; q <= (uint32_t)kSlices; ++q) g->sitem_off[q] = (uint32_t)at;
    NKPR_CHECK(at + g->n_ditems < 0x7FFFFFFFull, "too many work items");
    g->n_items = (uint32_t)(g->n_ditems + at);
    g->n_split_items = split_slots;
    g->ditems.alloc(sizeof(uint4) * std::max<size_t>(g->n_ditems, 1));
    g->sitems.alloc(sizeof(uint4) * std::max<size_t>(at, 1));
    if (nseg) {
        NKPR_HIP(hipMemcpyAsync(first_b.p, first.data(), 4 * (size_t)nseg, hipMemcpyHostToDevice, s));
        runs(first_b.as<uint32_t>(), g->ditems.as<uint4>(), g->sitems.as<uint4>());
    }
    for (uint32_t q = 0; q < S; ++q)
        if (!hitems[q].empty())
            NKPR_HIP(hipMemcpyAsync(g->sitems.as<uint4>() + g->sitem_off[q], hitems[q].data(),
                                    sizeof(uint4) * hitems[q].size(), hipMemcpyHostToDevice, s));
    std::vector<uint32_t> srows, sfirst, scount;
    for (auto &kv : splits) {
        srows.push_back(kv.first);
        for (uint32_t q = 0; q < S; ++q) {
            sfirst.push_back(kv.second.first[q]);
            scount.push_back(kv.second.count[q]);
        }
    }
    g->n_split_rows = (uint32_t)srows.size();
    upload(g, g->split_rows, srows);
    upload(g, g->split_first, sfirst);
    upload(g, g->split_count, scount);
    g->split_flag.alloc(std::max<uint32_t>(n_s, 1));
    NKPR_HIP(hipMemsetAsync(g->split_flag.p, 0, std::max<uint32_t>(n_s, 1), s));
    if (g->n_split_rows)
        hipLaunchKernelGGL(split_flag_kernel, dim3(blocks_for(g->n_split_rows)), dim3(256), 0, s,
                           (const uint32_t *)g->split_rows.as<uint32_t>(), g->n_split_rows, g->split_flag.as<uint8_t>());
    NKPR_HIP(hipGetLastError());
    g->claim.alloc(4 * (kArriveAt + kArriveWords));
    NKPR_HIP(hipMemsetAsync(g->claim.p, 0, 4 * (kArriveAt + kArriveWords), s));
    NKPR_HIP(hipStreamSynchronize(s));
    if (env_u32("NKPR_DEBUG", 0))
        std::fprintf(stderr, "[nkpr] n=%u direct rows %u (%u items), sliced rows %u (%u items), "
                             "slices %u, split rows %u\n", g->n, g->n_d, g->n_ditems, n_s,
                     g->n_items - g->n_ditems, S, g->n_split_rows);
}

int bits_for(uint64_t v) {
    int b = 1;
    while (b < 32 && (1ull << b) < v) ++b;
    return b;
}

}  // namespace

void create_graph(const nkpr_csc *c, nkpr_graph *g, const uint64_t *group_off,
                  uint32_t n_groups) {
    const auto t0 = std::chrono::steady_clock::now();
    NKPR_CHECK(c != nullptr, "csc is NULL");
    NKPR_CHECK(c->z < 0x7FFFFFFFull, "node-id bound must be < 2^31");
    NKPR_CHECK(c->colptr != nullptr, "colptr is NULL");
    const uint64_t z = c->z;
    const hipStream_t s = g->stream;
    const bool dev = c->device_ptrs != 0;
    g->z = z;

    // --- inputs on the device -------------------------------------------------------------
    uint64_t m = 0;
    if (dev) NKPR_HIP(hipMemcpy(&m, c->colptr + z, sizeof(uint64_t), hipMemcpyDeviceToHost));
    else m = c->colptr[z];
    NKPR_CHECK(m < 0xFFFFFFFFull, "more than 2^32-1 in-list entries");
    NKPR_CHECK(m == 0 || c->src != nullptr, "src is NULL");
    g->m = m;
    g->weighted = c->weight != nullptr;
    g->own_degrees = c->out_wdeg == nullptr;

    DevBuf colptr_in_b, src_in_b, w_in_b, exists_b, wdeg_b;
    const uint64_t *colptr_in = c->colptr;
    const int32_t *src_in = c->src;
    const float *w_in = c->weight;
    const double *w64_in = c->weight64;
    NKPR_CHECK(c->weight64 == nullptr || c->weight != nullptr, "weight64 given without weight");
    DevBuf w64_in_b;
    const uint8_t *exists = c->exists;
    auto h2d = [&](DevBuf &b, const void *p, size_t bytes) {
        b.alloc(bytes);
        if (bytes) NKPR_HIP(hipMemcpyAsync(b.p, p, bytes, hipMemcpyHostToDevice, s));
        return b.p;
    };
    if (!dev) {
        colptr_in = (const uint64_t *)h2d(colptr_in_b, c->colptr, 8 * (z + 1));
        src_in = (const int32_t *)h2d(src_in_b, c->src, 4 * m);
        if (c->weight) w_in = (const float *)h2d(w_in_b, c->weight, 4 * m);
        if (c->weight64) w64_in = (const double *)h2d(w64_in_b, c->weight64, 8 * m);
        if (c->exists) exists = (const uint8_t *)h2d(exists_b, c->exists, z);
    }
    g->exists_host.clear();
    if (c->exists) {
        g->exists_host.resize(z);
        if (dev) NKPR_HIP(hipMemcpy(g->exists_host.data(), c->exists, z, hipMemcpyDeviceToHost));
        else std::memcpy(g->exists_host.data(), c->exists, z);
    }

    // everything that starts at zero, cleared at once: weighted out-degrees, out-degrees, then flags,
    // counts (nodes, nodes with out-edges, hub edges), the schedule's counts and one more flag
    const size_t own_bytes = c->out_wdeg ? 0 : 8 * (z + 1), cnt_bytes = (4 * (z + 1) + 7) / 8 * 8;
    DevBuf zero_b;
    zero_b.alloc(own_bytes + cnt_bytes + 128);
    NKPR_HIP(hipMemsetAsync(zero_b.p, 0, own_bytes + cnt_bytes + 128, s));
    uint32_t *outcnt = reinterpret_cast<uint32_t *>(zero_b.as<char>() + own_bytes);
    char *tail = zero_b.as<char>() + own_bytes + cnt_bytes;
    uint32_t *flags = reinterpret_cast<uint32_t *>(tail), *sel = reinterpret_cast<uint32_t *>(tail + 64);
    uint32_t *inexact = reinterpret_cast<uint32_t *>(tail + 96);
    auto *counts = reinterpret_cast<unsigned long long *>(tail + 8);
    if (z)
        hipLaunchKernelGGL(validate_ptr_kernel, dim3(blocks_for(z)), dim3(256), 0, s, colptr_in, z,
                           m, exists, flags);
    const double *wdeg = nullptr;
    double *wdeg_own = nullptr;
    if (c->out_wdeg) {
        wdeg = dev ? c->out_wdeg : (const double *)h2d(wdeg_b, c->out_wdeg, 8 * z);
    } else {
        wdeg_own = zero_b.as<double>();
        wdeg = wdeg_own;
    }
    if (m) {
        hipLaunchKernelGGL(out_degree_kernel, dim3(agg_blocks(m)), dim3(kAggThreads), 0, s, src_in, m, z, exists, w_in,
                           w64_in, outcnt, wdeg_own, flags);
    }
    if (c->out_wdeg && z)
        hipLaunchKernelGGL(unit_degree_kernel, dim3((unsigned)std::min<uint64_t>(blocks_for(z), 65536)),
                           dim3(256), 0, s, wdeg, z, exists, flags);
    NKPR_HIP(hipGetLastError());
    if (z)
        hipLaunchKernelGGL(count_kernel, dim3((unsigned)std::min<uint64_t>(blocks_for(z), 1024)), dim3(256), 0, s,
                           outcnt, exists, z, counts, counts + 1);
    NKPR_HIP(hipGetLastError());
    uint32_t hflags = 0;
    unsigned long long hc[2] = {0, 0};
    read_back(s, {{&hflags, flags, 4}, {hc, counts, 16}});
    g->unit_degrees = c->out_wdeg != nullptr && !(hflags & kNotUnitDegree);
    NKPR_CHECK(!(hflags & kBadPtr), "colptr is not a non-decreasing offset array ending at m");
    NKPR_CHECK(!(hflags & kBadSrc), "an in-list names a source outside [0, z) or a deleted node");
    NKPR_CHECK(!(hflags & kBadExists), "a deleted slot has in-edges");

    // --- relabel: out-degree descending, deleted slots dropped ------------------------------
    const uint32_t n = (uint32_t)hc[0];
    g->n = n;
    g->sink_begin = (uint32_t)hc[1];

    DevBuf k1, k2, v1, v2, tmp;
    g->perm.alloc(4 * std::max<uint64_t>(n, 1));
    if (group_off) {
        // batch of graphs: relabel inside every graph, graphs stay contiguous in id order
        NKPR_CHECK(n_groups >= 1, "a batch needs at least one graph");
        NKPR_CHECK(group_off[0] == 0 && group_off[n_groups] == z, "graph offsets must span [0, z)");
        for (uint32_t q = 0; q < n_groups; ++q)
            NKPR_CHECK(group_off[q] <= group_off[q + 1], "graph offsets must be non-decreasing");
        DevBuf offb, gidb, ce, cn, fl;
        offb.alloc(8 * ((uint64_t)n_groups + 1));
        NKPR_HIP(hipMemcpyAsync(offb.p, group_off, 8 * ((uint64_t)n_groups + 1), hipMemcpyHostToDevice, s));
        gidb.alloc(4 * std::max<uint64_t>(z, 1));
        ce.alloc(4 * (uint64_t)n_groups);
        cn.alloc(4 * (uint64_t)n_groups);
        fl.alloc(4);
        NKPR_HIP(hipMemsetAsync(ce.p, 0, 4 * (uint64_t)n_groups, s));
        NKPR_HIP(hipMemsetAsync(cn.p, 0, 4 * (uint64_t)n_groups, s));
        NKPR_HIP(hipMemsetAsync(fl.p, 0, 4, s));
        DevBuf k64a, k64b;
        k64a.alloc(8 * std::max<uint64_t>(z, 1));
        k64b.alloc(8 * std::max<uint64_t>(z, 1));
        v1.alloc(4 * std::max<uint64_t>(z, 1));
        v2.alloc(4 * std::max<uint64_t>(z, 1));
        if (z) {
            hipLaunchKernelGGL(group_id_kernel, dim3(blocks_for(z)), dim3(256), 0, s,
                               offb.as<uint64_t>(), n_groups, z, gidb.as<uint32_t>());
            hipLaunchKernelGGL(group_keys_kernel, dim3(blocks_for(z)), dim3(256), 0, s,
                               outcnt, exists, gidb.as<uint32_t>(), n_groups, z,
                               k64a.as<uint64_t>(), v1.as<int32_t>(), ce.as<uint32_t>(), cn.as<uint32_t>());
            const unsigned eb = (unsigned)std::min<uint64_t>(blocks_for(z * 64), 1u << 18);
            hipLaunchKernelGGL(group_edges_kernel, dim3(eb), dim3(256), 0, s, colptr_in, src_in,
                               gidb.as<uint32_t>(), z, fl.as<uint32_t>());
            NKPR_HIP(hipGetLastError());
            hipcub::DoubleBuffer<uint64_t> kb(k64a.as<uint64_t>(), k64b.as<uint64_t>());
            hipcub::DoubleBuffer<int32_t> vb(v1.as<int32_t>(), v2.as<int32_t>());
            const int end_bit = 32 + bits_for((uint64_t)n_groups + 1);
            size_t tb = 0;
            NKPR_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, kb, vb, (size_t)z, 0, end_bit, s));
            tmp.alloc(tb);
            NKPR_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb, kb, vb, (size_t)z, 0, end_bit, s));
            if (n)
                NKPR_HIP(hipMemcpyAsync(g->perm.p, vb.Current(), 4 * (size_t)n,
                                        hipMemcpyDeviceToDevice, s));
        }
        std::vector<uint32_t> he(n_groups), hn(n_groups);
        uint32_t hf = 0;
        read_back(s, {{he.data(), ce.p, 4 * (uint64_t)n_groups},
                      {hn.data(), cn.p, 4 * (uint64_t)n_groups},
                      {&hf, fl.p, 4}});
        NKPR_CHECK(!(hf & kBadGroup), "an edge joins two graphs of the batch");
        g->n_groups = n_groups;
        g->goff.assign((size_t)n_groups + 1, 0);
        g->gsink.assign(n_groups, 0);
        g->gslot.assign(group_off, group_off + n_groups + 1);
        for (uint32_t q = 0; q < n_groups; ++q) {
            g->goff[q + 1] = g->goff[q] + he[q];
            g->gsink[q] = g->goff[q] + hn[q];
        }
        // no global sink range: sinks are the tail of every graph's range
        g->sink_begin = n;
    } else if (z) {
        k1.alloc(4 * z);
        k2.alloc(4 * z);
        v1.alloc(4 * z);
        v2.alloc(4 * z);
        hipLaunchKernelGGL(relabel_keys_kernel, dim3(blocks_for(z)), dim3(256), 0, s,
                           outcnt, exists, z, k1.as<uint32_t>(), v1.as<int32_t>());
        hipcub::DoubleBuffer<uint32_t> kb(k1.as<uint32_t>(), k2.as<uint32_t>());
        hipcub::DoubleBuffer<int32_t> vb(v1.as<int32_t>(), v2.as<int32_t>());
        size_t tb = 0;
        NKPR_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, kb, vb, (size_t)z, 0, 32, s));
        tmp.alloc(tb);
        NKPR_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb, kb, vb, (size_t)z, 0, 32, s));
        if (n)
            NKPR_HIP(hipMemcpyAsync(g->perm.p, vb.Current(), 4 * (size_t)n,
                                    hipMemcpyDeviceToDevice, s));
    }
    // iperm (slot -> compact id), reuse k1 storage
    DevBuf iperm_b;
    iperm_b.alloc(4 * std::max<uint64_t>(z, 1));
    int32_t *iperm = iperm_b.as<int32_t>();
    NKPR_HIP(hipMemsetAsync(iperm, 0xFF, 4 * std::max<uint64_t>(z, 1), s));
    if (n)
        hipLaunchKernelGGL(iperm_kernel, dim3(blocks_for(n)), dim3(256), 0, s, g->perm.as<int32_t>(),
                           n, iperm);
    if (n)
        hipLaunchKernelGGL(hub_edges_kernel, dim3(1), dim3(1024), 0, s, g->perm.as<int32_t>(),
                           std::min<uint32_t>(n, kHubSources), outcnt, counts + 2);
    NKPR_HIP(hipGetLastError());
    k1.reset(); k2.reset(); v1.reset(); v2.reset(); tmp.reset();

    // --- new colptr -------------------------------------------------------------------------
    DevBuf len_b;
    len_b.alloc(8 * ((uint64_t)n + 1));
    hipLaunchKernelGGL(new_lengths_kernel, dim3(blocks_for((uint64_t)n + 1)), dim3(256), 0, s,
                       g->perm.as<int32_t>(), n, colptr_in, len_b.as<uint64_t>());
    g->colptr.alloc(8 * ((uint64_t)n + 1));
    {
        size_t tb = 0;
        NKPR_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, len_b.as<uint64_t>(),
                                                  g->colptr.as<uint64_t>(), (size_t)n + 1, s));
        tmp.alloc(tb);
        NKPR_HIP(hipcub::DeviceScan::ExclusiveSum(tmp.p, tb, len_b.as<uint64_t>(),
                                                  g->colptr.as<uint64_t>(), (size_t)n + 1, s));
        tmp.reset();
    }
    len_b.reset();

    // --- edges: into the order of the sweep (kCap zero entries of padding after the last one) ---
    schedule_rows(g, sel, counts + 2);
    const uint64_t ns_tot = (uint64_t)g->n_slices * g->n_s, nseg = g->n_d + ns_tot;
    g->sptr.alloc(4 * (ns_tot + 1));
    g->src.alloc(4 * (m + kCap));
    if (g->weighted) {
        g->coef32.alloc(4 * (m + kCap));
        g->coef64.alloc(8 * (m + kCap));
    }
    hipLaunchKernelGGL(pad_kernel, dim3(kCap / 256), dim3(256), 0, s, g->src.as<int32_t>() + m,
                       g->weighted ? g->coef32.as<float>() + m : nullptr,
                       g->weighted ? g->coef64.as<double>() + m : nullptr);
    if (m) {
        DevBuf ka, kb2, va, vb2, place;
        ka.alloc(8 * m);
        kb2.alloc(8 * m);
        va.alloc(4 * m);
        vb2.alloc(4 * m);
        place.alloc(4 * z);
        if (g->n_d)
            hipLaunchKernelGGL(row_place_kernel, dim3(blocks_for(g->n_d)), dim3(256), 0, s, g->perm.as<int32_t>(),
                               (const uint32_t *)g->drow.as<uint32_t>(), g->n_d, 0u, place.as<uint32_t>());
        if (g->n_s)
            hipLaunchKernelGGL(row_place_kernel, dim3(blocks_for(g->n_s)), dim3(256), 0, s, g->perm.as<int32_t>(),
                               (const uint32_t *)g->srow.as<uint32_t>(), g->n_s, kSlicedRow, place.as<uint32_t>());
        const int vbits = bits_for(n);
        hipLaunchKernelGGL(edge_keys_kernel, dim3((unsigned)((m + kKeyTile - 1) / kKeyTile)), dim3(256), 0, s, colptr_in,
                           src_in, m, iperm, (const uint32_t *)place.as<uint32_t>(), z, g->n_d, g->n_s, g->n_slices,
                           env_u32("NKPR_SLICE_REPLICATE", kDefaultSliceReplicate), vbits, ka.as<uint64_t>(),
                           va.as<uint32_t>());
        NKPR_HIP(hipGetLastError());
        hipcub::DoubleBuffer<uint64_t> kd(ka.as<uint64_t>(), kb2.as<uint64_t>());
        hipcub::DoubleBuffer<uint32_t> vd(va.as<uint32_t>(), vb2.as<uint32_t>());
        int end_bit = vbits;
        while (end_bit < 64 && (1ull << (end_bit - vbits)) < nseg) ++end_bit;
        size_t tb = 0;
        NKPR_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, kd, vd, (size_t)m, 0, end_bit, s));
        tmp.alloc(tb);
        NKPR_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tb, kd, vd, (size_t)m, 0, end_bit, s));
        hipLaunchKernelGGL(segment_starts_kernel, dim3((unsigned)std::min<uint64_t>(blocks_for(ns_tot + 1), 65536)),
                           dim3(256), 0, s, (const uint64_t *)kd.Current(), m, vbits, (uint64_t)g->n_d, ns_tot,
                           g->sptr.as<uint32_t>());
        const unsigned gb = (unsigned)std::min<uint64_t>(blocks_for(m), 65536);
        hipLaunchKernelGGL(edge_output_kernel, dim3(gb), dim3(256), 0, s, kd.Current(), vd.Current(),
                           m, (1ull << vbits) - 1, g->weighted ? w_in : nullptr, g->weighted ? w64_in : nullptr, src_in,
                           wdeg, g->src.as<int32_t>(),
                           g->weighted ? g->coef32.as<float>() : nullptr,
                           g->weighted ? g->coef64.as<double>() : nullptr);
        NKPR_HIP(hipGetLastError());
        if (g->weighted) {
            // input position of every edge, kept so that new weights can be folded in place
            DevBuf &sorted = vd.Current() == va.as<uint32_t>() ? va : vb2;
            std::swap(g->emap.p, sorted.p);
            std::swap(g->emap.bytes, sorted.bytes);
        }
    } else {
        NKPR_HIP(hipMemsetAsync(g->sptr.p, 0, 4 * (ns_tot + 1), s));
    }
    if (g->own_degrees) g->deg64.alloc(8 * std::max<uint64_t>(n, 1));
    double *deg64 = g->own_degrees ? g->deg64.as<double>() : nullptr;
    if (!g->weighted) {
        g->inv32.alloc(4 * std::max<uint64_t>(n, 1));
        g->inv64.alloc(8 * std::max<uint64_t>(n, 1));
        if (n)
            hipLaunchKernelGGL(inv_degree_kernel, dim3(blocks_for(n)), dim3(256), 0, s,
                               g->perm.as<int32_t>(), n, outcnt, wdeg, g->inv64.as<double>(),
                               g->inv32.as<float>(), deg64);
        NKPR_HIP(hipGetLastError());
    } else {
        // 1 / weighted out-degree, and whether every weight is an FP32 number (then the binned
        // FP64 sweep reads 4-byte weights instead of 8-byte coefficients)
        g->invw64.alloc(8 * std::max<uint64_t>(n, 1));
        if (n)
            hipLaunchKernelGGL(inv_degree_kernel, dim3(blocks_for(n)), dim3(256), 0, s,
                               g->perm.as<int32_t>(), n, outcnt, wdeg, g->invw64.as<double>(),
                               (float *)nullptr, deg64);
        NKPR_HIP(hipGetLastError());
        g->w32_exact = true;
        if (w64_in && m) {
            hipLaunchKernelGGL(fp32_exact_kernel, dim3((unsigned)std::min<uint64_t>(blocks_for(m), 2048)), dim3(256), 0, s,
                               w_in, w64_in, m, inexact);
            NKPR_HIP(hipGetLastError());
            uint32_t hf = 0;
            read_back(s, {{&hf, inexact, 4}});
            g->w32_exact = hf == 0;
        }
    }

    // --- schedule ---------------------------------------------------------------------------
    schedule_items(g);
    NKPR_HIP(hipStreamSynchronize(s));
    g->prep_ms =
        std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

namespace {

// Weighted out-degree of every compact source from the edges in sweep order.
__global__ __launch_bounds__(kAggThreads) void sweep_wdeg_kernel(const int32_t *src, const uint32_t *emap,
                                                                 uint64_t m, const float *w,
                                                                 const double *w64, double *wdeg) {
    __shared__ AggTable agg;
    agg.clear();
    for (uint64_t i = (uint64_t)blockIdx.x * kAggThreads + threadIdx.x; i < m;
         i += (uint64_t)gridDim.x * kAggThreads) {
        const uint32_t o = emap[i];
        agg.add((uint32_t)src[i], w64 ? w64[o] : (double)w[o], nullptr, wdeg);
    }
    agg.flush(nullptr, wdeg);
}

__global__ void gather_wdeg_kernel(const double *wdeg_z, const int32_t *perm, uint32_t n,
                                   double *wdeg) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) wdeg[i] = wdeg_z[perm[i]];
}

// coef = w / deg(src) for every edge in sweep order (the fold of graph creation).
__global__ void refold_kernel(const int32_t *src, const uint32_t *emap, uint64_t m,
                              const float *w, const double *w64, const double *wdeg,
                              float *c32, double *c64) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t o = emap[i];
        const double c = (w64 ? w64[o] : (double)w[o]) / wdeg[src[i]];
        c64[i] = c;
        c32[i] = (float)c;
    }
}

}  // namespace

// New edge weights for the same structure (nkpr_graph_set_weights).
void set_weights(nkpr_graph *g, const float *w, const double *w64, const double *out_wdeg,
                 int device_ptrs) {
    NKPR_CHECK(g != nullptr, "graph is NULL");
    NKPR_CHECK(g->weighted, "the graph was created without weights");
    NKPR_CHECK(w != nullptr || w64 != nullptr, "weights are NULL");
    const hipStream_t s = g->stream;
    const uint64_t m = g->m, z = g->z;
    const uint32_t n = g->n;
    DevBuf wb, w64b, degz, deg;
    if (!device_ptrs) {
        if (w) {
            wb.alloc(4 * std::max<uint64_t>(m, 1));
            NKPR_HIP(hipMemcpyAsync(wb.p, w, 4 * m, hipMemcpyHostToDevice, s));
            w = wb.as<float>();
        }
        if (w64) {
            w64b.alloc(8 * std::max<uint64_t>(m, 1));
            NKPR_HIP(hipMemcpyAsync(w64b.p, w64, 8 * m, hipMemcpyHostToDevice, s));
            w64 = w64b.as<double>();
        }
    }
    deg.alloc(8 * std::max<uint32_t>(n, 1));
    if (out_wdeg) {
        const double *dz = out_wdeg;
        if (!device_ptrs) {
            degz.alloc(8 * std::max<uint64_t>(z, 1));
            NKPR_HIP(hipMemcpyAsync(degz.p, out_wdeg, 8 * z, hipMemcpyHostToDevice, s));
            dz = degz.as<double>();
        }
        if (n)
            hipLaunchKernelGGL(gather_wdeg_kernel, dim3(blocks_for(n)), dim3(256), 0, s, dz,
                               g->perm.as<int32_t>(), n, deg.as<double>());
        DevBuf uf;
        uf.alloc(4);
        NKPR_HIP(hipMemsetAsync(uf.p, 0, 4, s));
        if (n)
            hipLaunchKernelGGL(unit_degree_kernel, dim3((unsigned)std::min<uint64_t>(blocks_for(n), 65536)),
                               dim3(256), 0, s, (const double *)deg.as<double>(), (uint64_t)n,
                               (const uint8_t *)nullptr, uf.as<uint32_t>());
        NKPR_HIP(hipGetLastError());
        uint32_t hf = 0;
        read_back(s, {{&hf, uf.p, 4}});
        g->unit_degrees = !(hf & kNotUnitDegree);
    } else {
        g->unit_degrees = false;
        NKPR_HIP(hipMemsetAsync(deg.p, 0, 8 * std::max<uint32_t>(n, 1), s));
        if (m)
            hipLaunchKernelGGL(sweep_wdeg_kernel, dim3(agg_blocks(m)), dim3(kAggThreads), 0, s, g->src.as<int32_t>(), g->emap.as<uint32_t>(), m, w,
                               w64, deg.as<double>());
    }
    NKPR_HIP(hipGetLastError());
    if (m)
        hipLaunchKernelGGL(refold_kernel, dim3((unsigned)std::min<uint64_t>(blocks_for(m), 65536)),
                           dim3(256), 0, s, g->src.as<int32_t>(), g->emap.as<uint32_t>(), m, w, w64,
                           deg.as<double>(), g->coef32.as<float>(), g->coef64.as<double>());
    NKPR_HIP(hipGetLastError());
    if (n)
        hipLaunchKernelGGL(inv_of_kernel, dim3(blocks_for(n)), dim3(256), 0, s, (const double *)deg.as<double>(), n,
                           g->invw64.as<double>());
    NKPR_HIP(hipGetLastError());
    bool exact = true;
    if (w && w64 && m) {
        DevBuf flag;
        flag.alloc(4);
        NKPR_HIP(hipMemsetAsync(flag.p, 0, 4, s));
        hipLaunchKernelGGL(fp32_exact_kernel, dim3((unsigned)std::min<uint64_t>(blocks_for(m), 2048)), dim3(256), 0, s,
                           w, w64, m, flag.as<uint32_t>());
        NKPR_HIP(hipGetLastError());
        uint32_t hf = 0;
        read_back(s, {{&hf, flag.p, 4}});
        exact = hf == 0;
    } else if (!w) {
        exact = false;  // FP64 weights alone: not checked
    }
    if (exact != g->w32_exact) g->bn64.ready = false;  // the FP64 copy changes its coefficient type
    g->w32_exact = exact;
    NKPR_HIP(hipStreamSynchronize(s));
    g->own_degrees = out_wdeg == nullptr;
    if (g->own_degrees) {
        std::swap(g->deg64.p, deg.p);
        std::swap(g->deg64.bytes, deg.bytes);
    }
    // derived copies follow the coefficients
    g->b_coef_ready = false;
    g->rowsum_ready = false;
    g->bn32.coef_ready = false;
    g->bn64.coef_ready = false;
    g->adj_stale = true;
}

}  // namespace nkpr
