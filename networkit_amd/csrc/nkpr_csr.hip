// CSR matrix-vector products in NetworKit's CSR format, and AlgebraicPageRank on them.
//
// The matrix is a CSRGeneralMatrix<double> as NetworKit stores it
// (include/networkit/algebraic/CSRGeneralMatrix.hpp): row_idx[rows + 1] and col_idx[nnz]
// are 64-bit `index` values, values[nnz] are doubles, and a row keeps its entries in storage
// order (duplicates stay separate).  All arrays live in device memory.
//
//   nkpr_csr_spmv           CSRGeneralMatrix::operator*(const Vector&)
//                           (CSRGeneralMatrix.hpp:563-578): y[i] = sum_k values[k] x[col_idx[k]]
//   nkpr_csr_pagerank_step  one iteration of AlgebraicPageRank::run
//                           (AlgebraicPageRank.hpp:97-101): y = M x + shift and ||y - x||_2^2
//   nkpr_algebraic_pagerank AlgebraicPageRank::run (AlgebraicPageRank.hpp:94-119): the loop to
//                           ||y - x||_2 <= tol from 1/n, then y / sum(y)
//
// Kernels.  Every sum is added in an order fixed by the matrix alone (deterministic):
//   csr_tile_kernel   the rows' ends and the entries, merged into one list (Merrill and Garland,
//       "Merge-based parallel sparse matrix-vector multiplication", SC 2016), are cut into tiles of
//       equal length, so that a block has as much to do whatever the rows' lengths: it finds its
//       first row and entry by a search over row_idx (64 probes at a time, the lanes of a wave),
//       reads its entries as one stream, puts the products into LDS and adds them row by row, lane
//       groups for short rows, whole waves for long ones and all waves where few rows fill the
//       tile.  What is left after its last row end
//       is the tile's carry for the row that goes on.
//   csr_fix_kernel    adds the carries to the row that ended in a later tile.
//   csr_final_kernel  (steps of many tiles) adds the blocks' sums.
// The step's (y - x)^2 is added per block of either kernel.
//
// What bounds it: the two 8-byte streams (16 bytes per entry) and the gathers of x, in flight
// together for a whole tile.  A lane group per row with a block sum per long row kept one or two
// entries in flight per lane and left long rows to five more launches (one of them a single
// thread): 713 us for the step of an R-MAT matrix of 1e6 rows and 1.4e7 entries, 148 us now (the tiles
// 129 us).
//
// Scratch of a product: a carry (row and sum) per tile, 12 bytes for 4096 merged items, and the
// blocks' sums of squares.  A plain product and a step take it from the stream's memory pool for the duration
// of the call, the allocation-free step from a static device array (which caps the matrices it
// accepts).
//
// Algorithmic bytes per product (HBM-bound, random gathers of x): per entry col 8 + value 8 +
// gathered x 8; per row row_idx 8 + y 8 (+ x 8 for the step's norm).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <vector>

#include "nkpr_internal.hpp"

// Scratch of nkpr_csr_pagerank_step_noalloc (48.1 MiB): the tiles' carries and sums.  Every GPU the
// library runs on holds it until the process ends.  Host code never uses this name as an
// address: it takes the array's address per device with hipGetSymbolAddress
// (csr_noalloc_scratch).
static __device__ __align__(256) unsigned char scratch[(1u << 21) * 8 + (1u << 22) * 8 + 65536];

namespace nkpr {
namespace {

constexpr int kFinalThreads = 256;
// A tile: kThreads threads, kPer merged items each.  The small one spreads matrices of fewer than
// kSmallItems merged items over the device.
template <int THREADS, int PER> struct TileShape {
    static constexpr int kThreads = THREADS, kPer = PER, kItems = THREADS * PER;
};
using LargeTile = TileShape<512, 8>;
using SmallTile = TileShape<256, 4>;
constexpr uint64_t kSmallItems = 1ull << 22;
// a row longer than kTurns lanes' worth of its lane group is added by a whole wave
constexpr uint32_t kTurns = 32;
constexpr uint32_t kNoRow = 0xFFFFFFFFu;
// blocks of the tile kernel, at most (each steps over tiles); tiles whose carries one block of the
// fix kernel takes, and its blocks when there are more
constexpr uint32_t kTileGrid = 4096;
constexpr int kFixThreads = 1024;
constexpr uint32_t kFixAlone = 16384, kFixGrid = 512;
// matrices the allocation-free step accepts (see csr_step_noalloc_impl)
constexpr uint32_t kNoallocList = 1u << 21, kNoallocPieces = 1u << 22;
constexpr uint32_t kNoallocPiece = 4096;

struct CsrView {
    uint64_t rows, nnz;       // nnz: length of col_idx and values
    const uint64_t *row_idx;
    const uint64_t *col_idx;
    const double *val;
};

// The scratch of one product, carved from one buffer.
struct TileWork {
    double *carry;      // [tiles] sum of the entries after the tile's last row end
    double *partials;   // [kTileGrid + kFixGrid] (y - x)^2 per block of the two kernels
    uint32_t *row;      // [tiles] the row the carry belongs to, kNoRow without one
};

bool small_matrix(const CsrView &A) { return A.rows + A.nnz < kSmallItems; }

uint64_t tiles_of(const CsrView &A) {
    const uint64_t items = small_matrix(A) ? SmallTile::kItems : LargeTile::kItems;
    return (A.rows + A.nnz + items - 1) / items;
}

uint32_t tile_grid(uint64_t tiles) { return (uint32_t)std::min<uint64_t>(tiles, kTileGrid); }

size_t work_bytes(uint64_t tiles) { return 12 * (size_t)tiles + 8 * (size_t)(kTileGrid + kFixGrid); }

TileWork carve(void *base, uint64_t tiles) {
    TileWork w;
    w.carry = static_cast<double *>(base);
    w.partials = w.carry + tiles;
    w.row = reinterpret_cast<uint32_t *>(w.partials + kTileGrid + kFixGrid);
    return w;
}

// Block sum (fixed order: shuffles inside each wave, then thread 0 adds the waves); the
// result is valid in thread 0.
template <int kThreads>
__device__ __forceinline__ double block_sum(double v) {
    __shared__ double wsum[kThreads / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    double tot = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < kThreads / 64; ++w) tot += wsum[w];
    __syncthreads();
    return tot;
}

// The entries that the offsets name: `count` of them from `first` on.  col_idx and values may hold
// more, before them (offsets of some rows of a larger matrix) and after them (lists with room to
// spare); the host only knows their length, so it sizes the grid and the scratch for all of them.
struct Entries {
    uint64_t first, count;
};
__device__ __forceinline__ Entries entries_of(const CsrView &A) {
    const uint64_t first = A.row_idx[0];
    return {first, min(A.row_idx[A.rows] - first, A.nnz)};
}

// Rows that have ended before merged item d: the smallest i in [max(0, d - nnz), min(d, rows)] whose
// row end lies past entry d - i - 1; all rows for an item past the last one.  A wave probes 64 places
// of the range at a time.  The range does not depend on the extent, so that its loads and the first
// probes are on their way together.
__device__ __forceinline__ uint64_t rows_before(const CsrView &A, const Entries &E, uint64_t d) {
    const uint32_t lane = threadIdx.x & 63;
    uint64_t hi = d < A.rows ? d : A.rows, lo = d > A.nnz ? min(d - A.nnz, hi) : 0;
    while (lo < hi) {
        const uint64_t step = (hi - lo + 63) / 64;
        const uint64_t mid = lo + (lane + 1) * step - 1;
        const bool ended = mid < hi && A.row_idx[mid + 1] - E.first <= d - mid - 1;
        const uint64_t c = (uint64_t)__popcll(__ballot(ended));
        const uint64_t next = lo + (c + 1) * step - 1;
        lo += c * step;
        hi = next < hi ? next : hi;
    }
    return lo;
}

// Tile t: rows [i0, i1) end in it, with entries [k0, k1).  Tiles past the last merged item are empty
// and leave no carry.
// Six waves a SIMD: the large tile's LDS lets three blocks share a CU.
template <typename Shape, bool STEP>
__global__ __launch_bounds__(Shape::kThreads, 6) void csr_tile_kernel(CsrView A,
                                                                   const double *__restrict__ x,
                                                                   double shift, double *y,
                                                                   TileWork w, uint64_t tiles) {
    constexpr uint32_t kThreads = Shape::kThreads, kPer = Shape::kPer, kItems = Shape::kItems;
    static_assert(kItems < 65536, "ends are 16-bit offsets into the tile");
    __shared__ double prod[kItems];
    __shared__ uint16_t ends[kItems + 2];  // ends[j], ends[j + 1]: the tile's part of row i0 + j
    __shared__ uint16_t longs[kItems / kTurns];
    __shared__ uint32_t n_long;
    constexpr uint32_t kSpread = kItems / kThreads;
    __shared__ double share[kSpread][kThreads / 64];
    __shared__ uint64_t s_row[2];
    const uint32_t tid = threadIdx.x, wave = tid >> 6;
    const Entries E = entries_of(A);
    double sq = 0.0;
    for (uint64_t t = blockIdx.x; t < tiles; t += gridDim.x) {
        const uint64_t d0 = t * kItems, d1 = d0 + kItems;
        if (wave < 2) {
            const uint64_t i = rows_before(A, E, wave ? d1 : d0);
            if ((tid & 63) == 0) s_row[wave] = i;
        }
        if (tid == 0) n_long = 0;
        __syncthreads();
        const uint64_t i0 = s_row[0], i1 = s_row[1];
        const uint64_t k0 = min(d0 - i0, E.count), k1 = min(d1 - i1, E.count);
        const uint32_t cnt = (uint32_t)(k1 - k0), whole = (uint32_t)(i1 - i0);
        // the entries, every load before the gathers that need it
        const uint64_t *__restrict__ col = A.col_idx + E.first + k0;
        const double *__restrict__ val = A.val + E.first + k0;
        uint64_t c[kPer];
        double v[kPer];
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k) {
            const uint32_t e = tid + k * kThreads;
            c[k] = e < cnt ? __builtin_nontemporal_load(col + e) : 0;
            v[k] = e < cnt ? __builtin_nontemporal_load(val + e) : 0.0;
        }
        for (uint32_t j = tid; j < whole; j += kThreads)
            ends[j + 1] = (uint16_t)(min(A.row_idx[i0 + j + 1] - E.first, k1) - k0);
        if (tid == 0) {
            ends[0] = 0;
            ends[whole + 1] = (uint16_t)cnt;
        }
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k) {
            const uint32_t e = tid + k * kThreads;
            if (e < cnt) prod[e] = v[k] * x[c[k]];
        }
        __syncthreads();
        // row i0 began in an earlier tile: its sum, and its square, are finished by the fix kernel
        const bool continued = i0 < A.rows && A.row_idx[i0] - E.first < k0;
        const uint32_t R = whole + 1;  // the last one: what is left after the last row end
        const uint32_t tail = cnt - ends[whole];
        auto put = [&](uint32_t r, double sum) {
            if (r == whole) {
                w.carry[t] = sum;
                w.row[t] = tail ? (uint32_t)i1 : kNoRow;
                return;
            }
            const double yr = sum + shift;
            y[i0 + r] = yr;
            if (STEP && !(r == 0 && continued)) {
                const double d = yr - x[i0 + r];
                sq += d * d;
            }
        };
        // n rows (at most kSpread), a share of each for every wave: rows that fill a tile or a good part of
        // it would keep one wave each busy and the others waiting (us a step with a wave a row / so:
        // rows of 70000 entries 301 / 252, of 1500 99 / 94; one row of 5000 in 1000 61.3 both)
        auto spread = [&](uint32_t n, auto row) {
            for (uint32_t k = 0; k < n; ++k) {
                const uint32_t r = row(k), e = ends[r + 1];
                double acc = 0.0;
                for (uint32_t i = ends[r] + tid; i < e; i += kThreads) acc += prod[i];
                for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
                if ((tid & 63) == 0) share[k][wave] = acc;
            }
            __syncthreads();
            if (tid < n) {
                double sum = 0.0;
                for (uint32_t k = 0; k < kThreads / 64; ++k) sum += share[tid][k];
                put(row(tid), sum);
            }
        };
        if (cnt >= kThreads * R) {  // a turn of the block or more per row
            spread(R, [](uint32_t k) { return k; });
        } else {
            // G consecutive lanes a row, G ~ the average length
            const uint32_t avg = cnt / R;
            const int lg = avg >= 64 ? 6 : (avg >= 32 ? 5 : (avg >= 16 ? 4 : (avg >= 8 ? 3 : (avg >= 4 ? 2 : (avg >= 2 ? 1 : 0)))));
            const uint32_t G = 1u << lg, lane = tid & (G - 1), per_pass = kThreads >> lg;
            for (uint32_t base = 0; base < R; base += per_pass) {
                const uint32_t r = base + (tid >> lg);
                double acc = 0.0;
                bool own = r < R;
                if (own) {
                    const uint32_t b = ends[r], e = ends[r + 1];
                    if (e - b > kTurns * G) {
                        own = false;
                        if (lane == 0) longs[atomicAdd(&n_long, 1u)] = (uint16_t)r;
                    } else {
                        for (uint32_t i = b + lane; i < e; i += G) acc += prod[i];
                    }
                }
                for (uint32_t off = G >> 1; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
                if (own && lane == 0) put(r, acc);
            }
            __syncthreads();
            const uint32_t nl = n_long;
            if (nl == 1 || nl == 2) spread(nl, [&](uint32_t k) { return (uint32_t)longs[k]; });
            for (uint32_t k = nl > 2 ? wave : nl; k < nl; k += kThreads / 64) {
                const uint32_t r = longs[k];
                double acc = 0.0;
                for (uint32_t i = ends[r] + (tid & 63); i < ends[r + 1]; i += 64) acc += prod[i];
                for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
                if ((tid & 63) == 0) put(r, acc);
            }
        }
        __syncthreads();  // the next tile rewrites the shared arrays
    }
    if (STEP) {
        const double tot = block_sum<kThreads>(sq);
        if (tid == 0) w.partials[blockIdx.x] = tot;
    }
}

// The carries of row r from tile t on, added by the wave: lanes stride over kRunTurns * 64 tiles at a
// time, then a shuffle tree.  Every lane gets the sum.
constexpr uint32_t kRunTurns = 4;
__device__ __forceinline__ double sum_run(const TileWork &w, uint64_t t, uint32_t r, uint64_t tiles) {
    const uint32_t lane = threadIdx.x & 63;
    double acc = 0.0;
    for (uint64_t q0 = t + lane;; q0 += 64 * kRunTurns) {
        uint32_t row[kRunTurns];
        double c[kRunTurns];
#pragma unroll
        for (uint32_t k = 0; k < kRunTurns; ++k) {
            const uint64_t q = q0 + 64 * k;
            row[k] = q < tiles ? w.row[q] : kNoRow;
            c[k] = q < tiles ? w.carry[q] : 0.0;
        }
#pragma unroll
        for (uint32_t k = 0; k < kRunTurns; ++k)
            if (row[k] == r) acc += c[k];
        if (!__all(row[kRunTurns - 1] == r)) break;
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    return acc;
}

// The carries: the first of a run of tiles with the same carry row adds the run's carries, in an
// order fixed by the matrix, to that row: in tile order up to kRunAlone of them, a wave for more.
// For a step the squares of the rows finished here, after the first n_sq block sums of the tile
// kernel, go to out[blockIdx.x].
//
// Bound by latency: two rounds of loads.  A thread that walked a run alone waited for one tile's row
// after the other; steps with one row of 4e6, 1e7 and 1e8 entries took 594, 408 and 4040 us, now 33, 49
// and 365.
constexpr uint32_t kRunAlone = 8;
template <bool STEP>
__global__ __launch_bounds__(kFixThreads) void csr_fix_kernel(const double *__restrict__ x, double *y,
                                                              TileWork w, uint64_t tiles,
                                                              uint32_t n_sq, double *out) {
    double sq = 0.0;
    for (uint32_t b = threadIdx.x; STEP && b < n_sq; b += kFixThreads) sq += w.partials[b];
    const uint32_t lane = threadIdx.x & 63;
    for (uint64_t t0 = (uint64_t)blockIdx.x * kFixThreads + (threadIdx.x - lane); t0 < tiles;
         t0 += (uint64_t)gridDim.x * kFixThreads) {
        const uint64_t t = t0 + lane;
        const uint32_t r = t < tiles ? w.row[t] : kNoRow, last = t > 0 && t < tiles ? w.row[t - 1] : kNoRow;
        const uint32_t next = t + 1 < tiles ? w.row[t + 1] : kNoRow;
        const uint32_t far = t + kRunAlone < tiles ? w.row[t + kRunAlone] : kNoRow;
        double s = t < tiles ? w.carry[t] : 0.0;
        const bool first = r != kNoRow && last != r, many = first && far == r;
        if (first && !many && next == r) {
            s += w.carry[t + 1];
            for (uint64_t q = t + 2; q < tiles && w.row[q] == r; ++q) s += w.carry[q];
        }
        for (uint64_t left = __ballot(many); left; left &= left - 1) {
            const int l = __ffsll((long long)left) - 1;
            const double sum = sum_run(w, t0 + l, __shfl(r, l, 64), tiles);
            if ((int)lane == l) s = sum;
        }
        if (!first) continue;
        const double v = s + y[r];
        y[r] = v;
        if (STEP) {
            const double d = v - x[r];
            sq += d * d;
        }
    }
    if (STEP) {
        const double tot = block_sum<kFixThreads>(sq);
        if (threadIdx.x == 0) out[blockIdx.x] = tot;
    }
}

// out[0] = sum of partials[0, count) in a fixed order.
__global__ __launch_bounds__(kFinalThreads) void csr_final_kernel(const double *partials,
                                                                  uint32_t count, double *out) {
    __shared__ double part[kFinalThreads];
    double s = 0.0;
    for (uint32_t i = threadIdx.x; i < count; i += kFinalThreads) s += partials[i];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int h = kFinalThreads / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = part[0];
}

// Block partials of sum(x) over fixed row tiles (deterministic).
__global__ __launch_bounds__(kFinalThreads) void csr_sum_kernel(const double *x, uint64_t n,
                                                                double *partials) {
    __shared__ double part[kFinalThreads];
    double s = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * kFinalThreads + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * kFinalThreads)
        s += x[i];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int h = kFinalThreads / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = part[0];
}

__global__ void csr_fill_kernel(double *x, uint64_t n, double v) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        x[i] = v;
}

__global__ void csr_scale_kernel(double *x, uint64_t n, const double *sum) {
    const double s = sum[0];
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        x[i] /= s;
}

// Structure check of a matrix before a run: row_idx non-decreasing from 0, every column
// index below cols.  flag[0] is set when something is out of place.
__global__ void csr_check_kernel(CsrView A, uint64_t cols, uint64_t nnz, uint32_t *flag) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    bool bad = false;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < A.rows; i += stride)
        bad |= A.row_idx[i] > A.row_idx[i + 1] || A.row_idx[i + 1] > nnz;
    for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < nnz; k += stride)
        bad |= A.col_idx[k] >= cols;
    if (bad) atomicOr(flag, 1u);
}

CsrView view_of(const nkpr_csr *a) {
    NKPR_CHECK(a != nullptr, "matrix is NULL");
    NKPR_CHECK(a->rows == 0 || (a->row_idx && a->col_idx && a->values),
               "matrix arrays must not be NULL");
    NKPR_CHECK(a->rows < 0xFFFFFFFFull, "more than 2^32 - 2 rows");
    CsrView v;
    v.rows = a->rows;
    v.nnz = a->nnz;
    v.row_idx = a->row_idx;
    v.col_idx = a->col_idx;
    v.val = a->values;
    return v;
}

// The product kernels (and, for a step, the final sum of their block sums into *sq_out).
template <bool STEP>
void launch_product(const CsrView &A, const double *x, double shift, double *y, const TileWork &w,
                    double *sq_out, hipStream_t s) {
    if (A.rows == 0) {
        if (STEP) hipLaunchKernelGGL(csr_fill_kernel, dim3(1), dim3(64), 0, s, sq_out, 1, 0.0);
        return;
    }
    const uint64_t tiles = tiles_of(A);
    const uint32_t grid = tile_grid(tiles);
    if (small_matrix(A))
        hipLaunchKernelGGL((csr_tile_kernel<SmallTile, STEP>), dim3(grid), dim3(SmallTile::kThreads), 0, s, A, x,
                           shift, y, w, tiles);
    else
        hipLaunchKernelGGL((csr_tile_kernel<LargeTile, STEP>), dim3(grid), dim3(LargeTile::kThreads), 0, s, A, x,
                           shift, y, w, tiles);
    NKPR_HIP(hipGetLastError());
    if (tiles <= kFixAlone) {
        hipLaunchKernelGGL((csr_fix_kernel<STEP>), dim3(1), dim3(kFixThreads), 0, s, x, y, w, tiles, grid, sq_out);
    } else {
        // (more tiles than kFixAlone: the tile kernel ran on kTileGrid blocks)
        hipLaunchKernelGGL((csr_fix_kernel<STEP>), dim3(kFixGrid), dim3(kFixThreads), 0, s, x, y, w, tiles, 0u,
                           w.partials + kTileGrid);
        if (STEP)
            hipLaunchKernelGGL(csr_final_kernel, dim3(1), dim3(kFinalThreads), 0, s, w.partials,
                               kTileGrid + kFixGrid, sq_out);
    }
    NKPR_HIP(hipGetLastError());
}

// Device scratch of one call, taken from the stream's memory pool.
struct PoolBuf {
    void *p = nullptr;
    hipStream_t s = nullptr;
    PoolBuf(size_t bytes, hipStream_t st) : s(st) {
        hipError_t e = hipMallocAsync(&p, bytes, st);
        if (e != hipSuccess && !capturing(st)) {
            // as device_alloc does
            (void)hipGetLastError();
            release_kept();
            e = hipMallocAsync(&p, bytes, st);
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            p = nullptr;
            throw Error(NKPR_ERR_NOMEM, std::string("hipMallocAsync failed: ") + hipGetErrorString(e));
        }
    }
    ~PoolBuf() {
        if (p) (void)hipFreeAsync(p, s);
    }
    static bool capturing(hipStream_t st) {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        return hipStreamIsCapturing(st, &status) != hipSuccess || status != hipStreamCaptureStatusNone;
    }
};

// The address of `scratch` on the current device, taken once per device (each GPU holds its
// own copy of the array at its own address).
void *csr_noalloc_scratch() {
    constexpr int kMaxDevices = 64;
    static std::mutex mu;
    static void *addr[kMaxDevices] = {};
    int dev = -1;
    NKPR_HIP(hipGetDevice(&dev));
    NKPR_CHECK(dev >= 0 && dev < kMaxDevices, "device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void *p = nullptr;
        NKPR_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        NKPR_CHECK(p != nullptr, "hipGetSymbolAddress returned NULL");
        addr[dev] = p;
    }
    return addr[dev];
}

}  // namespace

void csr_spmv_impl(const nkpr_csr *a, const double *x, double *y, hipStream_t s) {
    const CsrView A = view_of(a);
    NKPR_CHECK(A.rows == 0 || (x && y), "x and y must not be NULL");
    NKPR_CHECK(x != y || A.rows == 0, "x and y must be different vectors");
    if (A.rows == 0) return;
    const uint64_t tiles = tiles_of(A);
    PoolBuf buf(work_bytes(tiles), s);
    launch_product<false>(A, x, 0.0, y, carve(buf.p, tiles), nullptr, s);
}

void csr_step_impl(const nkpr_csr *m, double shift, const double *x, double *y, double *step_sq,
                   hipStream_t s) {
    const CsrView A = view_of(m);
    NKPR_CHECK(m->rows == m->cols, "a PageRank step needs a square matrix");
    NKPR_CHECK(step_sq != nullptr, "step_sq must not be NULL");
    NKPR_CHECK(A.rows == 0 || (x && y), "x and y must not be NULL");
    NKPR_CHECK(x != y || A.rows == 0, "x and y must be different vectors");
    const uint64_t tiles = tiles_of(A);
    PoolBuf buf(work_bytes(tiles), s);
    launch_product<true>(A, x, shift, y, carve(buf.p, tiles), step_sq, s);
}

void csr_step_noalloc_impl(const nkpr_csr *m, double shift, const double *x, double *y,
                           double *step_sq, hipStream_t s) {
    const CsrView A = view_of(m);
    NKPR_CHECK(m->rows == m->cols, "a PageRank step needs a square matrix");
    NKPR_CHECK(step_sq != nullptr, "step_sq must not be NULL");
    NKPR_CHECK(A.rows == 0 || (x && y), "x and y must not be NULL");
    NKPR_CHECK(x != y || A.rows == 0, "x and y must be different vectors");
    // what this entry point accepts: at most 2^21 rows longer than 32 x the lanes that rows of
    // the average length take, and 2^22 pieces of 4096 entries, by the worst-case bounds
    const double avg = A.rows ? (double)A.nnz / (double)A.rows : 0.0;
    const uint64_t lanes = avg <= 6.0 ? 4 : (avg <= 12.0 ? 8 : (avg <= 24.0 ? 16 : (avg <= 48.0 ? 32 : 64)));
    const uint64_t lc = std::min<uint64_t>(A.rows, A.nnz / (32 * lanes + 1)) + 1;
    const uint64_t pc = A.nnz / kNoallocPiece + lc + 1;
    NKPR_CHECK(lc <= kNoallocList && pc <= kNoallocPieces,
               "matrix too large for the allocation-free step: it could have more than 2^21 rows "
               "longer than 32 x the lanes per row, or 2^22 pieces of 4096 entries (at most "
               "nnz / (32 lanes + 1) such rows: up to about 2.7e8 entries at an average row "
               "length of 6 or less, 1.07e9 at 24 or less, 4.3e9 above 48)");
    // rows / 4096 is below lc wherever nnz / 4096 is near the cap, so no such matrix has more than
    // 2^22 tiles
    static_assert(sizeof(scratch) >= 12 * (size_t)kNoallocPieces + 8 * (size_t)(kTileGrid + kFixGrid),
                  "the scratch holds the carries of 2^22 tiles");
    const uint64_t tiles = tiles_of(A);
    NKPR_CHECK(tiles <= kNoallocPieces, "matrix too large for the allocation-free step");
    launch_product<true>(A, x, shift, y, carve(csr_noalloc_scratch(), tiles), step_sq, s);
}

void csr_validate(const nkpr_csr *m, hipStream_t s) {
    const CsrView A = view_of(m);
    DevBuf flag;
    flag.alloc(4);
    NKPR_HIP(hipMemsetAsync(flag.p, 0, 4, s));
    hipLaunchKernelGGL(csr_check_kernel, dim3(2048), dim3(256), 0, s, A, m->cols, m->nnz,
                       flag.as<uint32_t>());
    NKPR_HIP(hipGetLastError());
    uint32_t bad = 0;
    uint64_t first = 0, last = 0;
    read_back(s, {{&bad, flag.p, 4}, {&first, A.row_idx, 8}, {&last, A.row_idx + A.rows, 8}});
    NKPR_CHECK(bad == 0 && first == 0 && last == m->nnz,
               "malformed CSR matrix (row_idx must rise from 0 to nnz, column indices < cols)");
}

void algebraic_pagerank_impl(const nkpr_csr *m, double damp, double tol, uint64_t max_iterations,
                             double *scores, int32_t scores_on_device, uint64_t *iterations) {
    const CsrView A = view_of(m);
    NKPR_CHECK(m->rows == m->cols, "AlgebraicPageRank needs a square matrix");
    NKPR_CHECK(m->rows > 0, "AlgebraicPageRank needs at least one row");
    NKPR_CHECK(scores != nullptr, "scores must not be NULL");
    NKPR_CHECK(damp >= 0.0 && damp <= 1.0, "damp must lie in [0, 1]");
    NKPR_CHECK(tol >= 0.0, "tol must be >= 0");
    NKPR_CHECK(max_iterations >= 1, "max_iterations must be >= 1");
    const uint64_t n = A.rows, nnz = m->nnz, tiles = tiles_of(A);
    // buffers first: the stream owner below is destroyed (and synchronised) before them
    DevBuf xa, xb, work, out, flag;
    xa.alloc(8 * n);
    xb.alloc(8 * n);
    work.alloc(std::max<size_t>(work_bytes(tiles), 8 * 1024));
    out.alloc(16);
    flag.alloc(4);
    int device = 0;
    NKPR_HIP(hipGetDevice(&device));
    const hipStream_t s = stream_get();
    struct StreamOwner {
        hipStream_t s;
        int device;
        ~StreamOwner() { stream_put(s, device); }
    } owner{s, device};
    // the reference reads whatever the indices point at; here a malformed matrix is an error
    hipLaunchKernelGGL(csr_fill_kernel, dim3(1), dim3(64), 0, s, out.as<double>(), 2, 0.0);
    NKPR_HIP(hipMemsetAsync(flag.p, 0, 4, s));
    hipLaunchKernelGGL(csr_check_kernel, dim3(2048), dim3(256), 0, s, A, m->cols, nnz,
                       flag.as<uint32_t>());
    NKPR_HIP(hipGetLastError());
    uint32_t bad = 0;
    uint64_t last = 0;
    read_back(s, {{&bad, flag.p, 4}, {&last, A.row_idx + n, 8}});
    NKPR_CHECK(bad == 0 && last == nnz,
               "malformed CSR matrix (row_idx must rise from 0 to nnz, column indices < cols)");
    const TileWork w = carve(work.p, tiles);
    const double tele = (1.0 - damp) / (double)n;
    hipLaunchKernelGGL(csr_fill_kernel, dim3(1024), dim3(256), 0, s, xa.as<double>(), n,
                       1.0 / (double)n);
    NKPR_HIP(hipGetLastError());
    double *cur = xa.as<double>(), *nxt = xb.as<double>();
    uint64_t it = 0;
    double sq = 0.0;
    do {
        launch_product<true>(A, cur, tele, nxt, w, out.as<double>(), s);
        read_back(s, {{&sq, out.p, 8}});
        std::swap(cur, nxt);
        ++it;
    } while (std::sqrt(sq) > tol && it < max_iterations);
    hipLaunchKernelGGL(csr_sum_kernel, dim3(1024), dim3(kFinalThreads), 0, s, cur, n, work.as<double>());
    hipLaunchKernelGGL(csr_final_kernel, dim3(1), dim3(kFinalThreads), 0, s, work.as<double>(), 1024u,
                       out.as<double>());
    hipLaunchKernelGGL(csr_scale_kernel, dim3(1024), dim3(256), 0, s, cur, n, out.as<double>());
    NKPR_HIP(hipGetLastError());
    if (scores_on_device) {
        NKPR_HIP(hipMemcpyAsync(scores, cur, 8 * n, hipMemcpyDeviceToDevice, s));
        NKPR_HIP(hipStreamSynchronize(s));
    } else {
        read_back(s, {{scores, cur, 8 * n}});
    }
    if (iterations) *iterations = it;
}

}  // namespace nkpr
