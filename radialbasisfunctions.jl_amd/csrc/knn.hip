// Exact grid-hashed k nearest neighbours for gfx950.
//
// Replaces find_neighbors (src/utils.jl:12-18: KDTree + knn(tree, eval, k, true)).
// The result is the set of the k data points with the smallest squared Euclidean
// distance to each query, ascending, computed in FP64 in dimension order without
// fused multiply-adds (the same rounding a KD-tree query sees); equal distances
// are ordered by lower index.
//
// Data points are binned into a uniform grid (counting sort: count, scan, scatter),
// queries are binned into the same grid so that a wavefront works on spatially adjacent
// queries (queries that are the data points share their binning), and every query scans
// cells outward until no unvisited cell can hold a point closer than its current k-th
// neighbour: first the block of two rings around its cell, row by row from the nearest,
// then ring by ring. Clouds of up to 4,000 points are binned by one workgroup, grid sizing
// included, with no host round trip.
//
// The top-k list lives in registers. A lane's candidates wait in LDS and are merged 16 at
// a time (sorting networks on all lanes at once): inserting each as it came cost the whole
// wavefront one insertion per candidate, since some lane accepts nearly every one.
// Bound: latency of the dependent cell-range and point loads at small sizes, VALU issue of
// the merges beyond. Measured, whole search, before (three points per cell
// whatever k, rings from the first, each candidate inserted as it came) and now: 900 points,
// 2-D, k = 12: 172 -> 70 us (a wavefront per query: 28 us); 100,000, 3-D, k = 20: 444 -> 216 us
// (170 us); 4M, 2-D, k = 20: 3.49 -> 2.16 ms; 2M, 3-D, k = 40: 9.0 -> 5.2 ms (3.5 ms).
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <stdint.h>

#include <utility>

#include "knn.h"
#include "knn_grid.h"

namespace rbfx {

struct Grid {
    double lo[3];
    double inv_s;  // 1 / cell size
    double s;
    int n[3];      // cells per dimension
    int dim;
};

__device__ __forceinline__ int cell_coord(double x, double lo, double inv_s, int n)
{
    int c = (int)floor((x - lo) * inv_s);
    return c < 0 ? 0 : (c >= n ? n - 1 : c);
}

template <int DIM>
__device__ __forceinline__ int64_t cell_of(const double* p, const Grid& G)
{
    int64_t id = 0;
#pragma unroll
    for (int d = DIM - 1; d >= 0; --d) id = id * G.n[d] + cell_coord(p[d], G.lo[d], G.inv_s, G.n[d]);
    return id;
}

// ---------------------------------------------------------------- bbox
// min / max of three coordinates over a workgroup of T threads (result in every thread 0..63)
template <int T>
__device__ __forceinline__ void block_box(double (&v)[6], double* lds)
{
#pragma unroll
    for (int s = 1; s < 64; s <<= 1)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            v[d] = fmin(v[d], __shfl_xor(v[d], s, 64));
            v[3 + d] = fmax(v[3 + d], __shfl_xor(v[3 + d], s, 64));
        }
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int d = 0; d < 6; ++d) lds[(threadIdx.x >> 6) * 6 + d] = v[d];
    __syncthreads();
#pragma unroll
    for (int w = 0; w < T / 64; ++w)
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            v[d] = fmin(v[d], lds[w * 6 + d]);
            v[3 + d] = fmax(v[3 + d], lds[w * 6 + 3 + d]);
        }
    __syncthreads();
}

__device__ __forceinline__ void box_of(const double* __restrict__ x, int64_t n, int dim, int64_t i, int64_t step,
                                       double (&v)[6])
{
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        v[d] = 1e300;
        v[3 + d] = -1e300;
    }
    for (; i < n; i += step)
#pragma unroll
        for (int d = 0; d < 3; ++d)
            if (d < dim) {
                const double c = x[i * dim + d];
                v[d] = fmin(v[d], c);
                v[3 + d] = fmax(v[3 + d], c);
            }
}

// Partial boxes, and the last workgroup to finish reduces them into `out` (pinned host
// memory) and clears the counter for the next call.
constexpr int kBoxBlocks = 256;
__global__ __launch_bounds__(256) void k_bbox(const double* __restrict__ x, int64_t n, int dim, double* part,
                                              unsigned int* done, double* out)
{
    __shared__ double lds[4 * 6];
    __shared__ unsigned int s_rank;
    double v[6];
    box_of(x, n, dim, blockIdx.x * (int64_t)256 + threadIdx.x, (int64_t)gridDim.x * 256, v);
    block_box<256>(v, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int d = 0; d < 6; ++d)
            __hip_atomic_store(&part[blockIdx.x * 6 + d], v[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __threadfence();
        s_rank = atomicAdd(done, 1u);
    }
    __syncthreads();
    if (s_rank != gridDim.x - 1) return;
    __threadfence();
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        v[d] = 1e300;
        v[3 + d] = -1e300;
    }
    if (threadIdx.x < gridDim.x)
#pragma unroll
        for (int d = 0; d < 6; ++d)
            v[d] = __hip_atomic_load(&part[threadIdx.x * 6 + d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    block_box<256>(v, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int d = 0; d < 6; ++d) out[d] = v[d];
        *done = 0u;
    }
}

// ---------------------------------------------------------------- binning
// plain fill kernel rather than a memset node, so the sequence stays capturable
__global__ void k_fill_i32(int32_t* __restrict__ p, int64_t n, int32_t v)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

template <int DIM>
__global__ void k_cell_count(const double* __restrict__ x, int64_t n, Grid G, int32_t* __restrict__ cell,
                             int32_t* __restrict__ count, Grid* out)
{
    if (out && blockIdx.x == 0 && threadIdx.x == 0) *out = G;  // (for the search, which reads it from memory)
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t c = (int32_t)cell_of<DIM>(x + i * DIM, G);
        cell[i] = c;
        atomicAdd(&count[c], 1);
    }
}

template <int DIM>
__global__ void k_scatter(const double* __restrict__ x, int64_t n, const int32_t* __restrict__ cell,
                          const int32_t* __restrict__ start, int32_t* __restrict__ count,
                          int32_t* __restrict__ sorted_idx, double* __restrict__ sorted_x)
{
    // (the counts run back down to zero as the slots are dealt out, last first)
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t slot = start[cell[i]] + atomicSub(&count[cell[i]], 1) - 1;
        sorted_idx[slot] = (int32_t)i;
        if (sorted_x)
#pragma unroll
            for (int d = 0; d < DIM; ++d) sorted_x[(int64_t)slot * DIM + d] = x[i * DIM + d];
    }
}

// ---------------------------------------------------------------- query
// (d2, idx) lexicographic order
__device__ __forceinline__ bool lt(double a, int ia, double b, int ib) { return a < b || (a == b && ia < ib); }

template <int DIM>
__device__ __forceinline__ double sqdist(const double* a, const double (&q)[DIM])
{
    // no contraction: same rounding as sum((x .- y).^2) evaluated term by term. The
    // operators must be written here, inside the pragma's scope: arithmetic helpers
    // defined elsewhere keep their own contraction setting and were fused into FMAs.
#pragma clang fp contract(off)
    double s = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const double t = a[d] - q[d];
        const double t2 = t * t;
        s = s + t2;
    }
    return s;
}

// ---------------------------------------------------------------- small clouds
constexpr int kSmallPoints = 4000;
constexpr int kSmallCells = 4 * kSmallPoints + 16;  // (knn_grid_size's bound; 64,064 bytes of LDS)

// Bounding box, grid, counting sort: one workgroup (512 threads: the grid sizing needs the
// registers that 1,024 would not leave).
constexpr int kSmallThreads = 512;
template <int DIM>
__global__ __launch_bounds__(kSmallThreads) void k_bin_small(const double* __restrict__ x, int n, double target, Grid* grid,
                                                    int32_t* __restrict__ start, int32_t* __restrict__ sorted_idx,
                                                    double* __restrict__ sorted_x)
{
    __shared__ int32_t cnt[kSmallCells];
    __shared__ double lds[kSmallThreads / 64 * 6];
    __shared__ int wsum[kSmallThreads / 64];
    __shared__ Grid G;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    double v[6];
    box_of(x, n, DIM, t, kSmallThreads, v);
    block_box<kSmallThreads>(v, lds);
    if (t == 0) {
        double ext[3];
        for (int d = 0; d < 3; ++d) ext[d] = v[3 + d] - v[d];
        G.dim = DIM;
        knn_grid_size(DIM, ext, n, &G.s, G.n, target);
        G.inv_s = 1.0 / G.s;
        for (int d = 0; d < 3; ++d) G.lo[d] = d < DIM ? v[d] : 0.0;
        *grid = G;
    }
    __syncthreads();
    const int ncell = G.n[0] * G.n[1] * G.n[2];
    for (int c = t; c < ncell; c += kSmallThreads) cnt[c] = 0;
    __syncthreads();
    for (int i = t; i < n; i += kSmallThreads) atomicAdd(&cnt[cell_of<DIM>(x + (int64_t)i * DIM, G)], 1);
    __syncthreads();
    // exclusive scan: each thread a run of cells, then over the threads
    const int run = (ncell + kSmallThreads - 1) / kSmallThreads, c0 = t * run;
    int sum = 0;
    for (int c = c0; c < c0 + run && c < ncell; ++c) sum += cnt[c];
    int inc = sum;
    for (int s = 1; s < 64; s <<= 1) {
        const int o = __shfl_up(inc, s, 64);
        if (lane >= s) inc += o;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    int at = inc - sum;
    for (int q = 0; q < w; ++q) at += wsum[q];
    for (int c = c0; c < c0 + run && c < ncell; ++c) {
        const int k = cnt[c];
        cnt[c] = at;
        start[c] = at;
        at += k;
    }
    if (t == 0) start[ncell] = n;
    __syncthreads();
    for (int i = t; i < n; i += kSmallThreads) {
        const int slot = atomicAdd(&cnt[cell_of<DIM>(x + (int64_t)i * DIM, G)], 1);
        sorted_idx[slot] = i;
#pragma unroll
        for (int d = 0; d < DIM; ++d) sorted_x[(int64_t)slot * DIM + d] = x[(int64_t)i * DIM + d];
    }
}

// ---------------------------------------------------------------- merging networks
struct NetPair {
    int a, b;
};
template <int CAP>
struct Net {
    int n = 0;
    NetPair c[CAP] = {};
};
// Batcher's odd-even mergesort of N = 2^m entries
template <int N>
constexpr Net<N * 8> sort_net()
{
    Net<N * 8> r;
    for (int p = 1; p < N; p *= 2)
        for (int k = p; k >= 1; k /= 2)
            for (int j = k % p; j + k < N; j += 2 * k)
                for (int i = 0; i < k; ++i)
                    if ((i + j) / (2 * p) == (i + j + k) / (2 * p) && i + j + k < N) r.c[r.n++] = {i + j, i + j + k};
    return r;
}
// merge of a bitonic sequence of P entries, the comparators that the first KEEP outputs need
template <int P, int KEEP>
constexpr Net<P * 4> merge_net()
{
    Net<P * 4> all, r;
    for (int k = P / 2; k >= 1; k /= 2)
        for (int i = 0; i < P; ++i)
            if ((i & k) == 0) all.c[all.n++] = {i, i + k};
    bool need[P] = {};
    bool use[P * 4] = {};
    for (int i = 0; i < KEEP; ++i) need[i] = true;
    for (int q = all.n - 1; q >= 0; --q)
        if (need[all.c[q].a] || need[all.c[q].b]) {
            use[q] = true;
            need[all.c[q].a] = need[all.c[q].b] = true;
        }
    for (int q = 0; q < all.n; ++q)
        if (use[q]) r.c[r.n++] = all.c[q];
    return r;
}

// (a, b) -> (smaller, larger) in (distance, index) order
__device__ __forceinline__ void comp(double& da, int& ia, double& db, int& ib)
{
    // (the instructions themselves: fmin would first quiet each operand; no NaN gets here)
    const bool sw = lt(db, ib, da, ia);
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(da), "v"(db));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(da), "v"(db));
    const int il = sw ? ib : ia, ih = sw ? ia : ib;
    da = lo;
    db = hi;
    ia = il;
    ib = ih;
}

template <int N, int... Q>
__device__ __forceinline__ void run_sort(double* d, int* i, std::integer_sequence<int, Q...>)
{
    constexpr auto net = sort_net<N>();
    (comp(d[net.c[Q].a], i[net.c[Q].a], d[net.c[Q].b], i[net.c[Q].b]), ...);
}
template <int P, int KEEP, int... Q>
__device__ __forceinline__ void run_merge(double* d, int* i, std::integer_sequence<int, Q...>)
{
    constexpr auto net = merge_net<P, KEEP>();
    (comp(d[net.c[Q].a], i[net.c[Q].a], d[net.c[Q].b], i[net.c[Q].b]), ...);
}

constexpr int kPend = 16;  // candidates waiting per lane

// KCAP sorted entries (bd, bi) and the lane's n pending candidates -> the KCAP smallest
template <int KCAP>
__device__ __forceinline__ void merge_pending(double (&bd)[KCAP], int (&bi)[KCAP], const double (*pd)[64],
                                              const int (*pi)[64], int n)
{
    constexpr int P = KCAP <= 16 ? 16 : 32;
    static_assert(KCAP <= 32, "longer lists are searched by wavefronts");
    const int lane = threadIdx.x & 63;
    double d[P];
    int i[P];
    double sd[kPend];
    int si[kPend];
#pragma unroll
    for (int u = 0; u < kPend; ++u) {
        const double dv = pd[u][lane];
        const int iv = pi[u][lane];
        sd[u] = u < n ? dv : __builtin_huge_val();
        si[u] = u < n ? iv : 0x7fffffff;
    }
    run_sort<kPend>(sd, si, std::make_integer_sequence<int, sort_net<kPend>().n>{});
    // the sorted candidates reversed behind the list: smaller of each overlapping pair
#pragma unroll
    for (int u = 0; u < P; ++u) {
        d[u] = u < KCAP ? bd[u < KCAP ? u : 0] : __builtin_huge_val();
        i[u] = u < KCAP ? bi[u < KCAP ? u : 0] : 0x7fffffff;
        if (P - 1 - u < kPend) {
            const double cd = sd[P - 1 - u < kPend ? P - 1 - u : 0];
            const int ci = si[P - 1 - u < kPend ? P - 1 - u : 0];
            const bool sw = lt(cd, ci, d[u], i[u]);
            d[u] = sw ? cd : d[u];
            i[u] = sw ? ci : i[u];
        }
    }
    run_merge<P, KCAP>(d, i, std::make_integer_sequence<int, merge_net<P, KCAP>().n>{});
#pragma unroll
    for (int u = 0; u < KCAP; ++u) {
        bd[u] = d[u];
        bi[u] = i[u];
    }
}

// rows (dy, dz) of the block of two rings, nearest first
__device__ constexpr int8_t kRowY[25] = {0, -1, 1, 0, 0, -1, 1, -1, 1, -2, 2, 0, 0, -2, -2, 2, 2, -1, 1, -1, 1, -2, 2, -2, 2};
__device__ constexpr int8_t kRowZ[25] = {0, 0, 0, -1, 1, -1, -1, 1, 1, 0, 0, -2, 2, -1, 1, -1, 1, -2, -2, 2, 2, -2, -2, 2, 2};
__device__ constexpr int8_t kRowY2[5] = {0, -1, 1, -2, 2};

template <int DIM, int KCAP>
__global__ __launch_bounds__(64) void k_query(const double* __restrict__ sx, const int32_t* __restrict__ sidx,
                                              const int32_t* __restrict__ cell_start,
                                              const double* __restrict__ query,
                                              const int32_t* __restrict__ qorder, int64_t n_query,
                                              const Grid* __restrict__ Gd, int kmax,
                                              const int64_t* __restrict__ q_ptr, int32_t* __restrict__ out)
{
    __shared__ double s_pd[kPend][64];
    __shared__ int s_pi[kPend][64];
    const int lane = threadIdx.x;
    const int64_t t = blockIdx.x * (int64_t)64 + lane;
    const Grid G = *Gd;
    const bool live = t < n_query;
    const int64_t qi = !live ? 0 : (qorder ? qorder[t] : t);
    double q[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) q[d] = query[qi * DIM + d];
    const int c0 = cell_coord(q[0], G.lo[0], G.inv_s, G.n[0]);
    const int c1 = DIM >= 2 ? cell_coord(q[DIM >= 2 ? 1 : 0], G.lo[1], G.inv_s, G.n[1]) : 0;
    const int c2 = DIM == 3 ? cell_coord(q[DIM - 1], G.lo[2], G.inv_s, G.n[2]) : 0;

    double bd[KCAP];
    int bi[KCAP];
    // slots [0, KCAP-kmax) hold sentinels below every real distance, so the threshold is
    // always the last slot
#pragma unroll
    for (int s = 0; s < KCAP; ++s) {
        bd[s] = (s < KCAP - kmax) ? -1.0 : __builtin_huge_val();
        bi[s] = (s < KCAP - kmax) ? -1 : 0x7fffffff;
    }
    auto row_id = [&](int cy, int cz) { return ((int64_t)cz * G.n[1] + cy) * G.n[0]; };
    // squared distance from the query to the box of cells [xl, xh] x cy x cz: no closer point
    // (relative to the grid's corner, so nothing is rounded at the size of the coordinates)
    auto side = [&](int d, int lo_cell, int hi_cell) __attribute__((always_inline)) {
        const double at = q[d] - G.lo[d];
        const double g = fmax(lo_cell * G.s - at, at - (hi_cell + 1) * G.s);
        return g > 0.0 ? g * g : 0.0;
    };
    auto run_gap = [&](int xl, int xh, int cy, int cz) __attribute__((always_inline)) {
        double g2 = side(0, xl, xh);
        if constexpr (DIM >= 2) g2 += side(1, cy, cy);
        if constexpr (DIM == 3) g2 += side(2, cz, cz);
        return g2 * (1.0 - 1e-9);
    };
    // whether the k-th neighbour is closer than everything outside the visited rings
    int maxn = G.n[0];
    if (DIM >= 2) maxn = max(maxn, G.n[1]);
    if (DIM == 3) maxn = max(maxn, G.n[2]);
    auto settled = [&](int rho) {
        double bound = 1e300;
        bool covers_all = true;
        auto side_bound = [&](int d, int cd) __attribute__((always_inline)) {
            const double at = q[d] - G.lo[d];
            if (cd - rho > 0) bound = fmin(bound, at - (cd - rho) * G.s);
            if (cd + rho + 1 < G.n[d]) bound = fmin(bound, (cd + rho + 1) * G.s - at);
            if (cd - rho > 0 || cd + rho + 1 < G.n[d]) covers_all = false;
        };
        side_bound(0, c0);
        if constexpr (DIM >= 2) side_bound(1, c1);
        if constexpr (DIM == 3) side_bound(2, c2);
        if (covers_all || rho > maxn) return true;
        return bi[KCAP - 1] != 0x7fffffff && bound > 0.0 && bd[KCAP - 1] < bound * bound * (1.0 - 1e-9);
    };

    // One loop over runs of cells: first the rows of the block of two rings, nearest first,
    // then, for the lanes that are not settled, ring by ring (whole rows on a ring's faces,
    // the two end cells elsewhere). The next run's range is loaded while a run is scanned.
    // Within a run, four candidates per step as long as any lane has some; a merge when any
    // lane might run out of room, and at the end of the block and of each ring. (The loop
    // holds the only copy of the merge.)
    // A wavefront most of whose lanes find eight times the mean in their first row, between an
    // eighth and half of it in their own cell, stands in a wide cluster, where the two rings
    // hold far more than the k nearest: it goes ring by ring from its own cells (300,000
    // points, a cluster of up to 400 times the mean density, k = 20: 3.38 -> 2.61 ms in 2-D;
    // where a single cell holds the row, the other order is the faster one: 11.2 against 14 ms).
    constexpr int R0 = 2, NROW = DIM == 1 ? 1 : (DIM == 2 ? 5 : 25), STEP = 4;
    int np = 0;  // pending candidates
    int rho = R0, j = 0, dy = 0, dz = 0, part = 0;
    bool block = true;
    bool open = live;
    struct Run {
        int32_t s0, s1;
        double gap;
        bool in, last;
    };
    auto next = [&]() __attribute__((always_inline)) {
        Run r;
        int cy, cz, xl = c0 - rho, xh = c0 + rho;
        bool in = open;
        if (block) {
            cy = c1 + (DIM == 3 ? kRowY[j] : (DIM == 2 ? kRowY2[j] : 0));
            cz = c2 + (DIM == 3 ? kRowZ[j] : 0);
            r.last = ++j == NROW;
        } else {
            cy = c1 + dy;
            cz = c2 + dz;
            const bool face = (DIM == 3 && (dz == -rho || dz == rho)) || (DIM >= 2 && (dy == -rho || dy == rho));
            if (!face) {
                if (part == 0) {
                    in = in && xl >= 0;
                    xh = xl;
                } else {
                    in = in && xh < G.n[0];
                    xl = xh;
                }
            }
            part = face ? 0 : part ^ 1;
            const bool step = part == 0, wrap = !(DIM >= 2 && dy < rho);
            dz += step && wrap ? 1 : 0;
            dy = !step ? dy : (wrap ? (DIM >= 2 ? -rho : 0) : dy + 1);
            r.last = part == 0 && (DIM == 3 ? dz > rho : dz > 0);
        }
        r.in = in && cy >= 0 && cy < G.n[1] && cz >= 0 && cz < G.n[2];
        r.gap = run_gap(xl, xh, cy, cz);
        r.in = r.in && (r.gap < bd[KCAP - 1] || bi[KCAP - 1] == 0x7fffffff);
        r.s0 = r.s1 = 0;
        if (r.in) {
            const int64_t id = row_id(cy, cz);
            r.s0 = cell_start[id + max(xl, 0)];
            r.s1 = cell_start[id + min(xh, G.n[0] - 1) + 1];
        }
        return r;
    };
    Run cur = next();
    if (DIM >= 2 && __popcll(__ballot(cur.s1 - cur.s0 > 4 * kmax)) > 32) {
        const int64_t own = row_id(c1, c2) + c0;
        const int32_t n_own = cell_start[own + 1] - cell_start[own], n_row = cur.s1 - cur.s0;
        if (__popcll(__ballot(n_row > 4 * kmax && 2 * n_own < n_row && n_row < 8 * n_own)) > 32) {
            block = false;
            rho = 0;
            cur = next();
        }
    }
    for (;;) {
        Run nxt;
        if (!cur.last) nxt = next();
        // (a run wholly farther than the k-th neighbour so far holds nothing)
        int32_t s0 = cur.s0;
        const int32_t s1 = cur.gap < bd[KCAP - 1] || bi[KCAP - 1] == 0x7fffffff ? cur.s1 : s0;
        bool more = __ballot(s0 < s1) != 0ull;
        while (more || cur.last) {
            if (more) {
                double x[STEP][DIM];
                int id[STEP];
#pragma unroll
                for (int u = 0; u < STEP; ++u) {
                    const int32_t s = s0 + u < s1 ? s0 + u : (s0 < s1 ? s0 : 0);
#pragma unroll
                    for (int d = 0; d < DIM; ++d) x[u][d] = sx[(int64_t)s * DIM + d];
                    id[u] = sidx[s];
                }
#pragma unroll
                for (int u = 0; u < STEP; ++u) {
                    const double d2 = sqdist<DIM>(x[u], q);
                    if (s0 + u < s1 && lt(d2, id[u], bd[KCAP - 1], bi[KCAP - 1])) {
                        s_pd[np][lane] = d2;
                        s_pi[np][lane] = id[u];
                        ++np;
                    }
                }
                s0 += STEP;
                more = __ballot(s0 < s1) != 0ull;
            }
            const bool full = __ballot(np > kPend - STEP) != 0ull;
            if (full || (cur.last && !more)) {
                merge_pending<KCAP>(bd, bi, s_pd, s_pi, np);
                np = 0;
            }
            if (!more) break;
        }
        if (cur.last) {
            open = open && !settled(rho);
            if (!__ballot(open)) break;
            block = false;
            ++rho;
            dy = DIM >= 2 ? -rho : 0;
            dz = DIM == 3 ? -rho : 0;
            part = 0;
            cur = next();
        } else {
            cur = nxt;
        }
    }
    if (!live) return;
    const int64_t base = q_ptr ? q_ptr[qi] : qi * (int64_t)kmax;
    const int kq = q_ptr ? (int)(q_ptr[qi + 1] - q_ptr[qi]) : kmax;
#pragma unroll
    for (int s = 0; s < KCAP; ++s) {
        const int o = s - (KCAP - kmax);
        if (o >= 0 && o < kq) out[base + o] = bi[s];
    }
}

// ---------------------------------------------------------------- few queries
// A wavefront per query, for lists too long for a lane's registers and for searches too small
// to fill the chip with a lane per query
// (where one wavefront's chain of runs and merges takes 36 us whatever the count): bound by
// the latency of its few dependent loads. The runs
// of cells are looked up by one lane each, their candidates taken 64 at a time, and a
// batch with many that beat the k-th so far is sorted over the lanes (DPP moves) and merged
// with the list; a batch with few is merged by rank: each is broadcast, and every lane
// counts how many come before its own. The distances, their order and the stopping test
// are k_query's, so the result is the same.
__device__ __forceinline__ int rdlane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ double rdlane(double v, int l)
{
    return __hiloint2double(rdlane(__double2hiint(v), l), rdlane(__double2loint(v), l));
}

// the value of lane ^ X: DPP moves inside a row of 16 lanes, a permute beyond
template <int X>
__device__ __forceinline__ int lane_xor(int v)
{
    if constexpr (X == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);
    else if constexpr (X == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);
    else if constexpr (X == 3) return __builtin_amdgcn_mov_dpp(v, 0x1B, 0xF, 0xF, true);
    else if constexpr (X == 4) return lane_xor<3>(__builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true));
    else if constexpr (X == 7) return __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true);   // row_half_mirror
    else if constexpr (X == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true);   // row_ror:8
    else if constexpr (X == 15) return __builtin_amdgcn_mov_dpp(v, 0x140, 0xF, 0xF, true);  // row_mirror
    else return __shfl_xor(v, X, 64);
}
template <int X>
__device__ __forceinline__ double lane_xor(double v)
{
    return __hiloint2double(lane_xor<X>(__double2hiint(v)), lane_xor<X>(__double2loint(v)));
}

// lanes l and l ^ X keep the smaller and the larger of their entries, the smaller in the
// lower lane
template <int X>
__device__ __forceinline__ void exchange(double& d, int& i, int lane)
{
    constexpr int top = X >= 32 ? 32 : (X >= 16 ? 16 : (X >= 8 ? 8 : (X >= 4 ? 4 : (X >= 2 ? 2 : 1))));
    const double od = lane_xor<X>(d);
    const int oi = lane_xor<X>(i);
    const bool take = lt(od, oi, d, i) == ((lane & top) == 0);
    d = take ? od : d;
    i = take ? oi : i;
}
// ascending over the 64 lanes (bitonic, each merge begun by the mirrored exchange)
__device__ __forceinline__ void lane_sort(double& d, int& i, int lane)
{
    exchange<1>(d, i, lane);
    exchange<3>(d, i, lane);
    exchange<1>(d, i, lane);
    exchange<7>(d, i, lane);
    exchange<2>(d, i, lane);
    exchange<1>(d, i, lane);
    exchange<15>(d, i, lane);
    exchange<4>(d, i, lane);
    exchange<2>(d, i, lane);
    exchange<1>(d, i, lane);
    exchange<31>(d, i, lane);
    exchange<8>(d, i, lane);
    exchange<4>(d, i, lane);
    exchange<2>(d, i, lane);
    exchange<1>(d, i, lane);
    exchange<63>(d, i, lane);
    exchange<16>(d, i, lane);
    exchange<8>(d, i, lane);
    exchange<4>(d, i, lane);
    exchange<2>(d, i, lane);
    exchange<1>(d, i, lane);
}
// the 64 smallest of two ascending lists, ascending
__device__ __forceinline__ void lane_merge(double& d, int& i, double nd, int ni, int lane)
{
    const double rd = lane_xor<63>(nd);
    const int ri = lane_xor<63>(ni);
    const bool take = lt(rd, ri, d, i);
    d = take ? rd : d;
    i = take ? ri : i;
    exchange<32>(d, i, lane);
    exchange<16>(d, i, lane);
    exchange<8>(d, i, lane);
    exchange<4>(d, i, lane);
    exchange<2>(d, i, lane);
    exchange<1>(d, i, lane);
}
// inclusive sum over the 64 lanes
__device__ __forceinline__ int lane_sum(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);   // row_shr:1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // lane 15 of a row to the next one
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // lane 31 to the upper half
    return v;
}

// candidates of the block of two rings that are read at once (eight batches; a uniform cloud's
// hold 50 to 330): 300,000 points, k = 40, most in a cluster of up to 400 times the mean density:
// 2-D 12.2 ms with blocks of any size, 2.0 with this limit (6.9 before there were wavefront
// searches); 3-D 107 and 8.5
constexpr int kBlockMost = 512;
// candidates that a batch merges by rank (14 instructions each) rather than by sorting (280)
constexpr int kRankMerge = 12;

template <int DIM>
__global__ __launch_bounds__(256) void k_query_wave(const double* __restrict__ sx, const int32_t* __restrict__ sidx,
                                                    const int32_t* __restrict__ cell_start,
                                                    const double* __restrict__ query, const int32_t* __restrict__ qorder,
                                                    int64_t n_query,
                                                    const Grid* __restrict__ Gd, int kmax,
                                                    const int64_t* __restrict__ q_ptr, int32_t* __restrict__ out)
{
    __shared__ double s_d[4][64];
    __shared__ int s_i[4][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t t = blockIdx.x * (int64_t)4 + w;
    if (t >= n_query) return;
    const int64_t qi = qorder ? qorder[t] : t;
    const Grid G = *Gd;
    double q[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) q[d] = query[qi * DIM + d];
    const int c0 = cell_coord(q[0], G.lo[0], G.inv_s, G.n[0]);
    const int c1 = DIM >= 2 ? cell_coord(q[DIM >= 2 ? 1 : 0], G.lo[1], G.inv_s, G.n[1]) : 0;
    const int c2 = DIM == 3 ? cell_coord(q[DIM - 1], G.lo[2], G.inv_s, G.n[2]) : 0;
    int maxn = G.n[0];
    if (DIM >= 2) maxn = max(maxn, G.n[1]);
    if (DIM == 3) maxn = max(maxn, G.n[2]);

    // the nearest 64 so far, ascending, one per lane; the k-th of them
    // (kd read from a lane: as a constant, the compiler loads this infinity into a scalar pair
    // with one 64-bit literal, which the hardware does not have, and gets 0)
    double bd = __builtin_huge_val();
    asm volatile("" : "+v"(bd));
    double kd = rdlane(bd, 0);
    int bi = 0x7fffffff, ki = bi, ki0 = bi;
    auto side = [&](int d, int lo_cell, int hi_cell) __attribute__((always_inline)) {
        const double at = q[d] - G.lo[d];
        const double g = fmax(lo_cell * G.s - at, at - (hi_cell + 1) * G.s);
        return g > 0.0 ? g * g : 0.0;
    };
    // The candidates of up to 64 runs of cells: rows of the block of two rings, or of ring rho
    // (whole on its faces, else the two end cells, one id each; only those closer than the
    // k-th so far). False, with nothing read, for a block of more than kBlockMost.
    auto scan = [&](auto blk, const int rho, const int id0, const int n_ids) __attribute__((always_inline)) {
        constexpr bool BLOCK = decltype(blk)::value;
        const int W = 2 * rho + 1;
        const int id = id0 + lane, r = BLOCK ? id : id >> 1, part = BLOCK ? 0 : id & 1;
        const int dy = DIM >= 2 ? r % W - rho : 0, dz = DIM == 3 ? r / W - rho : 0;
        const int cy = c1 + dy, cz = c2 + dz;
        const bool face = BLOCK || rho == 0 || (DIM >= 2 && (dy == -rho || dy == rho)) ||
                          (DIM == 3 && (dz == -rho || dz == rho));
        int xl = c0 - rho, xh = c0 + rho;
        bool in = id < n_ids && cy >= 0 && cy < G.n[1] && cz >= 0 && cz < G.n[2];
        if (face) {
            in = in && part == 0;
        } else if (part == 0) {
            in = in && xl >= 0;
            xh = xl;
        } else {
            in = in && xh < G.n[0];
            xl = xh;
        }
        if (!BLOCK && ki != 0x7fffffff) {
            double g2 = side(0, xl, xh);
            if constexpr (DIM >= 2) g2 += side(1, cy, cy);
            if constexpr (DIM == 3) g2 += side(2, cz, cz);
            in = in && g2 * (1.0 - 1e-9) < kd;
        }
        int32_t s0 = 0, cnt = 0;
        if (in) {
            const int64_t row = ((int64_t)cz * G.n[1] + cy) * G.n[0];
            s0 = cell_start[row + max(xl, 0)];
            cnt = cell_start[row + min(xh, G.n[0] - 1) + 1] - s0;
        }
        // candidate f of the batch lies in the first run whose inclusive count exceeds it
        const int inc = lane_sum(cnt), n_run = min(n_ids - id0, 64);
        const int total = rdlane(inc, 63);
        if (BLOCK && total > kBlockMost) return false;
        const int base = s0 - (inc - cnt);
        for (int f0 = 0; f0 < total; f0 += 64) {
            const int f = f0 + lane;
            int run = 0;
            for (int s = n_run > 32 ? 32 : (n_run > 16 ? 16 : (n_run > 4 ? 8 : 2)); s; s >>= 1) {
                const int v = __shfl(inc, run + s - 1, 64);
                run += v <= f ? s : 0;
            }
            const int b = __shfl(base, run & 63, 64);
            double cd = __builtin_huge_val();
            int ci = 0x7fffffff;
            if (f < total) {
                double x[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) x[d] = sx[(int64_t)(b + f) * DIM + d];
                cd = sqdist<DIM>(x, q);
                ci = sidx[b + f];
            }
            const bool pass = f < total && lt(cd, ci, kd, ki);
            const unsigned long long m = __ballot(pass);
            if (!m) continue;
            if (__popcll(m) > kRankMerge) {
                cd = pass ? cd : __builtin_huge_val();
                ci = pass ? ci : 0x7fffffff;
                lane_sort(cd, ci, lane);
                if (ki0 == 0x7fffffff) {  // nothing yet
                    bd = cd;
                    bi = ci;
                } else {
                    lane_merge(bd, bi, cd, ci, lane);
                }
                kd = rdlane(bd, kmax - 1);
                ki = rdlane(bi, kmax - 1);
                ki0 = rdlane(bi, 0);
                continue;
            }
            int rb = lane, rn = 0;
            for (unsigned long long left = m; left; left &= left - 1) {
                const int l = __builtin_ctzll(left);
                const double nd = rdlane(cd, l);
                const int ni = rdlane(ci, l);
                const bool before = lt(nd, ni, bd, bi);
                rb += before ? 1 : 0;
                rn += lt(nd, ni, cd, ci) ? 1 : 0;
                const int ahead = 64 - __popcll(__ballot(before));
                rn += lane == l ? ahead : 0;
            }
            if (rb < 64) {
                s_d[w][rb] = bd;
                s_i[w][rb] = bi;
            }
            if (pass && rn < 64) {
                s_d[w][rn] = cd;
                s_i[w][rn] = ci;
            }
            // (a wavefront's LDS accesses complete in order)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            bd = s_d[w][lane];
            bi = s_i[w][lane];
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            kd = rdlane(bd, kmax - 1);
            ki = rdlane(bi, kmax - 1);
            ki0 = rdlane(bi, 0);
        }
        return true;
    };
    // (k_query's stopping test)
    auto settled = [&](const int rho) {
        double bound = 1e300;
        bool covers_all = true;
        auto side_bound = [&](int d, int cd) __attribute__((always_inline)) {
            const double at = q[d] - G.lo[d];
            if (cd - rho > 0) bound = fmin(bound, at - (cd - rho) * G.s);
            if (cd + rho + 1 < G.n[d]) bound = fmin(bound, (cd + rho + 1) * G.s - at);
            if (cd - rho > 0 || cd + rho + 1 < G.n[d]) covers_all = false;
        };
        side_bound(0, c0);
        if constexpr (DIM >= 2) side_bound(1, c1);
        if constexpr (DIM == 3) side_bound(2, c2);
        return covers_all || rho > maxn || (ki != 0x7fffffff && bound > 0.0 && kd < bound * bound * (1.0 - 1e-9));
    };
    // The block of two rings, then ring by ring; in a cluster, where the block holds far more
    // than the k nearest, ring by ring from the query's own cell.
    const bool whole = scan(std::true_type{}, 2, 0, DIM == 1 ? 1 : (DIM == 2 ? 5 : 25));
    if (!whole || !settled(2))
        for (int rho = whole ? 3 : 0;; ++rho) {
            const int W = 2 * rho + 1, n_ids = rho == 0 ? 1 : 2 * (DIM == 1 ? 1 : (DIM == 2 ? W : W * W));
            for (int id0 = 0; id0 < n_ids; id0 += 64) scan(std::false_type{}, rho, id0, n_ids);
            if (settled(rho)) break;
        }
    const int64_t base = q_ptr ? q_ptr[qi] : qi * (int64_t)kmax;
    const int kq = q_ptr ? (int)(q_ptr[qi + 1] - q_ptr[qi]) : kmax;
    if (lane < kq && lane < kmax) out[base + lane] = bi;
}

// ---------------------------------------------------------------- processing order
__device__ __forceinline__ uint32_t compact_bits(uint32_t m, int dim, int d)
{
    uint32_t r = 0;
    for (int b = 0; b * dim + d < 31; ++b) r |= ((m >> (b * dim + d)) & 1u) << b;
    return r;
}
// number of points of each cell along the Z-curve (0 beyond the grid)
__global__ __launch_bounds__(256) void k_curve_count(Grid G, int64_t n_curve, const int32_t* __restrict__ start,
                                                     int32_t* __restrict__ cnt)
{
    const int64_t m = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (m > n_curve) return;
    int v = 0;
    if (m < n_curve) {
        int x[3];
        bool in = true;
        for (int d = 0; d < 3; ++d) {
            x[d] = d < G.dim ? (int)compact_bits((uint32_t)m, G.dim, d) : 0;
            in = in && x[d] < G.n[d];
        }
        if (in) {
            const int64_t c = ((int64_t)x[2] * G.n[1] + x[1]) * G.n[0] + x[0];
            v = start[c + 1] - start[c];
        }
    }
    cnt[m] = v;
}
__global__ __launch_bounds__(256) void k_curve_place(Grid G, int64_t n_curve, const int32_t* __restrict__ start,
                                                     const int32_t* __restrict__ at, const int32_t* __restrict__ sorted,
                                                     int32_t* __restrict__ order)
{
    const int64_t m = blockIdx.x * (int64_t)256 + threadIdx.x;
    if (m >= n_curve) return;
    int x[3];
    for (int d = 0; d < 3; ++d) {
        x[d] = d < G.dim ? (int)compact_bits((uint32_t)m, G.dim, d) : 0;
        if (x[d] >= G.n[d]) return;
    }
    const int64_t c = ((int64_t)x[2] * G.n[1] + x[1]) * G.n[0] + x[0];
    const int32_t b = start[c], e = start[c + 1];
    int32_t o = at[m];
    for (int32_t s = b; s < e; ++s) order[o++] = sorted[s];
}

// ---------------------------------------------------------------- driver
static hipError_t grow(void** p, size_t& cap, size_t need)
{
    if (need <= cap) return hipSuccess;
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    cap = 0;
    hipError_t e = hipMalloc(p, need);
    if (e == hipSuccess) cap = need;
    return e;
}

static hipError_t scan(KnnWorkspace& ws, const int32_t* in, int32_t* out, int64_t n, hipStream_t st)
{
    size_t need = 0;
    hipError_t e = hipcub::DeviceScan::ExclusiveSum(nullptr, need, in, out, (int)n, st);
    if (e == hipSuccess) e = grow(&ws.scan_tmp, ws.scan_tmp_bytes, need + 256);
    if (e != hipSuccess) return e;
    size_t have = ws.scan_tmp_bytes;
    return hipcub::DeviceScan::ExclusiveSum(ws.scan_tmp, have, in, out, (int)n, st);
}

// Searches that take a wavefront per query: all of more than 32 neighbours (a lane's list of
// 64 no longer hides its merges: 3M points, 2-D, k = 60: 6.6 ms against 11.9 with a lane per
// query; k = 35: 4.5 and 5.0), the others up to the count where lanes catch up. Whole
// searches in us, a wavefront and a lane per query: 2-D, k = 13: 900 points 28 and 61, 65,000
// 102 and 95, 300,000 294 and 169; k = 20: 900 31 and 111, 100,000 163 and 170, 150,000 220
// and 189; 3-D, k = 20: 900 34 and 190, 100,000 170 and 208, 300,000 419 and 406 (Halton)
// or 405 and 515 (random), 1M 1193 and 976.
constexpr int kMaxLaneList = 32;
static bool query_by_wavefront(int dim, int k, int64_t n_query)
{
    return k > kMaxLaneList || n_query <= (dim == 3 ? 262144 : 65536);
}

// the register list costs merges and VGPRs with KCAP, so KCAP follows k closely in the
// common range
template <int DIM>
static hipError_t launch_query(const KnnWorkspace& ws, const double* query, const int32_t* qorder, int64_t n_query,
                               int k, const int64_t* q_ptr, int32_t* out, hipStream_t st)
{
    if (query_by_wavefront(DIM, k, n_query)) {
        // (the spatial order pays for its load once the points outgrow the caches)
        hipLaunchKernelGGL(k_query_wave<DIM>, dim3((unsigned)((n_query + 3) / 4)), dim3(256), 0, st, ws.sx, ws.sidx,
                           ws.start, query, n_query > 16384 ? qorder : nullptr, n_query, (const Grid*)ws.grid, k, q_ptr, out);
        return hipGetLastError();
    }
    const dim3 gq((unsigned)((n_query + 63) / 64));
#define RBFX_KNN_LAUNCH(KC)                                                                                  \
    if (k <= KC) {                                                                                           \
        hipLaunchKernelGGL((k_query<DIM, KC>), gq, dim3(64), 0, st, ws.sx, ws.sidx, ws.start, query, qorder, \
                           n_query, (const Grid*)ws.grid, k, q_ptr, out);                                                   \
        return hipGetLastError();                                                                            \
    }
    RBFX_KNN_LAUNCH(16)
    RBFX_KNN_LAUNCH(20)
    RBFX_KNN_LAUNCH(24)
    RBFX_KNN_LAUNCH(kMaxLaneList)
#undef RBFX_KNN_LAUNCH
    return hipErrorInvalidValue;
}

// Z-curve order of the binned queries, by a counting sort over the curve. A grid whose
// curve is mostly outside it (very unequal sides) keeps the row-by-row cell order.
static hipError_t curve_order(KnnWorkspace& ws, const Grid& G, int64_t ncell, const int32_t* start,
                              const int32_t* sorted, int64_t n_query, int32_t* order, hipStream_t st)
{
    int bits = 0;
    for (int d = 0; d < G.dim; ++d)
        while ((1ll << bits) < G.n[d]) ++bits;
    const int64_t n_curve = bits * G.dim < 31 ? 1ll << (bits * G.dim) : INT64_MAX;
    if (n_curve > 8 * ncell + 1024)
        return hipMemcpyAsync(order, sorted, sizeof(int32_t) * n_query, hipMemcpyDeviceToDevice, st);
    hipError_t e;
    // (qcell is free by now when the queries are the data points, and large enough or grown)
    if ((e = grow((void**)&ws.qcount, ws.cap_qcount, (size_t)(n_curve + 1) * 4)) != hipSuccess) return e;
    if ((e = grow((void**)&ws.qcell, ws.cap_qcell, (size_t)(n_curve + 1) * 4)) != hipSuccess) return e;
    const dim3 grid((unsigned)((n_curve + 1 + 255) / 256));
    hipLaunchKernelGGL(k_curve_count, grid, dim3(256), 0, st, G, n_curve, start, ws.qcount);
    if ((e = scan(ws, ws.qcount, ws.qcell, n_curve + 1, st)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_curve_place, grid, dim3(256), 0, st, G, n_curve, start, ws.qcell, sorted, order);
    return hipGetLastError();
}

template <int DIM>
static hipError_t knn_dim(KnnWorkspace& ws, const double* data, int64_t n_data, const double* query, int64_t n_query,
                          int k, const int64_t* q_ptr, int32_t* out, int32_t* out_order, hipStream_t st)
{
    const bool self = query == data && n_query == n_data;
    const double target = knn_cell_target(DIM, k);
    hipError_t err;
    if ((err = ws.reserve_points(n_data, n_query, DIM, self, st)) != hipSuccess) return err;
    Grid G;
    // One workgroup's binning leaves queries that are not the points in their own order. With a
    // lane per query that costs coherence, in 3-D more than binning them costs: 4,000 points,
    // k = 20: 1M queries 1.37 ms against 0.88 binned, 4M 4.94 and 2.93 (900 points: 1.47 and
    // 1.12; 300: 1.67 and 1.48, but k = 16 1.12 and 1.20; 2-D, 4,000: 0.59 and 0.61).
    const bool binned_queries = DIM == 3 && !self && n_data > 512 && !query_by_wavefront(DIM, k, n_query);
    if (n_data <= kSmallPoints && !out_order && !binned_queries) {
        if ((err = ws.reserve_cells(kSmallCells, true)) != hipSuccess) return err;
        hipLaunchKernelGGL(k_bin_small<DIM>, dim3(1), dim3(kSmallThreads), 0, st, data, (int)n_data, target, (Grid*)ws.grid,
                           ws.start, ws.sidx, ws.sx);
        return launch_query<DIM>(ws, query, self ? ws.sidx : nullptr, n_query, k, q_ptr, out, st);
    }
    // bounding box of the data (queries outside it bin into boundary cells)
    const int nb = (int)std::min<int64_t>((n_data + 2047) / 2048, kBoxBlocks);
    hipLaunchKernelGGL(k_bbox, dim3(nb), dim3(256), 0, st, data, n_data, DIM, ws.bbox,
                       (unsigned int*)(ws.bbox + 6 * kBoxBlocks), ws.hbox);
    if ((err = hipStreamSynchronize(st)) != hipSuccess) return err;
    const double* bb = ws.hbox;
    G.dim = DIM;
    double ext[3] = {0, 0, 0};
    for (int d = 0; d < DIM; ++d) ext[d] = bb[3 + d] - bb[d];
    double s = 1.0;
    const int64_t ncell = knn_grid_size(DIM, ext, n_data, &s, G.n, target);
    G.s = s;
    G.inv_s = 1.0 / s;
    for (int d = 0; d < 3; ++d) G.lo[d] = (d < DIM) ? bb[d] : 0.0;

    if ((err = ws.reserve_cells(ncell, self)) != hipSuccess) return err;
    const int TB = 256;
    const int gridC = (int)std::min<int64_t>((ncell + 1 + TB - 1) / TB, 65535);
    // counting sort of a point set into cells
    auto bin = [&](const double* x, int64_t n, int32_t* cell, int32_t* count, int32_t* start, int32_t* idx,
                   double* sorted_x) -> hipError_t {
        const int gridN = (int)std::min<int64_t>((n + TB - 1) / TB, 65535);
        hipLaunchKernelGGL(k_fill_i32, dim3(gridC), dim3(TB), 0, st, count, ncell + 1, 0);
        hipLaunchKernelGGL(k_cell_count<DIM>, dim3(gridN), dim3(TB), 0, st, x, n, G, cell, count,
                           sorted_x ? (Grid*)ws.grid : nullptr);
        const hipError_t e = scan(ws, count, start, ncell + 1, st);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_scatter<DIM>, dim3(gridN), dim3(TB), 0, st, x, n, cell, start, count, idx, sorted_x);
        return hipGetLastError();
    };
    if ((err = bin(data, n_data, ws.cell, ws.count, ws.start, ws.sidx, ws.sx)) != hipSuccess) return err;
    const int32_t *qstart = ws.start, *qorder = ws.sidx;
    if (!self) {  // (spatially coherent wavefronts)
        if ((err = bin(query, n_query, ws.qcell, ws.qcount, ws.qstart, ws.qorder, nullptr)) != hipSuccess) return err;
        qstart = ws.qstart;
        qorder = ws.qorder;
    }
    if ((err = launch_query<DIM>(ws, query, qorder, n_query, k, q_ptr, out, st)) != hipSuccess) return err;
    if (out_order) return curve_order(ws, G, ncell, qstart, qorder, n_query, out_order, st);
    return hipSuccess;
}

hipError_t KnnWorkspace::reserve_points(int64_t n_data, int64_t n_query, int dim, bool self, hipStream_t st)
{
    hipError_t e;
    if (!bbox) {
        if ((e = hipMalloc((void**)&bbox, sizeof(double) * (6 * kBoxBlocks + 1))) != hipSuccess) return e;
        hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, st, (int32_t*)(bbox + 6 * kBoxBlocks), (int64_t)2, 0);
    }
    if (!hbox && (e = hipHostMalloc((void**)&hbox, sizeof(double) * 6, hipHostMallocDefault)) != hipSuccess) return e;
    if (!grid && (e = hipMalloc(&grid, sizeof(Grid))) != hipSuccess) return e;
    if ((e = grow((void**)&cell, cap_cell, (size_t)n_data * 4)) != hipSuccess) return e;
    if ((e = grow((void**)&sidx, cap_sidx, (size_t)n_data * 4)) != hipSuccess) return e;
    if ((e = grow((void**)&sx, cap_sx, (size_t)n_data * dim * 8)) != hipSuccess) return e;
    if (!self) {
        if ((e = grow((void**)&qcell, cap_qcell, (size_t)n_query * 4)) != hipSuccess) return e;
        if ((e = grow((void**)&qorder, cap_qorder, (size_t)n_query * 4)) != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t KnnWorkspace::reserve_cells(int64_t ncell, bool self)
{
    const size_t nc = (size_t)(ncell + 1) * 4;
    hipError_t e;
    if ((e = grow((void**)&count, cap_count, nc)) != hipSuccess) return e;
    if ((e = grow((void**)&start, cap_start, nc)) != hipSuccess) return e;
    if (!self) {
        if ((e = grow((void**)&qcount, cap_qcount, nc)) != hipSuccess) return e;
        if ((e = grow((void**)&qstart, cap_qstart, nc)) != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t run_knn(KnnWorkspace& ws, const double* data, int64_t n_data, const double* query, int64_t n_query,
                   int dim, int k, const int64_t* q_ptr, int32_t* out, int32_t* out_order, hipStream_t st)
{
    switch (dim) {
    case 1: return knn_dim<1>(ws, data, n_data, query, n_query, k, q_ptr, out, out_order, st);
    case 2: return knn_dim<2>(ws, data, n_data, query, n_query, k, q_ptr, out, out_order, st);
    case 3: return knn_dim<3>(ws, data, n_data, query, n_query, k, q_ptr, out, out_order, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace rbfx
