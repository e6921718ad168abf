// k-nearest-neighbour stencils on the GPU, bit-identical to the host kd-tree (rbfx_knn_kdtree,
// which follows the reference's external/kdtree/KDTree.h search step for step).
//
// Why an exact search suffices: the kd-tree returns its bounded max-heap's contents in
// ascending distance (KDTree.h:407-433), and its pruning keeps every point whose distance is
// below the k-th best. When the k+1 smallest distances of a query are all distinct, the result
// is therefore the unique list of the k nearest points in ascending distance, whatever order
// the tree visits them in. Only when two of those k+1 distances are equal do the heap's sift
// rules and the visit order decide which point comes first (or which of two equidistant
// points at the k-th place is kept). So:
//   * the GPU runs an exact search over a uniform grid of cubic cells, one query per wave;
//   * distances are computed exactly as the kd-tree does, (q0-p0)^2 + (q1-p1)^2 + (q2-p2)^2
//     summed left to right with every product and sum rounded on its own (no fused
//     multiply-add), so equal inputs give equal keys on both sides;
//   * a query whose k+1 best distances are not strictly increasing is handed back and
//     recomputed on the host by the kd-tree (rbfx_knn_kdtree_rows).
//
// The grid is built on the device too: bounding box, the number of occupied cells at halved cell
// sizes, the cell size between two of them at which a ball of its radius holds a little more than
// k+1 nodes, and a counting sort of the nodes by cell.
//
// One cell size does not serve nodes whose density varies by orders of magnitude (a refined cap, a
// graded boundary layer, clusters): a query next to a row of cells that holds far more than its share is
// put aside, the cells with too many nodes are cut into 4 x 4 x 4 of a quarter of the size, those
// again, and the queries put aside are searched through the cut cells (knn_tree_kernel).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "rbfx_ell_common.h"
#include "rbfx_host_internal.h"

namespace {

constexpr int KNN_CAP = 256;        // candidates a wave ranks
constexpr int KNN_MAX_K1 = 170;     // longer lists are left to the host kd-tree
constexpr int KNN_WAVES = 4;        // per workgroup
constexpr int KNN_PER_WAVE = 8;     // queries of a wave, one after the other
constexpr int KNN_LEVELS = 11;      // halvings of the cell size that are counted
constexpr int BOUND_BLOCKS = 256;
constexpr int KNN_DEPTH = 10;       // levels of cut cells at most
constexpr int KNN_FINE = 1 << 26;   // cells along an axis on the finest level
constexpr int REFINE_THREADS = 1024;
constexpr int SCAN_THREADS = 256, SCAN_PER = 16, SCAN_TILE = SCAN_THREADS * SCAN_PER;

struct Point {
    double x, y, z;
    int id, pad;
};

struct Grid {
    double lo[3], h, inv_h;
    int g[3];
    int n_cells;
};

struct Plan {
    Grid grid;
    double lo[3], hi[3];
    int bad;     // a coordinate is not finite
    int n_ties;   // rows handed back
    int n_aside;  // queries put aside for the cut cells
    int n_cut;    // cells cut on the level at hand
    // occupancy levels: grids of halved cells and where their cells' bytes start
    int n_levels;
    Grid level[KNN_LEVELS];
    int cell0[KNN_LEVELS + 1];
    int occupied[KNN_LEVELS];
};

__device__ __forceinline__ int cell_coord(double x, double lo, double inv_h, int g) {
    const int c = (int)((x - lo) * inv_h);  // x >= lo
    return c < 0 ? 0 : (c >= g ? g - 1 : c);
}

__device__ __forceinline__ int cell_index(const Grid& G, double x, double y, double z) {
    return (cell_coord(z, G.lo[2], G.inv_h, G.g[2]) * G.g[1] + cell_coord(y, G.lo[1], G.inv_h, G.g[1])) * G.g[0] +
           cell_coord(x, G.lo[0], G.inv_h, G.g[0]);
}

// Cells of size h over a box; false when they number more than max_cells.
__device__ bool set_cells(Grid& G, const double* lo, const double* hi, double h, int max_cells) {
    double total = 1.0;
    G.h = h;
    G.inv_h = 1.0 / h;
    for (int d = 0; d < 3; d++) {
        G.lo[d] = lo[d];
        const double c = floor((hi[d] - lo[d]) * G.inv_h) + 1.0;
        G.g[d] = c < 1.0 ? 1 : (c > 1e6 ? 1000000 : (int)c);
        total *= G.g[d];
    }
    G.n_cells = total <= (double)max_cells ? (int)total : 0;
    return G.n_cells > 0;
}

// Per block: the box of its nodes, lo and hi, and whether a coordinate is not finite.
__global__ void __launch_bounds__(256) knn_bounds_kernel(const double* __restrict__ xyz, int n, double* __restrict__ part) {
    __shared__ double s[256][7];
    double v[7] = {DBL_MAX, DBL_MAX, DBL_MAX, -DBL_MAX, -DBL_MAX, -DBL_MAX, 0.0};
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < (size_t)n; i += (size_t)gridDim.x * 256)
        for (int d = 0; d < 3; d++) {
            const double c = xyz[3 * i + d];
            v[6] = isfinite(c) ? v[6] : 1.0;
            v[d] = fmin(v[d], c);
            v[3 + d] = fmax(v[3 + d], c);
        }
    for (int q = 0; q < 7; q++) s[threadIdx.x][q] = v[q];
    for (int o = 128; o > 0; o >>= 1) {
        __syncthreads();
        if (threadIdx.x < o)
            for (int q = 0; q < 7; q++) {
                const double a = s[threadIdx.x][q], b = s[threadIdx.x + o][q];
                s[threadIdx.x][q] = q < 3 ? fmin(a, b) : fmax(a, b);
            }
    }
    if (threadIdx.x == 0)
        for (int q = 0; q < 7; q++) part[blockIdx.x * 7 + q] = s[0][q];
}

// The box of all nodes and the levels whose cells are counted: the largest extent cut into 4, 8,
// 16, ... cells, as long as they number at most max_cells.
__global__ void __launch_bounds__(64) knn_levels_kernel(const double* __restrict__ part, int n_part, int max_cells, Plan* P) {
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX}, bad = 0.0;
    for (int b = threadIdx.x; b < n_part; b += 64) {
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], part[b * 7 + d]);
            hi[d] = fmax(hi[d], part[b * 7 + 3 + d]);
        }
        bad = fmax(bad, part[b * 7 + 6]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], __shfl_xor(lo[d], o));
            hi[d] = fmax(hi[d], __shfl_xor(hi[d], o));
        }
        bad = fmax(bad, __shfl_xor(bad, o));
    }
    if (threadIdx.x) return;
    P->bad = bad != 0.0;
    P->n_ties = 0;
    P->n_aside = 0;
    for (int d = 0; d < 3; d++) {
        P->lo[d] = lo[d];
        P->hi[d] = hi[d];
    }
    double ext = fmax(hi[0] - lo[0], fmax(hi[1] - lo[1], hi[2] - lo[2]));
    if (!(ext > 0.0) || !isfinite(ext)) ext = 1.0;
    int l = 0, cell = 0;
    for (; l < KNN_LEVELS; l++) {
        // the bytes of all levels share max_cells
        if (!set_cells(P->level[l], lo, hi, ext * (1.0 + 1e-12) / (double)(4 << l), max_cells - cell - 4)) break;
        P->cell0[l] = cell;
        P->occupied[l] = 0;
        cell += (P->level[l].n_cells + 3) / 4 * 4;
    }
    P->n_levels = l;
    P->cell0[l] = cell;
}

// A byte per cell of every level, set by plain stores: all of them store the same 1. (Bits set by
// atomic or took 7.8 ms for a million nodes in a locality order, whose words many waves share.)
__global__ void __launch_bounds__(256) knn_mark_kernel(const double* __restrict__ xyz, int n, const Plan* __restrict__ P,
                                                      uint8_t* seen) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)n || P->bad) return;
    const double x = xyz[3 * i], y = xyz[3 * i + 1], z = xyz[3 * i + 2];
    for (int l = 0; l < P->n_levels; l++) {
        const int c = P->cell0[l] + cell_index(P->level[l], x, y, z);
        if (!seen[c]) seen[c] = 1;
    }
}

// blockIdx.y: level
__global__ void __launch_bounds__(256) knn_occupied_kernel(Plan* P, const uint8_t* __restrict__ seen) {
    const int l = blockIdx.y;
    if (l >= P->n_levels) return;
    const unsigned* words = reinterpret_cast<const unsigned*>(seen);  // levels start at multiples of 4, bytes past them are 0
    int c = 0;
    for (int w = P->cell0[l] / 4 + blockIdx.x * 256 + threadIdx.x; w < P->cell0[l + 1] / 4; w += gridDim.x * 256) c += __popc(words[w]);
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if (threadIdx.x % 64 == 0 && c) atomicAdd(&P->occupied[l], c);
}

// The cell size at which an occupied cell holds 0.29 (k+1) nodes, between the two levels around
// it: on a surface a ball of that radius then holds about 1.35 (k+1) nodes (a plane meets 1.5 cells
// per cell area on average, so the ball covers 1.5 pi of them), in a volume 1.2 (k+1). Mostly the
// 27 cells around a query then answer it, with one or two candidates per lane.
__global__ void knn_choose_kernel(Plan* P, int n, int k, int max_cells) {
    if (threadIdx.x || blockIdx.x || P->bad) return;
    const double want = fmax(1.5, 0.29 * (k + 1));
    double h = P->n_levels ? P->level[0].h : 1.0, above = 0.0;  // above: nodes per occupied cell one level up
    for (int l = 0; l < P->n_levels; l++) {
        const double per = (double)n / (double)max(1, P->occupied[l]);
        h = P->level[l].h;
        if (per <= want) {
            if (l > 0 && above > per) h *= exp2(log(want / per) / log(above / per));
            break;
        }
        above = per;
    }
    for (int it = 0; it < 64; it++, h *= 1.25)
        if (set_cells(P->grid, P->lo, P->hi, h, max_cells)) return;
    // no such size (the box's extent overflows): one cell, which every search covers at once
    P->grid = Grid{{P->lo[0], P->lo[1], P->lo[2]}, 1.0, 0.0, {1, 1, 1}, 1};
}

__global__ void __launch_bounds__(256) knn_count_kernel(const double* __restrict__ xyz, int n, const Plan* __restrict__ P,
                                                       int* __restrict__ count) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < (size_t)n) atomicAdd(&count[cell_index(P->grid, xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2])], 1);
}

// Exclusive prefix sums: tiles of SCAN_TILE counts, then the tiles' totals (one block), then both.
__global__ void __launch_bounds__(SCAN_THREADS) knn_scan_kernel(const int* __restrict__ count, int n, int* __restrict__ start,
                                                               int* __restrict__ total) {
    __shared__ int s[SCAN_THREADS / 64];
    const int t = threadIdx.x, lane = t % 64;
    const int i0 = blockIdx.x * SCAN_TILE + t * SCAN_PER;
    int v[SCAN_PER], sum = 0;
#pragma unroll
    for (int q = 0; q < SCAN_PER; q++) {
        v[q] = sum;
        sum += i0 + q < n ? count[i0 + q] : 0;
    }
    int in = sum;
    for (int o = 1; o < 64; o <<= 1) {
        const int up = __shfl_up(in, o);
        if (lane >= o) in += up;
    }
    if (lane == 63) s[t / 64] = in;
    __syncthreads();
    int before = in - sum;
    for (int w = 0; w < t / 64; w++) before += s[w];
#pragma unroll
    for (int q = 0; q < SCAN_PER; q++)
        if (i0 + q < n) start[i0 + q] = before + v[q];
    if (t == SCAN_THREADS - 1) total[blockIdx.x] = before + sum;
}

__global__ void __launch_bounds__(1024) knn_scan_totals_kernel(int* __restrict__ total, int n) {
    __shared__ int s[16];
    const int t = threadIdx.x, lane = t % 64;
    int carry = 0;
    for (int i0 = 0; i0 < n; i0 += 1024) {
        const int v = i0 + t < n ? total[i0 + t] : 0;
        int in = v;
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(in, o);
            if (lane >= o) in += up;
        }
        if (lane == 63) s[t / 64] = in;
        __syncthreads();
        int before = carry, all = 0;
        for (int w = 0; w < 16; w++) {
            if (w < t / 64) before += s[w];
            all += s[w];
        }
        if (i0 + t < n) total[i0 + t] = before + in - v;
        carry += all;
        __syncthreads();
    }
}

__global__ void __launch_bounds__(256) knn_scan_add_kernel(int* __restrict__ start, int n, const int* __restrict__ total,
                                                          int n_points) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) start[i] += total[i / SCAN_TILE];
    if (i == n) start[n] = n_points;
}

// Every node into its cell's run; the order inside a cell does not matter to the search.
__global__ void __launch_bounds__(256) knn_scatter_kernel(const double* __restrict__ xyz, int n, const Plan* __restrict__ P,
                                                         const int* __restrict__ start, int* __restrict__ count,
                                                         Point* __restrict__ pts) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)n) return;
    const Point p = {xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], (int)i, 0};
    const int c = cell_index(P->grid, p.x, p.y, p.z);
    pts[start[c] + atomicSub(&count[c], 1) - 1] = p;
}

struct KnnArgs {
    const Point* pts;   // nodes sorted by cell
    const int* start;   // cell c holds pts[start[c]] .. pts[start[c + 1]]
    Plan* plan;
    int32_t* out;       // n x k neighbour ids
    int32_t* ties;      // rows with a distance tie among their k+1 best; from the end, queries put aside
    int n, k, nb;
    int crowd;          // nodes in a row of cells above which a query is put aside
};

// The cut cells. Cut cell b of level l has 64 cells of level l + 1, z slowest, which are runs of its own run of
// nodes: cell s holds pts[start[65 b + s]] .. pts[start[65 b + s + 1]].
struct Tree {
    const double* xyz;
    const int32_t* q;   // the queries
    int n_q;
    const int* child0;  // number of a grid cell's cut, -1 for none; nullptr: no cell is cut
    const int* start;
    const int* child;   // number of cell 64 b + s
};

// Numbers the cells of one level that hold more than `crowd` nodes, as long as there are fewer than max_cut. The cells
// lie in groups of `per`, each with per + 1 starts.
__global__ void __launch_bounds__(256) knn_cut_kernel(const int* __restrict__ start, size_t n_cells, int per, int crowd, int max_cut,
                                                     int* __restrict__ child, int2* __restrict__ range, Plan* P) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n_cells) return;
    const size_t at = i / per * ((size_t)per + 1) + i % per;
    const int p0 = start[at], p1 = start[at + 1];
    int b = -1;
    if (p1 - p0 > crowd) {
        b = atomicAdd(&P->n_cut, 1);
        if (b < max_cut) range[b] = make_int2(p0, p1);
        else b = -1;
    }
    child[i] = b;
}

// Sorts the nodes of cut cells first .. by their 64 cells, a block each (scale: 4^l, l the level of the 64). The
// coordinate on level l is the grid's with its factor scaled by a power of two: the same cell, four times
// as fine on every level.
__global__ void __launch_bounds__(REFINE_THREADS) knn_refine_kernel(Point* pts, Point* tmp, const int2* __restrict__ range,
                                                                   const Plan* __restrict__ P, int scale, int first,
                                                                   int* __restrict__ start) {
    __shared__ int count[64];
    const int t = threadIdx.x, b = first + blockIdx.x;
    const int p0 = range[b].x, p1 = range[b].y;
    const Grid G = P->grid;
    const double inv_h = G.inv_h * scale;
    auto cell = [&](const Point& o) {
        return (cell_coord(o.z, G.lo[2], inv_h, G.g[2] * scale) & 3) * 16 + (cell_coord(o.y, G.lo[1], inv_h, G.g[1] * scale) & 3) * 4 +
               (cell_coord(o.x, G.lo[0], inv_h, G.g[0] * scale) & 3);
    };
    if (t < 64) count[t] = 0;
    __syncthreads();
    for (int p = p0 + t; p < p1; p += REFINE_THREADS) atomicAdd(&count[cell(pts[p])], 1);
    __syncthreads();
    if (t < 64) {
        const int c = count[t];
        int in = c;
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(in, o);
            if (t >= o) in += up;
        }
        count[t] = p0 + in - c;
        start[(size_t)b * 65 + t] = p0 + in - c;
        if (t == 63) start[(size_t)b * 65 + 64] = p1;
    }
    __syncthreads();
    for (int p = p0 + t; p < p1; p += REFINE_THREADS) {
        const Point o = pts[p];
        tmp[atomicAdd(&count[cell(o)], 1)] = o;
    }
    __syncthreads();
    for (int p = p0 + t; p < p1; p += REFINE_THREADS) pts[p] = tmp[p];
}

__device__ __forceinline__ void knn_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wave's candidates for one query.
struct Candidates {
    double D[KNN_CAP];
    int id[KNN_CAP], out[KNN_CAP];
};

// Keeps the nodes of the lanes' runs [p0, p1) that are closer than bound (or all); quarter waves take a run
// each. kept counts all of them, the first KNN_CAP are stored.
__device__ __forceinline__ void knn_take_runs(const Point* __restrict__ pts, const Point& q, int p0, int p1, double bound, bool all,
                                              int lane, Candidates& C, int& kept) {
    unsigned long long runs = __ballot(p1 > p0);
    while (runs) {
        int run[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            run[u] = runs ? __ffsll(runs) - 1 : -1;
            runs &= runs - 1;
        }
        const int u = lane / 16;
        const int mine = u == 0 ? run[0] : u == 1 ? run[1] : u == 2 ? run[2] : run[3];
        int p = __shfl(p0, max(mine, 0));
        const int last = __shfl(p1, max(mine, 0));  // by every lane: a shuffle reads active lanes only
        const int end = mine < 0 ? p : last;
        for (p += lane % 16; __any(p < end); p += 16) {
            double d = 0.0;
            int id = 0;
            bool keep = false;
            if (p < end) {
                const Point o = pts[p];
                const double e0 = q.x - o.x, e1 = q.y - o.y, e2 = q.z - o.z;
                d = dadd_nc(dadd_nc(dmul_nc(e0, e0), dmul_nc(e1, e1)), dmul_nc(e2, e2));
                id = o.id;
                keep = all || d < bound;
            }
            const unsigned long long m = __ballot(keep);
            const int at = kept + __popcll(m & ((1ull << lane) - 1));
            if (keep && at < KNN_CAP) {
                C.D[at] = d;
                C.id[at] = id;
            }
            kept += __popcll(m);
        }
    }
}

// The k best of query q into a.out, or the query to the rows handed back. collect(bound, all) keeps the nodes closer
// than bound (or all) and returns how many there are: n_c of them at `bound` (at least k+1, or all), n_lo < k+1 at lo.
template <typename F>
__device__ __forceinline__ void knn_finish(const KnnArgs& a, const Point& q, int lane, Candidates& C, const F& collect, int n_c,
                                           int n_lo, double lo, double bound, bool all) {
    const int K1 = a.k + 1;
    if (n_c > KNN_CAP) {
        // the number of nodes is about linear in the squared distance on a surface; with all nodes
        // taken, the largest distance in the box bounds it
        double hi = bound;
        if (all) {
            hi = 0.0;
            for (int d = 0; d < 3; d++) hi += (a.plan->hi[d] - a.plan->lo[d]) * (a.plan->hi[d] - a.plan->lo[d]);
            hi *= 1.0 + 1e-9;
        }
        double n_hi = n_c;
        for (int it = 0; it < 100 && (n_c < K1 || n_c > KNN_CAP); it++) {
            double part = (0.5 * (K1 + KNN_CAP) - n_lo) / (n_hi - n_lo);
            part = it % 2 ? 0.5 : fmin(fmax(part, 0.02), 0.98);
            bound = lo + (hi - lo) * part;
            n_c = collect(bound, false);
            if (n_c < K1) {
                lo = bound;
                n_lo = n_c;
            } else {
                hi = bound;
                n_hi = n_c;
            }
        }
    }
    bool tie = n_c < K1 || n_c > KNN_CAP;  // no bound found: many nodes at one distance
    if (tie && n_lo == a.k) {              // it is the (k+1)-th distance: the k below it are the list
        n_c = collect(lo, false);
        tie = n_c != a.k;
    }
    const int i = q.id;
    if (!tie) {
        int place[KNN_CAP / 64];
#pragma unroll
        for (int c = 0; c < KNN_CAP / 64; c++) {
            place[c] = KNN_CAP;
            if (c * 64 < n_c) {
                const int j = c * 64 + lane;
                const double d = j < n_c ? C.D[j] : DBL_MAX;
                int closer = 0;
                for (int m = 0; m < n_c; m++) closer += C.D[m] < d;
                if (j < n_c && closer < a.k) {
                    place[c] = closer;
                    C.out[closer] = j;
                }
            }
        }
        knn_wave_sync();
        // equal distances share a place: all but one of them find another candidate there
#pragma unroll
        for (int c = 0; c < KNN_CAP / 64; c++)
            if (c * 64 < n_c) tie |= place[c] < a.k && C.out[place[c]] != c * 64 + lane;
        tie = __any(tie);
        if (!tie)
            for (int t = lane; t < a.k; t += 64) a.out[(size_t)i * a.k + t] = C.id[C.out[t]];
    }
    if (tie && lane == 0) a.ties[atomicAdd(&a.plan->n_ties, 1)] = i;
}

// One query per wave at a time, queries in cell order. All nodes in the cells within Chebyshev distance r of
// the query's are looked at, and those closer than r * h (with a 1e-9 relative margin for the rounding
// of cell assignment and distances; every other node is farther) are kept in LDS. Fewer than k+1:
// r grows. More than KNN_CAP: the bound is narrowed until between k+1 and KNN_CAP are kept. They hold the
// k+1 best; the place of each is the number of closer ones. The cells of a row along x are one run of
// sorted nodes. A row of more than a.crowd nodes puts the query aside (knn_tree_kernel).
//
// Bound: instruction issue, about 200 candidates and 70 x 70 compared distances a query. N = 10^6, k = 50:
// 1.14 ms; a query per thread with a sorted list of k+1 in LDS (four waves per CU, 130 insertions of
// 25 moves each) took 11.3 ms. The grid kernels take 0.2 ms; binning on the host, with its copies,
// took 27 ms of a call of 41-50 ms, which now takes 2.2 ms.
__global__ void __launch_bounds__(64 * KNN_WAVES) knn_grid_kernel(KnnArgs a) {
    __shared__ Candidates s_c[KNN_WAVES];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    Candidates& C = s_c[wave];
    const Grid G = a.plan->grid;
    const int K1 = a.k + 1, g_max = max(G.g[0], max(G.g[1], G.g[2]));
    const long long q0 = ((long long)xcd_tile(blockIdx.x, a.nb) * KNN_WAVES + wave) * KNN_PER_WAVE;
    for (long long s = q0; s < q0 + KNN_PER_WAVE && s < a.n; s++) {
        const Point q = a.pts[s];
        const int cx = cell_coord(q.x, G.lo[0], G.inv_h, G.g[0]), cy = cell_coord(q.y, G.lo[1], G.inv_h, G.g[1]),
                  cz = cell_coord(q.z, G.lo[2], G.inv_h, G.g[2]);
        int r = 1;
        // keeps the nodes within r cells that are closer than bound (or all); returns how many there are, -1
        // to put the query aside
        auto collect = [&](double bound, bool all) {
            int kept = 0;
            const int x0 = max(cx - r, 0), x1 = min(cx + r, G.g[0] - 1);
            const int y0 = max(cy - r, 0), ny = min(cy + r, G.g[1] - 1) - y0 + 1;
            const int z0 = max(cz - r, 0), nz = min(cz + r, G.g[2] - 1) - z0 + 1;
            for (int c0 = 0; c0 < ny * nz; c0 += 64) {
                const int j = c0 + lane;
                int p0 = 0, p1 = 0;
                if (j < ny * nz) {
                    const int row = ((z0 + j / ny) * G.g[1] + y0 + j % ny) * G.g[0];
                    p0 = a.start[row + x0];
                    p1 = a.start[row + x1 + 1];
                }
                if (__any(p1 - p0 > a.crowd)) return -1;
                knn_take_runs(a.pts, q, p0, p1, bound, all, lane, C, kept);
            }
            knn_wave_sync();
            return kept;
        };
        knn_wave_sync();  // the last query's lists have been read
        int n_c = 0, n_lo = 0;
        double lo = 0.0, bound = 0.0;
        bool all = false;
        for (;;) {
            all = r >= g_max;  // every cell is covered
            bound = (double)r * G.h;
            bound = bound * bound * (1.0 - 1e-9);
            n_c = collect(bound, all);
            if (n_c >= K1 || all || n_c < 0) break;
            lo = bound;
            n_lo = n_c;
            r += max(1, r / 2);
        }
        if (n_c < 0) {
            if (lane == 0) a.ties[a.n - 1 - atomicAdd(&a.plan->n_aside, 1)] = q.id;
            continue;
        }
        knn_finish(a, q, lane, C, collect, n_c, n_lo, lo, bound, all);
    }
}

// The queries put aside, one per wave at a time. The ball around the query that should hold a little more than
// k+1 nodes, by the finest cell it lies in, grows until it does. Rows of grid cells that meet it and hold few nodes
// are runs as above; of the others its cells are looked at one by one, cut cells that meet it a level
// further down, 64 lanes for their 64 cells.
//
// Bound: latency, three dependent loads per level and pass. 300,000 nodes on a sphere, half of them in a cap of 1/50
// of its radius, k = 50: 2.8 ms of a call of 6.9; passes over all nodes of the grid's cells took 525 ms.
__global__ void __launch_bounds__(64 * KNN_WAVES) knn_tree_kernel(KnnArgs a, Tree T) {
    __shared__ Candidates s_c[KNN_WAVES];
    struct Open {  // a cut cell with cells still to go down into
        unsigned long long todo;
        int b, x, y, z;
    };
    __shared__ Open s_open[KNN_WAVES][KNN_DEPTH + 1];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    Candidates& C = s_c[wave];
    Open(&open)[KNN_DEPTH + 1] = s_open[wave];
    const Grid G = a.plan->grid;
    const int K1 = a.k + 1, g_max = max(G.g[0], max(G.g[1], G.g[2]));
    const long long q0 = ((long long)xcd_tile(blockIdx.x, a.nb) * KNN_WAVES + wave) * KNN_PER_WAVE;
    for (long long s = q0; s < q0 + KNN_PER_WAVE && s < T.n_q; s++) {
        Point q;
        q.id = T.q[s];
        q.x = T.xyz[3 * (size_t)q.id];
        q.y = T.xyz[3 * (size_t)q.id + 1];
        q.z = T.xyz[3 * (size_t)q.id + 2];
        // the query in cells of the grid, from the cell's lower end
        const double tx = (q.x - G.lo[0]) * G.inv_h, ty = (q.y - G.lo[1]) * G.inv_h, tz = (q.z - G.lo[2]) * G.inv_h;
        const int cx = cell_coord(q.x, G.lo[0], G.inv_h, G.g[0]), cy = cell_coord(q.y, G.lo[1], G.inv_h, G.g[1]),
                  cz = cell_coord(q.z, G.lo[2], G.inv_h, G.g[2]);
        // distance along an axis to cells c .. c1 of level l (4^l = scale), in these cells; a coordinate of at
        // most 2^26 cells is off by 2^-26 of one, and the last cell takes what lies beyond
        auto apart = [](double t, int c, int c1, int g, int scale) {
            const double u = t * scale;
            return fmax(fmax(c - u, c1 + 1 >= (long long)g * scale ? 0.0 : u - (c1 + 1)) - 1e-6, 0.0);
        };
        auto meets = [&](double dx, double dy, double dz, int scale, double bound) {
            const double h = G.h / scale;
            return !((dx * dx + dy * dy + dz * dz) * (h * h) * (1.0 - 1e-9) >= bound);  // true where it overflows
        };
        auto collect = [&](double bound, bool all) {
            int kept = 0;
            // the cells of cut cell b of level 0 at (x, y, z), and of those below
            auto go_down = [&](int b, int x, int y, int z) {
                unsigned long long todo = 0;
                for (int l = 1, scale = 4;;) {
                    const int ux = 4 * x + lane % 4, uy = 4 * y + lane / 4 % 4, uz = 4 * z + lane / 16;
                    int p0 = T.start[(size_t)b * 65 + lane], p1 = T.start[(size_t)b * 65 + lane + 1], c = -1;
                    const bool near = p1 > p0 && (all || meets(apart(tx, ux, ux, G.g[0], scale), apart(ty, uy, uy, G.g[1], scale),
                                                               apart(tz, uz, uz, G.g[2], scale), scale, bound));
                    if (near) c = T.child[(size_t)b * 64 + lane];
                    todo = __ballot(c >= 0);
                    if (!near || c >= 0) p1 = p0;
                    knn_take_runs(a.pts, q, p0, p1, bound, all, lane, C, kept);
                    while (!todo) {
                        if (l == 1) return;
                        l--;
                        scale /= 4;
                        const Open o = open[l];
                        todo = o.todo;
                        b = o.b;
                        x = o.x;
                        y = o.y;
                        z = o.z;
                    }
                    const int s64 = __ffsll(todo) - 1;
                    todo &= todo - 1;
                    knn_wave_sync();
                    if (lane == 0) open[l] = Open{todo, b, x, y, z};
                    knn_wave_sync();
                    b = T.child[(size_t)b * 64 + s64];
                    x = 4 * x + s64 % 4;
                    y = 4 * y + s64 / 4 % 4;
                    z = 4 * z + s64 / 16;
                    l++;
                    scale *= 4;
                }
            };
            const int r = all ? g_max : (int)fmin(sqrt(bound) * G.inv_h * (1.0 + 1e-9) + 1e-6, (double)g_max) + 1;
            const int x0 = max(cx - r, 0), x1 = min(cx + r, G.g[0] - 1);
            const int y0 = max(cy - r, 0), ny = min(cy + r, G.g[1] - 1) - y0 + 1;
            const int z0 = max(cz - r, 0), nz = min(cz + r, G.g[2] - 1) - z0 + 1;
            for (int c0 = 0; c0 < ny * nz; c0 += 64) {
                const int j = c0 + lane;
                int p0 = 0, p1 = 0, row = 0;
                if (j < ny * nz) {
                    const int y = y0 + j % ny, z = z0 + j / ny;
                    row = (z * G.g[1] + y) * G.g[0];
                    if (all || meets(0.0, apart(ty, y, y, G.g[1], 1), apart(tz, z, z, G.g[2], 1), 1, bound)) {
                        p0 = a.start[row + x0];
                        p1 = a.start[row + x1 + 1];
                    }
                }
                const bool full = T.child0 && p1 - p0 > KNN_CAP;
                unsigned long long rows = __ballot(full);
                knn_take_runs(a.pts, q, p0, full ? p0 : p1, bound, all, lane, C, kept);
                while (rows) {
                    const int j1 = __ffsll(rows) - 1;
                    rows &= rows - 1;
                    const int row1 = __shfl(row, j1), y = y0 + (c0 + j1) % ny, z = z0 + (c0 + j1) / ny;
                    for (int xc = x0; xc <= x1; xc += 64) {
                        const int x = xc + lane;
                        int c = -1;
                        p0 = p1 = 0;
                        if (x <= x1 && (all || meets(apart(tx, x, x, G.g[0], 1), apart(ty, y, y, G.g[1], 1), apart(tz, z, z, G.g[2], 1), 1, bound))) {
                            p0 = a.start[row1 + x];
                            p1 = a.start[row1 + x + 1];
                            c = T.child0[row1 + x];
                        }
                        unsigned long long cut = __ballot(c >= 0);
                        knn_take_runs(a.pts, q, p0, c >= 0 ? p0 : p1, bound, all, lane, C, kept);
                        while (cut) {
                            const int i = __ffsll(cut) - 1;
                            cut &= cut - 1;
                            go_down(__shfl(c, i), xc + i, y, z);
                        }
                    }
                }
            }
            knn_wave_sync();
            return kept;
        };
        knn_wave_sync();  // the last query's lists have been read
        // the finest cell around the query, its size and nodes
        const int c = (cz * G.g[1] + cy) * G.g[0] + cx;
        int held = a.start[c + 1] - a.start[c], scale = 1;
        if (T.child0)
            for (int b = T.child0[c]; b >= 0;) {
                scale *= 4;
                const int s64 = (cell_coord(q.z, G.lo[2], G.inv_h * scale, G.g[2] * scale) & 3) * 16 +
                                (cell_coord(q.y, G.lo[1], G.inv_h * scale, G.g[1] * scale) & 3) * 4 +
                                (cell_coord(q.x, G.lo[0], G.inv_h * scale, G.g[0] * scale) & 3);
                held = T.start[(size_t)b * 65 + s64 + 1] - T.start[(size_t)b * 65 + s64];
                b = T.child[(size_t)b * 64 + s64];
            }
        // as knn_choose_kernel: a ball of the cell's size holds enough where the cell holds 0.29 (k+1)
        double R = G.h / scale * fmin(fmax(sqrt(0.29 * K1 / held), 0.25), 2.0);
        int n_c = 0, n_lo = 0;
        double lo = 0.0, bound = 0.0;
        bool all = false;
        for (;;) {
            all = !(R * G.inv_h < (double)g_max);  // every cell is covered
            bound = R * R;
            n_c = collect(bound, all);
            if (n_c >= K1 || all) break;
            lo = bound;
            n_lo = n_c;
            R *= fmin(fmax(sqrt(1.35 * K1 / max(n_c, 1)), 1.3), 2.0);
        }
        knn_finish(a, q, lane, C, collect, n_c, n_lo, lo, bound, all);
    }
}

// Rows of k entries from the host to their places.
__global__ void __launch_bounds__(256) knn_put_rows_kernel(const int32_t* __restrict__ rows, const int32_t* __restrict__ val, int n,
                                                          int k, int32_t* __restrict__ out) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e < (size_t)n * k) out[(size_t)rows[e / k] * k + e % k] = val[e];
}

struct DevBuf {
    rbfx_ctx* ctx;
    void* p = nullptr;
    ~DevBuf() { rbfx_pool_free(ctx, p); }
};

unsigned blocks_for(size_t n, size_t per) { return (unsigned)((n + per - 1) / per); }

// The cut cells, level by level, and the search of the n_q queries put aside (at the end of a.ties). Without the
// memory for cut cells the queries are searched on the grid, as slow as that is.
int search_aside(rbfx_ctx* ctx, KnnArgs& a, Point* pts, const double* d_xyz, const Grid& G, int n_q) {
    hipStream_t st = ctx->stream;
    const int crowd = std::max(32, 2 * (a.k + 1));
    const size_t n = (size_t)a.n;
    // a level has at most n / (crowd + 1) cut cells, and mostly far fewer; where the room ends, cells stay uncut
    const int max_cut = (int)std::min<size_t>(3 * (n / ((size_t)crowd + 1)) + 256, INT32_MAX / 65);
    int32_t* q = nullptr;
    Point* tmp = nullptr;
    int *child0 = nullptr, *start = nullptr, *child = nullptr;
    int2* range = nullptr;
    bool cuts = G.inv_h > 0.0;
    auto carve = [&](Carver& m) {
        m.take(&q, (size_t)n_q);
        if (!cuts) return;
        m.take(&tmp, n);
        m.take(&child0, (size_t)G.n_cells);
        m.take(&start, (size_t)max_cut * 65);
        m.take(&child, (size_t)max_cut * 64);
        m.take(&range, (size_t)max_cut);
    };
    DevBuf mem{ctx};
    Carver m;
    carve(m);
    hipError_t e = rbfx_pool_alloc(ctx, &mem.p, m.used);
    if (e != hipSuccess && cuts) {
        cuts = false;
        m = Carver();
        carve(m);
        e = rbfx_pool_alloc(ctx, &mem.p, m.used);
    }
    if (e != hipSuccess) return rbfx_fail(ctx, RBFX_E_NOMEM, "knn_gpu: %s", hipGetErrorString(e));
    m = Carver{(unsigned char*)mem.p};
    carve(m);
    RBFX_HIP_CHECK(ctx, hipMemcpyAsync(q, a.ties + a.n - n_q, (size_t)n_q * sizeof(int32_t), hipMemcpyDeviceToDevice, st));
    if (cuts) {
        RBFX_HIP_CHECK(ctx, hipMemsetAsync(&a.plan->n_cut, 0, sizeof(int), st));
        knn_cut_kernel<<<blocks_for((size_t)G.n_cells, 256), 256, 0, st>>>(a.start, (size_t)G.n_cells, G.n_cells, crowd, max_cut, child0,
                                                                          range, a.plan);
        const long long g_max = std::max({G.g[0], G.g[1], G.g[2]});
        int done = 0;  // cut cells whose 64 cells are there
        for (int l = 1;; l++) {
            int n_cut = 0;
            RBFX_LAUNCH_CHECK(ctx, "knn_cut_kernel");
            RBFX_HIP_CHECK(ctx, hipMemcpyAsync(&n_cut, &a.plan->n_cut, sizeof(int), hipMemcpyDeviceToHost, st));
            RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
            n_cut = std::min(n_cut, max_cut);
            const int now = n_cut - done;
            if (now <= 0) break;
            knn_refine_kernel<<<now, REFINE_THREADS, 0, st>>>(pts, tmp, range, a.plan, 1 << 2 * l, done, start);
            RBFX_LAUNCH_CHECK(ctx, "knn_refine_kernel");
            // the next level's cells must not be finer than their coordinates can tell
            const bool last = l >= KNN_DEPTH || g_max << 2 * (l + 1) > KNN_FINE;
            knn_cut_kernel<<<blocks_for((size_t)now * 64, 256), 256, 0, st>>>(start + (size_t)done * 65, (size_t)now * 64, 64,
                                                                             last ? INT32_MAX : crowd, max_cut, child + (size_t)done * 64,
                                                                             range, a.plan);
            done = n_cut;
        }
    }
    const Tree T = {d_xyz, q, n_q, cuts ? child0 : nullptr, start, child};
    a.nb = (int)((blocks_for((size_t)n_q, KNN_WAVES * KNN_PER_WAVE) + 7) / 8 * 8);
    knn_tree_kernel<<<a.nb, 64 * KNN_WAVES, 0, st>>>(a, T);
    RBFX_LAUNCH_CHECK(ctx, "knn_tree_kernel");
    RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
    return RBFX_OK;
}

// The search with its output either in host memory (out_host) or in device memory (d_out).
int knn_gpu_impl(rbfx_ctx* ctx, int32_t n_nodes, const double* xyz, int32_t k, int32_t* out_host, int32_t* d_out,
                 int32_t* n_host_rows) {
    if (n_host_rows) *n_host_rows = 0;
    RBFX_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    // host kd-tree answers for `rows`, written to the output wherever it lives
    auto host_rows = [&](std::vector<int32_t>& rows) -> int {
        if (n_host_rows) *n_host_rows = (int32_t)rows.size();
        if (rows.empty()) return RBFX_OK;
        if (out_host) return rbfx_knn_kdtree_rows(n_nodes, xyz, k, rows.data(), (int32_t)rows.size(), out_host, 0);
        const size_t m = rows.size();
        rows.resize(m * ((size_t)k + 1));  // the rows, then their lists
        int rc = rbfx_knn_kdtree_rows(n_nodes, xyz, k, rows.data(), (int32_t)m, rows.data() + m, 1);
        if (rc != RBFX_OK) return rc;
        DevBuf put{ctx};
        if (rbfx_pool_alloc(ctx, &put.p, rows.size() * sizeof(int32_t)) != hipSuccess)
            return rbfx_fail(ctx, RBFX_E_NOMEM, "knn_gpu: rows from the host");
        RBFX_HIP_CHECK(ctx, hipMemcpyAsync(put.p, rows.data(), rows.size() * sizeof(int32_t), hipMemcpyHostToDevice, st));
        knn_put_rows_kernel<<<blocks_for(m * k, 256), 256, 0, st>>>((int32_t*)put.p, (int32_t*)put.p + m, (int)m, k, d_out);
        RBFX_LAUNCH_CHECK(ctx, "knn_put_rows_kernel");
        RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
        return RBFX_OK;
    };
    if (k + 1 > n_nodes || k + 1 > KNN_MAX_K1) {
        for (size_t i = 0; i < 3 * (size_t)n_nodes; i++)
            if (!std::isfinite(xyz[i])) return rbfx_fail(ctx, RBFX_E_INVALID, "knn_gpu: non-finite coordinate");
        std::vector<int32_t> rows((size_t)n_nodes);
        for (int32_t i = 0; i < n_nodes; i++) rows[(size_t)i] = i;
        return host_rows(rows);
    }
    const size_t n = (size_t)n_nodes;
    const int max_cells = (int)std::min<size_t>((size_t)1 << 24, std::max<size_t>(4096, 16 * n));
    double *d_xyz = nullptr, *part = nullptr;
    Plan* plan = nullptr;
    Point* pts = nullptr;
    uint8_t* seen = nullptr;
    int *count = nullptr, *start = nullptr, *total = nullptr;
    int32_t *ties = nullptr, *out = d_out;
    auto carve = [&](Carver& m) {
        m.take(&d_xyz, 3 * n);
        m.take(&pts, n);
        m.take(&part, BOUND_BLOCKS * 7);
        m.take(&plan, 1);
        m.take(&seen, (size_t)max_cells);
        m.take(&count, (size_t)max_cells);
        m.take(&start, (size_t)max_cells + 1);
        m.take(&total, (size_t)max_cells / SCAN_TILE + 1);
        m.take(&ties, n);
        if (out_host) m.take(&out, n * k);
    };
    Carver m;
    carve(m);
    DevBuf mem{ctx};
    hipError_t e = rbfx_pool_alloc(ctx, &mem.p, m.used);
    if (e != hipSuccess) return rbfx_fail(ctx, RBFX_E_NOMEM, "knn_gpu: %s", hipGetErrorString(e));
    m = Carver{(unsigned char*)mem.p};
    carve(m);
    RBFX_HIP_CHECK(ctx, hipMemcpyAsync(d_xyz, xyz, 3 * n * sizeof(double), hipMemcpyHostToDevice, st));
    RBFX_HIP_CHECK(ctx, hipMemsetAsync(seen, 0, (size_t)max_cells, st));
    const int bound_blocks = (int)std::min<size_t>(BOUND_BLOCKS, (n + 255) / 256);
    knn_bounds_kernel<<<bound_blocks, 256, 0, st>>>(d_xyz, n_nodes, part);
    knn_levels_kernel<<<1, 64, 0, st>>>(part, bound_blocks, max_cells, plan);
    knn_mark_kernel<<<blocks_for(n, 256), 256, 0, st>>>(d_xyz, n_nodes, plan, seen);
    knn_occupied_kernel<<<dim3(32, KNN_LEVELS), 256, 0, st>>>(plan, seen);
    knn_choose_kernel<<<1, 64, 0, st>>>(plan, n_nodes, k, max_cells);
    RBFX_LAUNCH_CHECK(ctx, "knn grid kernels");
    Plan host;
    RBFX_HIP_CHECK(ctx, hipMemcpyAsync(&host, plan, sizeof(Plan), hipMemcpyDeviceToHost, st));
    RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
    if (host.bad) return rbfx_fail(ctx, RBFX_E_INVALID, "knn_gpu: non-finite coordinate");
    const int n_cells = host.grid.n_cells, tiles = (int)blocks_for(n_cells, SCAN_TILE);
    RBFX_HIP_CHECK(ctx, hipMemsetAsync(count, 0, (size_t)n_cells * sizeof(int), st));
    knn_count_kernel<<<blocks_for(n, 256), 256, 0, st>>>(d_xyz, n_nodes, plan, count);
    knn_scan_kernel<<<tiles, SCAN_THREADS, 0, st>>>(count, n_cells, start, total);
    knn_scan_totals_kernel<<<1, 1024, 0, st>>>(total, tiles);
    knn_scan_add_kernel<<<blocks_for((size_t)n_cells + 1, 256), 256, 0, st>>>(start, n_cells, total, n_nodes);
    knn_scatter_kernel<<<blocks_for(n, 256), 256, 0, st>>>(d_xyz, n_nodes, plan, start, count, pts);
    KnnArgs a;
    a.pts = pts;
    a.start = start;
    a.plan = plan;
    a.out = out;
    a.ties = ties;
    a.n = n_nodes;
    a.k = k;
    // A row of three cells holds 0.87 (k+1) nodes or so where the nodes are even. 24 (k+1): a cubic box whose nodes crowd
    // towards its corner, 200,000 nodes, k = 50, took 44.6 ms on the grid alone and 3.7 with the cut cells (towards a
    // face, z^8: 1.93 and 2.01); 12 (k+1) cuts where the grid is still faster (z^8: 3.2 ms), 48 (k+1) too late (half the
    // nodes in a cap of 0.2: 5.4 ms against 2.9).
    a.crowd = 24 * (k + 1);
    a.nb = (int)((blocks_for(n, KNN_WAVES * KNN_PER_WAVE) + 7) / 8 * 8);
    knn_grid_kernel<<<a.nb, 64 * KNN_WAVES, 0, st>>>(a);
    RBFX_LAUNCH_CHECK(ctx, "knn_grid_kernel");
    RBFX_HIP_CHECK(ctx, hipMemcpyAsync(&host, plan, sizeof(Plan), hipMemcpyDeviceToHost, st));
    RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
    if (host.n_aside) {
        const int rc = search_aside(ctx, a, pts, d_xyz, host.grid, host.n_aside);
        if (rc != RBFX_OK) return rc;
        RBFX_HIP_CHECK(ctx, hipMemcpyAsync(&host.n_ties, &plan->n_ties, sizeof(int), hipMemcpyDeviceToHost, st));
    }
    if (out_host)
        RBFX_HIP_CHECK(ctx, hipMemcpyAsync(out_host, out, sizeof(int32_t) * n * k, hipMemcpyDeviceToHost, st));
    if (host.n_aside || out_host) RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
    const int n_ties = host.n_ties;
    std::vector<int32_t> rows((size_t)n_ties);
    if (n_ties) {
        RBFX_HIP_CHECK(ctx, hipMemcpyAsync(rows.data(), ties, (size_t)n_ties * sizeof(int32_t), hipMemcpyDeviceToHost, st));
        RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
    }
    return host_rows(rows);
}

}  // namespace

extern "C" {

// Exact k-nearest-neighbour stencils, bit-identical to rbfx_knn_kdtree (host arrays in and
// out). Replaces the query loop of Grid::generateStencils(ST_KDTREE)
// (grid_interface.cpp:688-725) with a GPU search; rows with distance ties come from the
// kd-tree on the host, and n_host_rows (optional) receives how many rows that was.
int rbfx_knn_gpu(rbfx_ctx* ctx, int32_t n_nodes, const double* xyz, int32_t k, int32_t* out_idx,
                 int32_t* n_host_rows) {
    if (!ctx) return RBFX_E_INVALID;
    if (n_nodes <= 0 || !xyz || !out_idx || k <= 0 || k > n_nodes)
        return rbfx_fail(ctx, RBFX_E_INVALID, "knn_gpu: bad arguments (n_nodes %d, k %d)", n_nodes, k);
    return knn_gpu_impl(ctx, n_nodes, xyz, k, out_idx, nullptr, n_host_rows);
}

// The same lists written to device memory (d_out_idx: n_nodes * k int32 on the context's
// device), so that the weights and operators can be built from them without a round trip
// through host memory. Tie rows are recomputed on the host and uploaded.
int rbfx_knn_gpu_device(rbfx_ctx* ctx, int32_t n_nodes, const double* xyz, int32_t k, int32_t* d_out_idx,
                        int32_t* n_host_rows) {
    if (!ctx) return RBFX_E_INVALID;
    if (n_nodes <= 0 || !xyz || !d_out_idx || k <= 0 || k > n_nodes)
        return rbfx_fail(ctx, RBFX_E_INVALID, "knn_gpu_device: bad arguments (n_nodes %d, k %d)", n_nodes, k);
    return knn_gpu_impl(ctx, n_nodes, xyz, k, nullptr, d_out_idx, n_host_rows);
}

}  // extern "C"
