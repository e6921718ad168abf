// Steady Stokes flow on the sphere on the device: the coupled velocity-pressure operator of
// StokesSteadyPDE (src/pdes/elliptic/stokes_steady_pde.cpp:61-230), the ILU(0) preconditioner
// of its velocity block (src/precond/ilu0.hpp:157-327 with ilu0_tag(0, 3N), as in
// tests/util/viennacl_gmres_poisson/main_stokes.cpp:83) and restarted GMRES with left
// preconditioning (the ViennaCL solve the reference calls), in FP64 or as FP32 inner solves
// inside FP64 refinement.
//
// Vectors use the reference's block layout: u (rows 0..N), v (N..2N), w (2N..3N), p (3N..4N)
// and the four constraint multipliers (4N..4N+3).
//
// Operator. One thread per stencil row gathers u, v, w and p of its neighbours once and forms
// the four block rows from the four operators of an ELL set (LSFC, XSFC, YSFC, ZSFC):
//   row u: -eta L u + D_x p + lambda_u, ..., row p: D_x u + D_y v + D_z w + lambda_p,
// and a reduction forms the constraint rows (the sums of u, v, w, p).
//
// Preconditioner. ilu0_tag(0, 3N) restricts ILU(0) to the velocity block, whose three
// diagonal blocks are the same matrix -eta L (rows of one component couple only to that
// component), with identity rows elsewhere. The factor of -eta L is computed once and applied
// to the three components. The dependencies of the factorization and of both sweeps follow
// the stencil graph; rows are grouped into dependency levels on the host (a row's level is one
// more than the deepest of the rows it reads). The factorization runs a wave per row on the whole
// device, each entry its own signal; each sweep runs the three components on a workgroup each, its
// waves handing the levels on through a counter in LDS. Every row accumulates in the reference's
// order, without fused multiply-adds, so the factor and the sweeps match the CPU restatement bit
// for bit.
//
// GMRES. Arnoldi with classical Gram-Schmidt applied twice (each pass one multi-dot kernel over
// the basis and one multi-axpy), Givens rotations on the host. The stopping test is the
// reference's: the estimate of ||M^-1 (b - A x)|| / ||b|| below tol.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

#include "rbfx_ell_common.h"
#include "rbfx_stokes_order.h"

namespace {

constexpr int FACTOR_WAVES = 4;       // per workgroup
constexpr int FACTOR_BLOCKS = 256;
constexpr int FACTOR_AHEAD = 2;       // lower entries whose values a wave asks for at once
// What a factor entry holds until it is computed: a signalling NaN, which no operation returns.
constexpr unsigned long long FACTOR_UNSET = 0x7ff4a5a5a5a5a5a5ull;
// A sweep's variants hold rows of up to 32, 40, 48, 56 or 64 entries on one side of the diagonal in
// registers: 12 waves of at most 168 VGPRs for the first, 8 of at most 256 for the others. The longest row decides, and the
// first and last rows of a set have n - 1 entries on one side: n = 34 and up run 8 waves. 64 entries in FP64
// do not fit: 64 and 67 VGPRs spill, and N = 20,000 takes 2.87 ms for both sweeps at n = 58 against 1.45 at n = 57
// (4.67 with a barrier per 32 rows).
constexpr int sweep_variant(int blks) { return blks <= 4 ? 4 : blks <= 7 ? blks : 8; }
__host__ __device__ constexpr int sweep_waves(int nb) { return nb <= 4 ? 12 : 8; }
constexpr int SWEEP_RING = 16384;  // solved values kept in LDS: the last 16384 tasks
constexpr int SWEEP_ZERO = SWEEP_RING, SWEEP_ONE = SWEEP_RING + 1;  // LDS places holding 0 and 1
constexpr int FACTOR_MAX_WIDTH = 64;  // one lane per stencil entry in the factorization
constexpr int DOT_THREADS = 256;
constexpr int DOT_BLOCKS = 256;

__device__ __forceinline__ float fadd_nc(float a, float b) {
#pragma clang fp contract(off)
    return a + b;
}
__device__ __forceinline__ float fmul_nc(float a, float b) {
#pragma clang fp contract(off)
    return a * b;
}
__device__ __forceinline__ double add_nc(double a, double b) { return dadd_nc(a, b); }
__device__ __forceinline__ double mul_nc(double a, double b) { return dmul_nc(a, b); }
__device__ __forceinline__ float add_nc(float a, float b) { return fadd_nc(a, b); }
__device__ __forceinline__ float mul_nc(float a, float b) { return fmul_nc(a, b); }

template <typename WT>
__device__ __forceinline__ void load_w4(const WT* p, WT (&w)[4]) {
#pragma unroll
    for (int o = 0; o < 4; o++) w[o] = p[o];
}

// y = A x for the stencil rows (constraint_rows_kernel writes the last four).
template <typename WT, typename T>
__global__ void __launch_bounds__(256) stokes_apply_kernel(const int32_t* __restrict__ idx_t, const WT* __restrict__ w_t,
                                                           const int32_t* __restrict__ order, int N, int width, T eta,
                                                           const T* __restrict__ x, T* __restrict__ y) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const int row = ell_row_at(order, p);
    const size_t base = ell_row_base(p, width);
    const T* xu = x;
    const T* xv = x + N;
    const T* xw = x + 2 * (size_t)N;
    const T* xp = x + 3 * (size_t)N;
    T lu = 0, lv = 0, lw = 0, gx = 0, gy = 0, gz = 0, dv = 0;
    for (int j = 0; j < width; j++) {
        const size_t e = base + (size_t)j * ELL_TILE;
        const int nb = idx_t[e];
        WT w[4];
        load_w4<WT>(w_t + e * 4, w);
        const T a = xu[nb], b = xv[nb], c = xw[nb], q = xp[nb];
        lu += (T)w[0] * a;
        lv += (T)w[0] * b;
        lw += (T)w[0] * c;
        gx += (T)w[1] * q;
        gy += (T)w[2] * q;
        gz += (T)w[3] * q;
        dv += (T)w[1] * a + (T)w[2] * b + (T)w[3] * c;
    }
    const T* lam = x + 4 * (size_t)N;
    y[row] = -eta * lu + gx + lam[0];
    y[N + row] = -eta * lv + gy + lam[1];
    y[2 * (size_t)N + row] = -eta * lw + gz + lam[2];
    y[3 * (size_t)N + row] = dv + lam[3];
}

template <typename T>
__device__ __forceinline__ T block_sum(T v, T* red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    const int wv = threadIdx.x / 64, lane = threadIdx.x % 64;
    if (lane == 0) red[wv] = v;
    __syncthreads();
    T s = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int)(blockDim.x / 64); i++) s += red[i];
    __syncthreads();
    return s;
}

// partial[k * gridDim.x + b] = sum over block b's share of V[k*ldv + i] * w[i] (w == nullptr:
// the plain sum of V[k]); blockIdx.y = k.
template <typename T>
__global__ void __launch_bounds__(DOT_THREADS) mdot_partial_kernel(const T* __restrict__ V, size_t ldv,
                                                                   const T* __restrict__ w, size_t n,
                                                                   double* __restrict__ partial) {
    __shared__ double red[DOT_THREADS / 64];
    const int k = blockIdx.y;
    const T* v = V + (size_t)k * ldv;
    double s = 0.0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        s += w ? (double)v[i] * (double)w[i] : (double)v[i];
    s = block_sum<double>(s, red);
    if (threadIdx.x == 0) partial[(size_t)k * gridDim.x + blockIdx.x] = s;
}

// out[k] (+)= sum_b partial[k * nb + b], in block order; one wave per k.
__global__ void mdot_final_kernel(const double* __restrict__ partial, int nb, int K, double* __restrict__ out,
                                  int accumulate) {
    const int k = blockIdx.x;
    if (k >= K) return;
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += 64) s += partial[(size_t)k * nb + b];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (threadIdx.x == 0) out[k] = accumulate ? out[k] + s : s;
}

// w[i] += sign * sum_k c[k] * V[k*ldv + i]
template <typename T>
__global__ void __launch_bounds__(256) maxpy_kernel(T* __restrict__ w, const T* __restrict__ V, size_t ldv, int K,
                                                    const double* __restrict__ c, double sign, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int k = 0; k < K; k++) s += c[k] * (double)V[(size_t)k * ldv + i];
    w[i] = (T)((double)w[i] + sign * s);
}

// y = a * x + b * y (b == 0: y = a * x); x may be y
template <typename T, typename U>
__global__ void __launch_bounds__(256) axpby_kernel(T* y, const U* x, double a, double b, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    y[i] = (T)(a * (double)x[i] + (b == 0.0 ? 0.0 : b * (double)y[i]));
}

// Writes the constraint rows y[4N + c] from the per-block sums of x's blocks.
template <typename T>
__global__ void constraint_rows_kernel(const double* __restrict__ sums, int N, T* __restrict__ y) {
    if (threadIdx.x < 4) y[4 * (size_t)N + threadIdx.x] = (T)sums[threadIdx.x];
}

// ILU(0) of A_L (N rows of W entries, columns ascending, diagonal at diag[r]), one wave per row, lane
// p holding entry p. For every lower entry q (ascending, column k): t = w_q / U_kk, and every later
// entry whose column row k's upper part holds, if the input is not zero there, subtracts t * U_kj.
// Each entry sees its updates in that order, without fused multiply-adds, as the reference.
//
// Rows are taken from a counter in level order, and a row's values are their own signal: f starts
// at FACTOR_UNSET everywhere, a row's entries are stored as single 8-byte values in device scope, and a
// wave asks for the entries it needs (up to FACTOR_AHEAD rows k at once) until they are set. Where row k's
// columns sit in the row does not depend on values and is found while earlier rows are computed:
// upos[q][p] is the upper entry of row k = column q that updates entry p.
// Every wait ends: a row's entries come from rows of lower levels, which were taken from the counter
// before it and run in waves that are resident; the lowest unfinished row waits for nothing.
//
// Bound: latency, per level one value from another CU and then a division and an update per lower
// entry left. N = 40962, n = 31 (1735 levels): 1.6 ms, 0.9 us per level; one workgroup of 16 waves
// with a barrier per level took 56.7 ms. Asking for 1, 4 and 8 rows at once: 1.6, 2.1 and 2.9 ms;
// 128 and 512 workgroups: 1.8 and 1.7 ms.
__global__ void __launch_bounds__(64 * FACTOR_WAVES) ilu0_factor_kernel(const int32_t* __restrict__ col,
                                                                       const int32_t* __restrict__ diag,
                                                                       const double* __restrict__ a_in,
                                                                       const int32_t* __restrict__ rows, int N, int W,
                                                                       int* counter, double* f) {
    __shared__ int s_col[FACTOR_WAVES][FACTOR_MAX_WIDTH];
    __shared__ uint8_t s_upos[FACTOR_WAVES][FACTOR_MAX_WIDTH][FACTOR_MAX_WIDTH];
    constexpr int NONE = 255;
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    int(&wc)[FACTOR_MAX_WIDTH] = s_col[wave];
    uint8_t(&upos)[FACTOR_MAX_WIDTH][FACTOR_MAX_WIDTH] = s_upos[wave];
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto value = [&](int q) {
        return __hip_atomic_load((unsigned long long*)f + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    for (;;) {
        int t = 0;
        if (lane == 0) t = atomicAdd(counter, 1);
        t = __builtin_amdgcn_readfirstlane(t);
        if (t >= N) return;
        const int r = rows[t];
        const bool in = lane < W;
        const int c = in ? col[r * W + lane] : INT_MAX;
        double w = in ? a_in[r * W + lane] : 0.0;
        const bool nz = w != 0.0;  // entries the input holds: updates allowed
        const int dpos = diag[r] - r * W;
        const int dk = lane < dpos ? diag[c] : 0;  // lane q: place of the diagonal of row k = column q
        wave_sync();                               // the last row's places have been read
        wc[lane] = c;
        for (int q = 0; q < dpos; q++) upos[q][lane] = NONE;
        wave_sync();
        for (int q0 = 0; q0 < dpos; q0 += 8) {
            int j[8];
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const int q = q0 + b < dpos ? q0 + b : q0;
                const int d = __builtin_amdgcn_readlane(dk, q), k = __builtin_amdgcn_readlane(c, q);
                const int at = d + 1 + lane;
                j[b] = at < (k + 1) * W ? col[at] : INT_MAX;
            }
#pragma unroll
            for (int b = 0; b < 8; b++) {
                int lo = 0, hi = W;  // j[b] among the row's ascending columns
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (wc[mid] < j[b]) lo = mid + 1; else hi = mid;
                }
                if (q0 + b < dpos && lo < W && wc[lo] == j[b]) upos[q0 + b][lo] = (uint8_t)lane;
            }
        }
        wave_sync();
        for (int q = 0; q < dpos;) {
            int u[FACTOR_AHEAD];
            unsigned long long x[FACTOR_AHEAD], d[FACTOR_AHEAD];
#pragma unroll
            for (int b = 0; b < FACTOR_AHEAD; b++) {
                const int qq = q + b < dpos ? q + b : q;
                const int at = __builtin_amdgcn_readlane(dk, qq);
                u[b] = nz ? upos[qq][lane] : NONE;
                d[b] = value(at);
                x[b] = u[b] != NONE ? value(at + 1 + u[b]) : 0;
            }
            bool go = true;
            int n = 0;
#pragma unroll
            for (int b = 0; b < FACTOR_AHEAD; b++)
                if (go && q + b < dpos) {
                    go = !__any(d[b] == FACTOR_UNSET || x[b] == FACTOR_UNSET);
                    if (go) {
                        const unsigned long long wb = (unsigned long long)__double_as_longlong(w);
                        const int lo = __builtin_amdgcn_readlane((int)wb, q + b);
                        const int hi = __builtin_amdgcn_readlane((int)(wb >> 32), q + b);
                        const double wq = __longlong_as_double((long long)((unsigned long long)(unsigned)hi << 32 | (unsigned)lo));
                        const double m = wq / __longlong_as_double((long long)d[b]);
                        if (u[b] != NONE) w = dadd_nc(w, -dmul_nc(m, __longlong_as_double((long long)x[b])));
                        if (lane == q + b) w = m;
                        n++;
                    }
                }
            q += n;
            if (n == 0) __builtin_amdgcn_s_sleep(1);
        }
        unsigned long long out = (unsigned long long)__double_as_longlong(w);
        if (out == FACTOR_UNSET) out |= 1ull << 51;  // an input NaN of that value, made quiet
        if (in) __hip_atomic_store((unsigned long long*)f + r * W + lane, out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

__global__ void factor_init_kernel(unsigned long long* f, size_t n, int* counter, int* err) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) f[i] = FACTOR_UNSET;
    if (i == 0) {
        *counter = 0;
        *err = INT_MAX;
    }
}

// One triangular sweep of the factor over one velocity block (blockIdx.x: u, v or w; the three do
// not depend on each other and run on a CU each).
//
// The rows of a level are cut into chunks of at most SWEEP_ROWS, chunks are numbered in level
// order, and the workgroup's waves take them in turn: one row per lane, its entries (columns
// ascending, at most 8 * NB of them) in registers. A row's sum has to run in column order, but its
// products do not depend on each other, and most of its entries were solved long before the level
// above. So while the waves before it still work, a wave forms the products of a block of 8 entries
// as soon as the chunks they come from are done (need[b]), and, forward, where the latest solved
// entries come last, subtracts them. On the critical path of a level stay the count of finished
// chunks seen in LDS, the reads of the last block's values, the rest of the sum and (backward) the
// division. There is no barrier, and a chunk's loads are issued when the wave's chunk before is
// done, 11 (7) chunks ahead.
//
// Solved values stay in LDS for SWEEP_RING tasks (ring; the place of task t is t mod SWEEP_RING):
// an entry's pk_idx is its value's place there, or, when more than SWEEP_RING tasks lie between,
// ~row: those products are formed from memory when the entries arrive, and the entry then
// multiplies the ring's constant 1. Pads are 0 times the ring's constant 0: s - (+0) = s for every s.
//
// Order. Only the wave of chunk *s_done writes to the ring, and then raises the count to its
// successor; a wave that reads count d therefore reads values of tasks before chunk d, and finds
// none overwritten, as pk_idx keeps to the last SWEEP_RING tasks before its own chunk. LDS operations
// of a wave execute in the order they were issued. Values read from memory were stored at least
// SWEEP_RING / SWEEP_ROWS chunks before, by this CU, and a wave has waited for its store by the time
// it works on its next chunk. Every wait ends: the wave of chunk *s_done waits for no one, and all
// waves of the workgroup are resident.
//
// Bound: the latency of that chain, measured in cycles per chunk forward / backward: count seen 155 /
// 139, reads, products and sum 268 / 572 (an FP64 add takes 9.5, a division 81, a read of 8 scattered
// values about 200), value and count written 76. N = 40962, n = 31 (1736 / 1755 chunks): 0.45 / 0.60
// ms. One workgroup for the three components, products handed over through LDS and a barrier per 32
// rows, took 1.83 / 2.01 ms; this kernel with scalar loads of the entries (64 per lane and chunk, the
// CU's load rate) 0.57 / 0.63, with the final block read ahead of the count 0.70 / 0.80, with
// 4-entry blocks 0.96 / 1.12.
template <typename T, bool UPPER, int NB>
__global__ void __launch_bounds__(64 * sweep_waves(NB)) ilu0_sweep_kernel(const SweepChunk* __restrict__ chunks, int n_chunks,
                                                                     const int32_t* __restrict__ rows,
                                                                     const int32_t* __restrict__ pk_idx,
                                                                     const T* __restrict__ pk_val,
                                                                     const T* __restrict__ pk_diag, int N, T* v_all) {
    constexpr int WAVES = sweep_waves(NB), PER16 = 16 / (int)sizeof(T);
    constexpr int YB = !UPPER && NB <= 6 ? 2 : 1;  // blocks of values read at once
    extern __shared__ __align__(16) unsigned char smem[];
    T* ring = reinterpret_cast<T*>(smem);
    int* s_done = reinterpret_cast<int*>(ring + SWEEP_RING + 2);
    T* v = v_all + (size_t)blockIdx.x * N;
    const int lane = threadIdx.x % 64;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    if (threadIdx.x == 0) {
        ring[SWEEP_ZERO] = T(0);
        ring[SWEEP_ONE] = T(1);
        *s_done = 0;
    }
    __syncthreads();
    auto done = [&] {
        const int d = __hip_atomic_load(s_done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        asm volatile("" ::: "memory");  // the ring is read after the count
        return __builtin_amdgcn_readfirstlane(d);
    };
    // the next chunk's description and row are loaded with this chunk's entries
    SweepChunk next_C = chunks[min(wave, n_chunks - 1)];
    int next_r = rows[next_C.t0 + min(lane, next_C.nr - 1)];
    for (int c = wave; c < n_chunks; c += WAVES) {
        const SweepChunk C = next_C;
        const int r = next_r;
        next_C = chunks[min(c + WAVES, n_chunks - 1)];
        const int nblk = C.nblk & 0xff;
        const int l = lane < C.nr ? lane : C.nr - 1;  // lanes past the last row repeat it
        int id[NB * SWEEP_BLK];
        T p[NB * SWEEP_BLK];  // the factor's entries, then their products
#pragma unroll
        for (int b = 0; b < NB; b++)
            if (UPPER ? b < nblk : b >= NB - nblk) {
                const size_t at = (size_t)C.base * SWEEP_BLK + (UPPER ? b : b - (NB - nblk)) * SWEEP_BLK * C.nr;
#pragma unroll
                for (int e = 0; e < SWEEP_BLK; e += 4) {
                    int i4[4];
                    load_pack<int, 4>(pk_idx + at + e * C.nr + 4 * l, i4);
#pragma unroll
                    for (int q = 0; q < 4; q++) id[b * SWEEP_BLK + e + q] = i4[q];
                }
#pragma unroll
                for (int e = 0; e < SWEEP_BLK; e += PER16) {
                    T v16[PER16];
                    load_pack<T, PER16>(pk_val + at + e * C.nr + PER16 * l, v16);
#pragma unroll
                    for (int q = 0; q < PER16; q++) p[b * SWEEP_BLK + e + q] = v16[q];
                }
            }
        T s = v[r];  // written by this task only
        const T dg = UPPER ? pk_diag[C.t0 + l] : T(1);
        next_r = rows[next_C.t0 + min(lane, next_C.nr - 1)];
        if (C.nblk >> 8) {
#pragma unroll
            for (int b = 0; b < NB; b++)
                if (UPPER ? b < nblk : b >= NB - nblk) {
                    T y[SWEEP_BLK];
#pragma unroll
                    for (int e = 0; e < SWEEP_BLK; e++) {
                        const int k = id[b * SWEEP_BLK + e];
                        y[e] = __hip_atomic_load(v + (k < 0 ? ~k : r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
#pragma unroll
                    for (int e = 0; e < SWEEP_BLK; e++) {
                        int& k = id[b * SWEEP_BLK + e];
                        T& x = p[b * SWEEP_BLK + e];
                        x = k < 0 ? mul_nc(x, y[e]) : x;
                        k = k < 0 ? SWEEP_ONE : k;
                    }
                }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the entries, and this wave's last store
        auto gather = [&](int b, T(&y)[SWEEP_BLK]) {
#pragma unroll
            for (int e = 0; e < SWEEP_BLK; e++) y[e] = ring[id[b * SWEEP_BLK + e]];
        };
        auto products = [&](int b, const T(&y)[SWEEP_BLK]) {
#pragma unroll
            for (int e = 0; e < SWEEP_BLK; e++) p[b * SWEEP_BLK + e] = mul_nc(p[b * SWEEP_BLK + e], y[e]);
        };
        auto subtract = [&](int b) {
#pragma unroll
            for (int e = 0; e < SWEEP_BLK; e++) s = add_nc(s, -p[b * SWEEP_BLK + e]);
        };
        T* const place = ring + ((C.t0 + l) & (SWEEP_RING - 1));
        // While earlier chunks work, what they have left of this chunk. Forward: block by block from
        // the first one (first = first block not subtracted), backward: products from the last
        // block to the first (last = blocks still without), the sum has to wait for block 0.
        int first = NB - nblk, last = nblk;
        int d = done();
        for (;;) {
            if constexpr (!UPPER) {
                StaticFor<0, NB>::run([&](auto B) {
                    constexpr int b = decltype(B)::value;
                    if (first == b && d >= C.need[b]) {
                        T y[SWEEP_BLK];
                        gather(b, y);
                        products(b, y);
                        subtract(b);
                        first = b + 1;
                    }
                });
            } else {
                StaticFor<0, NB>::run([&](auto B) {
                    constexpr int b = NB - 1 - decltype(B)::value;
                    if (last == b + 1 && d >= C.need[b]) {
                        T y[SWEEP_BLK];
                        gather(b, y);
                        products(b, y);
                        last = b;
                    }
                });
            }
            if (d >= c - 1) break;
            if (d < c - 2) __builtin_amdgcn_s_sleep(1);
            d = done();
        }
        // next in line: what is left takes one path without branches per number of blocks
        __builtin_amdgcn_s_setprio(3);
        while (d != c) d = done();
        if constexpr (!UPPER) {
            StaticFor<0, NB>::run([&](auto F) {
                constexpr int f = decltype(F)::value;
                if (first == f) {
                    T y[YB][SWEEP_BLK];  // a block's values are read while the one before is subtracted
                    gather(f, y[0]);
                    StaticFor<f, NB>::run([&](auto B) {
                        constexpr int b = decltype(B)::value;
                        if constexpr (b + 1 < NB && YB == 2) gather(b + 1, y[(b + 1 - f) % YB]);
                        products(b, y[(b - f) % YB]);
                        if constexpr (b + 1 < NB && YB == 1) gather(b + 1, y[0]);
                        subtract(b);
                        if constexpr (b + 2 < NB) asm volatile("" ::: "memory");
                    });
                    first = NB;
                }
            });
        } else {
            StaticFor<1, NB + 1>::run([&](auto L) {
                constexpr int f = decltype(L)::value;
                if (last == f) {
                    T y[YB][SWEEP_BLK];
                    gather(0, y[0]);
                    StaticFor<0, f>::run([&](auto B) {
                        constexpr int b = decltype(B)::value;
                        if constexpr (b + 1 < f && YB == 2) gather(b + 1, y[(b + 1) % YB]);
                        products(b, y[b % YB]);
                        if constexpr (b + 1 < f && YB == 1) gather(b + 1, y[0]);
                        if constexpr (b + 2 < f) asm volatile("" ::: "memory");
                    });
                    last = 0;
                }
            });
            StaticFor<0, NB>::run([&](auto B) {
                if (decltype(B)::value < nblk) subtract(decltype(B)::value);
            });
            s = s / dg;
        }
        *place = s;  // lanes past the last row write its value again
        asm volatile("" ::: "memory");  // the values before the count
        __hip_atomic_store(s_done, c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __builtin_amdgcn_s_setprio(0);
        v[r] = s;
    }
}

// A_L = -eta L by rows with each row's columns ascending (the reference's compressed_matrix), and
// the places of the diagonals, one wave per layout position; the stencils come from the operator
// set's layout, L is its first operator. err receives the first position whose stencil holds a
// node twice or misses its centre.
__global__ void __launch_bounds__(256) stokes_rows_kernel(const int32_t* __restrict__ idx_t, const double* __restrict__ w_t,
                                                         const int32_t* __restrict__ order, int N, int W, double eta,
                                                         int32_t* __restrict__ col, double* __restrict__ a,
                                                         int32_t* __restrict__ diag, int* __restrict__ err) {
    const int p = blockIdx.x * 4 + (int)threadIdx.x / 64, lane = threadIdx.x % 64;
    if (p >= N) return;  // uniform over the wave
    const int r = ell_row_at(order, p);
    const size_t e = ell_row_base(p, W) + (size_t)(lane < W ? lane : 0) * ELL_TILE;
    const int c = lane < W ? idx_t[e] : INT_MAX;
    const double v = lane < W ? w_t[e * 4] : 0.0;
    int place = 0;
    bool twice = false;
    for (int q = 0; q < W; q++) {
        const int o = __builtin_amdgcn_readlane(c, q);
        place += o < c;
        twice |= o == c && q != lane;
    }
    const bool bad = __any(lane < W && twice) || !__any(lane < W && c == r);
    if (bad) {
        if (lane == 0) atomicMin(err, p);
        return;
    }
    if (lane < W) {
        col[(size_t)r * W + place] = c;
        a[(size_t)r * W + place] = dmul_nc(-eta, v);
        if (c == r) diag[r] = r * W + place;
    }
}

// Packs one sweep's entries from the factor f, one wave per chunk (t0, nr, base and nblk given):
// where their values lie, the entries in FP64 and (val32 given) FP32, which chunks each block of 8
// waits for, and the rows' diagonals (dg64 given). Forward, pads come first and block b of nblk is
// the sweep's block nb - nblk + b (the last entries are the latest solved); backward, pads come last.
// 16 bytes of a lane lie side by side: 4 places, 2 or 4 values.
__global__ void __launch_bounds__(256) pack_sweep_kernel(SweepChunk* __restrict__ chunks, int n_chunks,
                                                        const int32_t* __restrict__ rows, const int32_t* __restrict__ task,
                                                        const int32_t* __restrict__ chunk_of, const int32_t* __restrict__ col,
                                                        const int32_t* __restrict__ diag, const double* __restrict__ f, int W,
                                                        int nb, int upper, int32_t* __restrict__ idx,
                                                        double* __restrict__ val64, float* __restrict__ val32,
                                                        double* __restrict__ dg64, float* __restrict__ dg32) {
    const int c = blockIdx.x * 4 + (int)threadIdx.x / 64, lane = threadIdx.x % 64;
    if (c >= n_chunks) return;  // uniform over the wave
    const int t0 = chunks[c].t0, nr = chunks[c].nr, nblk = chunks[c].nblk;
    const size_t base = (size_t)chunks[c].base * SWEEP_BLK;
    const bool in = lane < nr;
    const int r = rows[t0 + (in ? lane : 0)], dr = diag[r];
    const int a = upper ? dr + 1 : r * W, b = upper ? (r + 1) * W : dr;
    bool far = false;
    for (int blk = 0; blk < nblk; blk++) {
        int need = 0;
        for (int e = blk * SWEEP_BLK; e < (blk + 1) * SWEEP_BLK; e++) {
            const int q = upper ? a + e : b - (nblk * SWEEP_BLK - e);
            int at = SWEEP_ZERO;
            double v = 0.0;
            if (in && q >= a && q < b) {
                const int k = col[q], tk = task[k];
                v = f[q];
                if (tk >= t0 - SWEEP_RING) {
                    at = tk & (SWEEP_RING - 1);
                    need = max(need, chunk_of[k] + 1);
                } else {
                    at = ~k;
                    far = true;
                }
            }
            if (in) {
                const size_t at4 = base + (size_t)(e / 4 * 4) * nr + 4 * lane + e % 4;
                idx[at4] = at;
                val64[base + (size_t)(e / 2 * 2) * nr + 2 * lane + e % 2] = v;
                if (val32) val32[at4] = (float)v;
            }
        }
        for (int o = 32; o > 0; o >>= 1) need = max(need, __shfl_xor(need, o));
        if (lane == 0) chunks[c].need[(upper ? 0 : nb - nblk) + blk] = need;
    }
    if (__any(far) && lane == 0) chunks[c].nblk = nblk | 256;
    if (dg64 && in) {
        dg64[t0 + lane] = f[dr];
        if (dg32) dg32[t0 + lane] = (float)f[dr];
    }
}

__global__ void to_f32_kernel(const double* __restrict__ in, float* __restrict__ out, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (float)in[i];
}

inline int blocks_for(size_t n, int t) { return (int)((n + t - 1) / t); }

}  // namespace

struct rbfx_stokes {
    rbfx_ctx* ctx = nullptr;
    rbfx_ell* e64 = nullptr;
    rbfx_ell* e32 = nullptr;
    double eta = 1.0;
    int N = 0, width = 0;
    size_t n_tot = 0;
    void* rows_mem = nullptr;   // one allocation: col, diag, a_in, f64, counter, err, low.rows
    void* sweep_mem = nullptr;  // one allocation: the sweeps' arrays
    // A_L = -eta L and its factor, N rows of the stencil width, columns ascending
    int32_t *col = nullptr, *diag = nullptr;
    double *a_in = nullptr, *f64 = nullptr;
    int *counter = nullptr, *err = nullptr;  // the factorization's next row; first bad stencil
    int n_lev_l = 0, n_lev_u = 0;
    // the sweeps: chunks, their tasks' rows, packed entries (places of the values they multiply,
    // values in FP64 and FP32), the backward tasks' diagonals
    struct Side {
        SweepChunk* chunks = nullptr;
        int32_t *rows = nullptr, *task = nullptr, *chunk_of = nullptr, *idx = nullptr;
        double* val64 = nullptr;
        float* val32 = nullptr;
        int n_chunks = 0;
    } low, up;
    int nb = 0;  // the sweeps' variant: blocks of 8 entries a row may take on one side
    double* ud64 = nullptr;
    float* ud32 = nullptr;
    // GMRES workspace
    int ws_m = -1;
    void* V = nullptr;    // (m + 1) * n_tot values of the run's type (FP64 size)
    void* w = nullptr;    // n_tot
    double* r64 = nullptr;  // n_tot: outer residual of the refinement
    double* x32d = nullptr;  // n_tot: FP32 correction, scratch of the refinement
    double* partial = nullptr;  // (m + 1) * DOT_BLOCKS
    double* hbuf = nullptr;     // 2 * (m + 2): CGS coefficients, norm
    double* coef = nullptr;     // m + 1 coefficients for the solution update
};

namespace {

void stokes_free(rbfx_stokes* S) {
    for (void* p : {S->rows_mem, S->sweep_mem, S->V, S->w, (void*)S->r64, (void*)S->x32d, (void*)S->partial,
                    (void*)S->hbuf, (void*)S->coef})
        rbfx_pool_free(S->ctx, p);
}

// The error of the stencil at layout position p, which holds a node twice or misses its centre.
int bad_stencil(rbfx_ctx* ctx, const rbfx_ell* ops, int p) {
    const int W = ops->width;
    int r = p;
    std::vector<int32_t> c(W);
    if (ops->order) RBFX_HIP_CHECK(ctx, hipMemcpy(&r, ops->order + p, sizeof(int32_t), hipMemcpyDeviceToHost));
    for (int j = 0; j < W; j++)
        RBFX_HIP_CHECK(ctx, hipMemcpy(&c[j], ops->idx_t + ell_row_base(p, W) + (size_t)j * ELL_TILE, sizeof(int32_t),
                                      hipMemcpyDeviceToHost));
    std::sort(c.begin(), c.end());
    for (int j = 1; j < W; j++)
        if (c[j] == c[j - 1])
            return rbfx_fail(ctx, RBFX_E_INVALID, "stokes_create: stencil %d holds node %d twice", r, c[j]);
    return rbfx_fail(ctx, RBFX_E_INVALID, "stokes_create: stencil %d does not contain its centre", r);
}

// y = A x (block layout, n_tot values) for the FP64 or FP32 operator set.
template <typename T>
int apply(rbfx_stokes* S, const T* x, T* y) {
    rbfx_ctx* ctx = S->ctx;
    hipStream_t st = ctx->stream;
    rbfx_ell* e = sizeof(T) == 8 ? S->e64 : S->e32;
    const int N = S->N;
    if (sizeof(T) == 8)
        stokes_apply_kernel<double, double><<<blocks_for(N, 256), 256, 0, st>>>(
            e->idx_t, (const double*)e->w_t, e->order, N, S->width, S->eta, (const double*)x, (double*)y);
    else
        stokes_apply_kernel<float, float><<<blocks_for(N, 256), 256, 0, st>>>(
            e->idx_t, (const float*)e->w_t, e->order, N, S->width, (float)S->eta, (const float*)x, (float*)y);
    RBFX_LAUNCH_CHECK(ctx, "stokes_apply_kernel");
    mdot_partial_kernel<T><<<dim3(DOT_BLOCKS, 4), DOT_THREADS, 0, st>>>(x, (size_t)N, nullptr, (size_t)N, S->partial);
    RBFX_LAUNCH_CHECK(ctx, "mdot_partial_kernel");
    mdot_final_kernel<<<4, 64, 0, st>>>(S->partial, DOT_BLOCKS, 4, S->hbuf, 0);
    RBFX_LAUNCH_CHECK(ctx, "mdot_final_kernel");
    constraint_rows_kernel<T><<<1, 64, 0, st>>>(S->hbuf, N, y);
    RBFX_LAUNCH_CHECK(ctx, "constraint_rows_kernel");
    return RBFX_OK;
}

template <typename T, bool UPPER, int NB>
void launch_sweep_nb(const rbfx_stokes* S, const rbfx_stokes::Side& D, const T* pk_val, const T* pk_diag, T* v) {
    const size_t lds = (SWEEP_RING + 2) * sizeof(T) + 16;
    ilu0_sweep_kernel<T, UPPER, NB><<<3, 64 * sweep_waves(NB), lds, S->ctx->stream>>>(D.chunks, D.n_chunks, D.rows, D.idx,
                                                                                     pk_val, pk_diag, S->N, v);
}

template <typename T, bool UPPER>
int launch_sweep(const rbfx_stokes* S, const rbfx_stokes::Side& D, const T* pk_val, const T* pk_diag, T* v) {
    switch (S->nb) {
        case 4: launch_sweep_nb<T, UPPER, 4>(S, D, pk_val, pk_diag, v); break;
        case 5: launch_sweep_nb<T, UPPER, 5>(S, D, pk_val, pk_diag, v); break;
        case 6: launch_sweep_nb<T, UPPER, 6>(S, D, pk_val, pk_diag, v); break;
        case 7: launch_sweep_nb<T, UPPER, 7>(S, D, pk_val, pk_diag, v); break;
        default: launch_sweep_nb<T, UPPER, SWEEP_MAX_BLKS>(S, D, pk_val, pk_diag, v);
    }
    RBFX_LAUNCH_CHECK(S->ctx, "ilu0_sweep_kernel");
    return RBFX_OK;
}

// v = M^-1 v: both sweeps on the three velocity blocks; the other rows are identity rows.
template <typename T>
int precond(rbfx_stokes* S, T* v) {
    const bool d = sizeof(T) == 8;
    const T* lv = d ? (const T*)S->low.val64 : (const T*)S->low.val32;
    const T* uv = d ? (const T*)S->up.val64 : (const T*)S->up.val32;
    const T* ud = d ? (const T*)S->ud64 : (const T*)S->ud32;
    const int rc = launch_sweep<T, false>(S, S->low, lv, nullptr, v);
    return rc ? rc : launch_sweep<T, true>(S, S->up, uv, ud, v);
}

// out[0..K) = V[0..K)^T w (w == nullptr: plain sums), accumulate: out += instead.
template <typename T>
int mdot(rbfx_stokes* S, const T* V, int K, const T* w, double* out, int accumulate) {
    rbfx_ctx* ctx = S->ctx;
    mdot_partial_kernel<T><<<dim3(DOT_BLOCKS, K), DOT_THREADS, 0, ctx->stream>>>(V, S->n_tot, w, S->n_tot, S->partial);
    RBFX_LAUNCH_CHECK(ctx, "mdot_partial_kernel");
    mdot_final_kernel<<<K, 64, 0, ctx->stream>>>(S->partial, DOT_BLOCKS, K, out, accumulate);
    RBFX_LAUNCH_CHECK(ctx, "mdot_final_kernel");
    return RBFX_OK;
}

int workspace(rbfx_stokes* S, int m) {
    if (S->ws_m >= m) return RBFX_OK;
    for (void** p : {&S->V, &S->w, (void**)&S->r64, (void**)&S->x32d, (void**)&S->coef})
        if (*p) {
            rbfx_pool_free(S->ctx, *p);
            *p = nullptr;
        }
    S->ws_m = -1;
    const size_t n = S->n_tot;
    bool ok = rbfx_pool_alloc(S->ctx, &S->V, (size_t)(m + 1) * n * sizeof(double)) == hipSuccess &&
              rbfx_pool_alloc(S->ctx, &S->w, n * sizeof(double)) == hipSuccess &&
              rbfx_pool_alloc(S->ctx, &S->r64, n * sizeof(double)) == hipSuccess &&
              rbfx_pool_alloc(S->ctx, &S->x32d, n * sizeof(double)) == hipSuccess &&
              rbfx_pool_alloc(S->ctx, &S->coef, (size_t)(m + 1) * sizeof(double)) == hipSuccess;
    if (!ok) {
        S->ws_m = -1;
        return rbfx_fail(S->ctx, RBFX_E_NOMEM, "stokes_gmres: workspace for Krylov dimension %d", m);
    }
    rbfx_pool_free(S->ctx, S->partial);
    rbfx_pool_free(S->ctx, S->hbuf);
    S->partial = nullptr;
    S->hbuf = nullptr;
    if (rbfx_pool_alloc(S->ctx, &S->partial, (size_t)(m + 4) * DOT_BLOCKS * sizeof(double)) != hipSuccess ||
        rbfx_pool_alloc(S->ctx, &S->hbuf, (size_t)2 * (m + 2) * sizeof(double)) != hipSuccess) {
        S->ws_m = -1;
        return rbfx_fail(S->ctx, RBFX_E_NOMEM, "stokes_gmres: reduction buffers");
    }
    S->ws_m = m;
    return RBFX_OK;
}

// Restarted GMRES(m) in type T on A x = b with left preconditioning, from the x given
// (zero_x: from x = 0). Cycles as ViennaCL counts them: max_iter / m, one fewer when m
// divides max_iter. The test is ||M^-1 r|| / ||b|| < tol, or with rel_prec
// ||M^-1 r|| / ||M^-1 r_0|| < tol. Returns 0 (converged), 1 (not converged) or a negative code.
template <typename T>
int gmres(rbfx_stokes* S, const T* b, T* x, double tol, int max_iter, int m, bool zero_x, bool rel_prec, int* iters,
          double* err) {
    rbfx_ctx* ctx = S->ctx;
    hipStream_t st = ctx->stream;
    const size_t n = S->n_tot;
    const int nb = blocks_for(n, 256);
    T* V = (T*)S->V;
    T* w = (T*)S->w;
    int rc;
    if (zero_x) RBFX_HIP_CHECK(ctx, hipMemsetAsync(x, 0, n * sizeof(T), st));
    if ((rc = mdot<T>(S, b, 1, b, S->hbuf, 0))) return rc;
    double nb2 = 0.0;
    RBFX_HIP_CHECK(ctx, hipMemcpyAsync(&nb2, S->hbuf, sizeof(double), hipMemcpyDeviceToHost, st));
    RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
    double norm_b = std::sqrt(nb2);
    *err = 0.0;
    if (norm_b == 0.0) {
        RBFX_HIP_CHECK(ctx, hipMemsetAsync(x, 0, n * sizeof(T), st));
        return 0;
    }
    int cycles = max_iter / m;
    if (cycles > 0 && cycles * m == max_iter) cycles -= 1;
    std::vector<double> H((size_t)(m + 1) * m), cs(m), sn(m), g(m + 1), y(m), hv(m + 2);
    for (int cycle = 0; cycle <= cycles; cycle++) {
        // V_0 = M^-1 (b - A x) / beta
        if ((rc = apply<T>(S, x, V))) return rc;
        axpby_kernel<T, T><<<nb, 256, 0, st>>>(V, b, 1.0, -1.0, n);
        RBFX_LAUNCH_CHECK(ctx, "axpby_kernel");
        if ((rc = precond<T>(S, V))) return rc;
        if ((rc = mdot<T>(S, V, 1, V, S->hbuf, 0))) return rc;
        double b2 = 0.0;
        RBFX_HIP_CHECK(ctx, hipMemcpyAsync(&b2, S->hbuf, sizeof(double), hipMemcpyDeviceToHost, st));
        RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
        const double beta = std::sqrt(b2);
        if (rel_prec && cycle == 0) {
            if (beta == 0.0) return 0;
            norm_b = beta;
        }
        *err = beta / norm_b;
        if (!(beta / norm_b >= tol)) return std::isfinite(beta) ? 0 : 1;
        axpby_kernel<T, T><<<nb, 256, 0, st>>>(V, V, 1.0 / beta, 0.0, n);
        RBFX_LAUNCH_CHECK(ctx, "axpby_kernel");
        std::fill(g.begin(), g.end(), 0.0);
        g[0] = beta;
        int k_used = 0;
        bool done = false;
        for (int k = 0; k < m; k++) {
            (*iters)++;
            if ((rc = apply<T>(S, V + (size_t)k * n, w))) return rc;
            if ((rc = precond<T>(S, w))) return rc;
            // classical Gram-Schmidt, twice: h = V^T w; w -= V h
            for (int pass = 0; pass < 2; pass++) {
                if ((rc = mdot<T>(S, V, k + 1, w, S->hbuf + pass * (m + 2), 0))) return rc;
                maxpy_kernel<T><<<nb, 256, 0, st>>>(w, V, n, k + 1, S->hbuf + pass * (m + 2), -1.0, n);
                RBFX_LAUNCH_CHECK(ctx, "maxpy_kernel");
            }
            if ((rc = mdot<T>(S, w, 1, w, S->hbuf + 2 * (m + 2) - 1, 0))) return rc;
            std::vector<double> h2(2 * (m + 2));
            RBFX_HIP_CHECK(ctx, hipMemcpyAsync(h2.data(), S->hbuf, h2.size() * sizeof(double), hipMemcpyDeviceToHost, st));
            RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
            double* hk = &H[(size_t)k * (m + 1)];  // column k of the Hessenberg matrix
            for (int i = 0; i <= k; i++) hk[i] = h2[i] + h2[(m + 2) + i];
            const double hn = std::sqrt(h2[2 * (m + 2) - 1]);
            hk[k + 1] = hn;
            for (int i = 0; i < k; i++) {  // earlier rotations
                const double a = hk[i], c = hk[i + 1];
                hk[i] = cs[i] * a + sn[i] * c;
                hk[i + 1] = -sn[i] * a + cs[i] * c;
            }
            const double den = std::hypot(hk[k], hk[k + 1]);
            cs[k] = den > 0 ? hk[k] / den : 1.0;
            sn[k] = den > 0 ? hk[k + 1] / den : 0.0;
            hk[k] = den;
            hk[k + 1] = 0.0;
            g[k + 1] = -sn[k] * g[k];
            g[k] = cs[k] * g[k];
            k_used = k + 1;
            *err = std::fabs(g[k + 1]) / norm_b;
            if (!(*err >= tol) || hn == 0.0) {
                done = true;
                break;
            }
            axpby_kernel<T, T><<<nb, 256, 0, st>>>(V + (size_t)(k + 1) * n, w, 1.0 / hn, 0.0, n);
            RBFX_LAUNCH_CHECK(ctx, "axpby_kernel");
        }
        // y = R^-1 g, x += V y
        for (int i = k_used - 1; i >= 0; i--) {
            double s = g[i];
            for (int j = i + 1; j < k_used; j++) s -= H[(size_t)j * (m + 1) + i] * y[j];
            y[i] = s / H[(size_t)i * (m + 1) + i];
        }
        RBFX_HIP_CHECK(ctx, hipMemcpyAsync(S->coef, y.data(), k_used * sizeof(double), hipMemcpyHostToDevice, st));
        maxpy_kernel<T><<<nb, 256, 0, st>>>(x, V, n, k_used, S->coef, 1.0, n);
        RBFX_LAUNCH_CHECK(ctx, "maxpy_kernel");
        RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));  // y is a host array
        if (done && std::isfinite(*err)) return 0;
        if (!std::isfinite(*err)) return 1;
    }
    return 1;
}

}  // namespace

extern "C" {

int rbfx_stokes_create(rbfx_ctx* ctx, rbfx_ell* ops64, rbfx_ell* ops32, double eta, rbfx_stokes** out) {
    if (!ctx || !out) return RBFX_E_INVALID;
    *out = nullptr;
    const uint32_t want[4] = {RBFX_LSFC, RBFX_XSFC, RBFX_YSFC, RBFX_ZSFC};
    for (rbfx_ell* e : {ops64, ops32}) {
        if (!e) continue;
        if (e->ctx != ctx || e->n_ops != 4 || e->n_rows != e->n_cols || std::memcmp(e->types, want, sizeof(want)) != 0)
            return rbfx_fail(ctx, RBFX_E_INVALID,
                             "stokes_create: the operator sets must be square with the operators LSFC, XSFC, YSFC, ZSFC");
    }
    if (!ops64 || ops64->storage != RBFX_F64) return rbfx_fail(ctx, RBFX_E_INVALID, "stokes_create: ops64 must store FP64");
    if (ops32 && (ops32->storage != RBFX_F32 || ops32->n_rows != ops64->n_rows || ops32->width != ops64->width))
        return rbfx_fail(ctx, RBFX_E_INVALID, "stokes_create: ops32 must be the same operators in FP32 storage");
    const int N = ops64->n_rows, W = ops64->width;
    if (W > FACTOR_MAX_WIDTH) return rbfx_fail(ctx, RBFX_E_TOO_LARGE, "stokes_create: stencil width %d above %d", W, FACTOR_MAX_WIDTH);
    RBFX_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    rbfx_stokes* S = new rbfx_stokes();
    S->ctx = ctx;
    S->e64 = ops64;
    S->e32 = ops32;
    S->eta = eta;
    S->N = N;
    S->width = W;
    S->n_tot = 4 * (size_t)N + 4;
    auto fail = [&](int code, const char* what, hipError_t err) {
        hipStreamSynchronize(st);
        stokes_free(S);
        delete S;
        return rbfx_fail(ctx, code, "stokes_create: %s: %s", what, hipGetErrorString(err));
    };
    const size_t nnz = (size_t)N * W;
    auto carve_rows = [&](Carver& m) {
        m.take(&S->col, nnz);
        m.take(&S->diag, N);
        m.take(&S->a_in, nnz);
        m.take(&S->f64, nnz);
        m.take(&S->counter, 1);
        m.take(&S->err, 1);
        m.take(&S->low.rows, N);  // the factorization's order too
    };
    Carver rows_mem;
    carve_rows(rows_mem);
    hipError_t e = rbfx_pool_alloc(ctx, &S->rows_mem, rows_mem.used);
    if (e != hipSuccess) return fail(RBFX_E_NOMEM, "matrix and factor", e);
    rows_mem = Carver{(unsigned char*)S->rows_mem};
    carve_rows(rows_mem);
    // A_L by rows on the device; its pattern comes back for the dependency levels
    factor_init_kernel<<<blocks_for(nnz, 256), 256, 0, st>>>((unsigned long long*)S->f64, nnz, S->counter, S->err);
    stokes_rows_kernel<<<blocks_for(N, 4), 256, 0, st>>>(ops64->idx_t, (const double*)ops64->w_t, ops64->order, N, W, eta, S->col,
                                                        S->a_in, S->diag, S->err);
    std::vector<int32_t> col(nnz), dg(N);
    int bad = 0;
    if ((e = hipGetLastError()) != hipSuccess ||
        (e = hipMemcpyAsync(col.data(), S->col, nnz * sizeof(int32_t), hipMemcpyDeviceToHost, st)) != hipSuccess ||
        (e = hipMemcpyAsync(dg.data(), S->diag, N * sizeof(int32_t), hipMemcpyDeviceToHost, st)) != hipSuccess ||
        (e = hipMemcpyAsync(&bad, S->err, sizeof(int), hipMemcpyDeviceToHost, st)) != hipSuccess ||
        (e = hipStreamSynchronize(st)) != hipSuccess)
        return fail(RBFX_E_HIP, "assembly", e);
    if (bad < N) {
        stokes_free(S);
        delete S;
        return bad_stencil(ctx, ops64, bad);
    }
    // dependency levels: the lower sweep and the factorization read rows k < r of row r's
    // pattern, the upper sweep rows k > r (found while the factorization runs)
    std::vector<int32_t> lev(N);
    int n_lev = 0, max_side = 0;
    for (int r = 0; r < N; r++) {
        int m = -1;
        for (int q = r * W; q < dg[r]; q++) m = std::max(m, lev[col[q]]);
        lev[r] = m + 1;
        n_lev = std::max(n_lev, m + 2);
        max_side = std::max({max_side, dg[r] - r * W, (r + 1) * W - dg[r] - 1});
    }
    HostSide low, up;
    order_side(lev, n_lev, [&](int r) { return dg[r] - r * W; }, low);
    auto send = [&](auto* d, const auto& h) {
        if (e == hipSuccess) e = hipMemcpyAsync(d, h.data(), h.size() * sizeof(h[0]), hipMemcpyHostToDevice, st);
    };
    send(S->low.rows, low.rows);
    if (e == hipSuccess) {
        ilu0_factor_kernel<<<FACTOR_BLOCKS, 64 * FACTOR_WAVES, 0, st>>>(S->col, S->diag, S->a_in, S->low.rows, N, W, S->counter,
                                                                       S->f64);
        e = hipGetLastError();
    }
    if (e != hipSuccess) return fail(RBFX_E_HIP, "ILU(0) factorization", e);
    n_lev = 0;
    for (int r = N - 1; r >= 0; r--) {
        int m = -1;
        for (int q = dg[r] + 1; q < (r + 1) * W; q++) m = std::max(m, lev[col[q]]);
        lev[r] = m + 1;
        n_lev = std::max(n_lev, m + 2);
    }
    order_side(lev, n_lev, [&](int r) { return (r + 1) * W - dg[r] - 1; }, up);
    S->nb = sweep_variant((max_side + SWEEP_BLK - 1) / SWEEP_BLK);
    // what rbfx_stokes_info reports: levels in steps of at most 32 rows (16 for wide stencils)
    const int slots = max_side > 32 ? 16 : 32;
    auto steps = [&](const std::vector<int32_t>& off) {
        int n = 0;
        for (size_t l = 0; l + 1 < off.size(); l++) n += (off[l + 1] - off[l] + slots - 1) / slots;
        return n;
    };
    S->n_lev_l = steps(low.off);
    S->n_lev_u = steps(up.off);
    const bool fp32 = ops32 != nullptr;  // the FP32 copy of the factor serves the FP32 inner solves
    auto carve_sweeps = [&](Carver& m) {
        for (auto [D, H] : {std::pair{&S->low, &low}, std::pair{&S->up, &up}}) {
            D->n_chunks = (int)H->chunks.size();
            m.take(&D->chunks, H->chunks.size());
            if (D == &S->up) m.take(&D->rows, N);
            m.take(&D->task, N);
            m.take(&D->chunk_of, N);
            m.take(&D->idx, H->n_ent);
            m.take(&D->val64, H->n_ent);
            if (fp32) m.take(&D->val32, H->n_ent);
        }
        m.take(&S->ud64, N);
        if (fp32) m.take(&S->ud32, N);
    };
    Carver sweep_mem;
    carve_sweeps(sweep_mem);
    if ((e = rbfx_pool_alloc(ctx, &S->sweep_mem, sweep_mem.used)) != hipSuccess) return fail(RBFX_E_NOMEM, "packed factor entries", e);
    sweep_mem = Carver{(unsigned char*)S->sweep_mem};
    carve_sweeps(sweep_mem);
    const int rc = workspace(S, 1);
    if (rc) {
        hipStreamSynchronize(st);
        stokes_free(S);
        delete S;
        return rc;
    }
    for (auto [D, H] : {std::pair{&S->low, &low}, std::pair{&S->up, &up}}) {
        const bool upper = D == &S->up;
        send(D->chunks, H->chunks);
        if (upper) send(D->rows, H->rows);
        send(D->task, H->task);
        send(D->chunk_of, H->chunk_of);
        if (e == hipSuccess) {
            pack_sweep_kernel<<<blocks_for(D->n_chunks, 4), 256, 0, st>>>(D->chunks, D->n_chunks, D->rows, D->task, D->chunk_of,
                                                                         S->col, S->diag, S->f64, W, S->nb, upper, D->idx,
                                                                         D->val64, D->val32, upper ? S->ud64 : nullptr, S->ud32);
            e = hipGetLastError();
        }
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return fail(RBFX_E_HIP, "ILU(0) factorization", e);
    *out = S;
    return RBFX_OK;
}

void rbfx_stokes_destroy(rbfx_stokes* S) {
    if (!S) return;
    hipSetDevice(S->ctx->device);
    hipStreamSynchronize(S->ctx->stream);
    stokes_free(S);
    delete S;
}

int rbfx_stokes_info(const rbfx_stokes* S, int32_t* n_unknowns, int32_t* lower_levels, int32_t* upper_levels) {
    if (!S) return RBFX_E_INVALID;
    if (n_unknowns) *n_unknowns = (int32_t)S->n_tot;
    if (lower_levels) *lower_levels = S->n_lev_l;
    if (upper_levels) *upper_levels = S->n_lev_u;
    return RBFX_OK;
}

int rbfx_stokes_apply(rbfx_stokes* S, const double* d_x, double* d_y) {
    if (!S || !d_x || !d_y) return RBFX_E_INVALID;
    return apply<double>(S, d_x, d_y);
}

int rbfx_stokes_factor(rbfx_stokes* S, double* d_f) {
    if (!S || !d_f) return RBFX_E_INVALID;
    RBFX_HIP_CHECK(S->ctx, hipMemcpyAsync(d_f, S->f64, (size_t)S->N * S->width * sizeof(double), hipMemcpyDeviceToDevice,
                                          S->ctx->stream));
    return RBFX_OK;
}

int rbfx_stokes_precond(rbfx_stokes* S, double* d_v) {
    if (!S || !d_v) return RBFX_E_INVALID;
    return precond<double>(S, d_v);
}

int rbfx_stokes_gmres(rbfx_stokes* S, const double* d_b, double* d_x, double tol, int32_t max_iter, int32_t krylov,
                      int32_t mode, int32_t* iters, double* error) {
    if (!S || !d_b || !d_x || !iters || !error || !(tol > 0) || max_iter <= 0 || krylov <= 0 || krylov > max_iter)
        return RBFX_E_INVALID;
    rbfx_ctx* ctx = S->ctx;
    if (mode != RBFX_F64 && mode != RBFX_F32) return rbfx_fail(ctx, RBFX_E_INVALID, "stokes_gmres: mode %d", mode);
    if (mode == RBFX_F32 && !S->e32)
        return rbfx_fail(ctx, RBFX_E_STATE, "stokes_gmres: FP32 refinement needs the FP32 operator set");
    RBFX_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    int rc = workspace(S, krylov);
    if (rc) return rc;
    *iters = 0;
    *error = 0.0;
    if (mode == RBFX_F64) {
        rc = gmres<double>(S, d_b, d_x, tol, max_iter, krylov, true, false, iters, error);
        return rc < 0 ? rc : RBFX_OK;
    }
    // FP32 inner solves (operator, factor and Krylov basis in FP32) inside FP64 refinement:
    // r = b - A x and the test ||M^-1 r|| / ||b|| < tol in FP64, the correction from one
    // FP32 GMRES(krylov) cycle that reduces its preconditioned residual by 1e-4, x += d.
    hipStream_t st = ctx->stream;
    const size_t n = S->n_tot;
    const int nb = blocks_for(n, 256);
    RBFX_HIP_CHECK(ctx, hipMemsetAsync(d_x, 0, n * sizeof(double), st));
    if ((rc = mdot<double>(S, d_b, 1, d_b, S->hbuf, 0))) return rc;
    double nb2 = 0.0;
    RBFX_HIP_CHECK(ctx, hipMemcpyAsync(&nb2, S->hbuf, sizeof(double), hipMemcpyDeviceToHost, st));
    RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
    const double norm_b = std::sqrt(nb2);
    if (norm_b == 0.0) return RBFX_OK;
    float* r32 = (float*)S->r64;   // the FP32 vectors live in the FP64 buffers' space
    float* d32 = (float*)S->x32d;
    while (true) {
        if ((rc = apply<double>(S, d_x, (double*)S->w))) return rc;
        axpby_kernel<double, double><<<nb, 256, 0, st>>>((double*)S->w, d_b, 1.0, -1.0, n);  // w = b - A x
        RBFX_LAUNCH_CHECK(ctx, "axpby_kernel");
        to_f32_kernel<<<nb, 256, 0, st>>>((const double*)S->w, r32, n);
        RBFX_LAUNCH_CHECK(ctx, "to_f32_kernel");
        if ((rc = precond<double>(S, (double*)S->w))) return rc;
        if ((rc = mdot<double>(S, (double*)S->w, 1, (double*)S->w, S->hbuf, 0))) return rc;
        double p2 = 0.0;
        RBFX_HIP_CHECK(ctx, hipMemcpyAsync(&p2, S->hbuf, sizeof(double), hipMemcpyDeviceToHost, st));
        RBFX_HIP_CHECK(ctx, hipStreamSynchronize(st));
        *error = std::sqrt(p2) / norm_b;
        if (!(*error >= tol) || !std::isfinite(*error) || *iters >= max_iter) return RBFX_OK;
        const int budget = std::min<int>(krylov, max_iter - *iters);
        double inner_err = 0.0;
        const int before = *iters;
        rc = gmres<float>(S, r32, d32, 1e-4, budget, budget, true, true, iters, &inner_err);
        if (rc < 0) return rc;
        if (*iters == before) return RBFX_OK;  // the FP32 residual vanished: nothing left to correct
        axpby_kernel<double, float><<<nb, 256, 0, st>>>(d_x, d32, 1.0, 1.0, n);
        RBFX_LAUNCH_CHECK(ctx, "axpby_kernel");
    }
}

}  // extern "C"
