// ELL operator sets: device layout build, SpMV and fused multi-operator multi-field SpMM.
//
// Replaces the reference's per-DerType padded row-major buffers and one-thread-per-row
// gather-dot (src/rbffd/rbffd_cl.cpp:215-257, 306-463; src/cl_kernels/computeDeriv.cl:7-25)
// and ViennaCL's column-major ELL vec_mul (ell_matrix_source.h:12-40). Differences by
// design: one index array serves all operators, the operators' weights of a (slot,row) are
// adjacent, several fields are gathered per neighbour, and nothing crosses PCIe per call.
#include <algorithm>
#include <cstring>
#include <vector>

#include <type_traits>

#include "rbfx_ell_common.h"
#include "rbfx_ell_local.h"
#include "rbfx_host_internal.h"

namespace {

struct WPtrs {
    const double* p[16];
};

// The device layout from the row-major stencils and weights, FP32 storage rounded on the way.
// A block takes R consecutive rows: it copies them into LDS as they lie in memory (rows are
// contiguous), rounds them there and writes them out slot by slot, R rows of all the operators
// side by side. Straight from memory every lane of a wave would read another row's cache line
// (the reads) and round its row at one memory latency per weight. Slots go through LDS in chunks of
// at most PACK_SLOTS (one chunk up to n = 128), operators in groups of PACK_OPS; R is what keeps
// the block's LDS below 32 KB (five blocks per CU; n = 50, 4 operators: 16 rows).
// Bound: memory (8 bytes read per weight), with one wave of four busy while a block rounds.
// 400,009 rows, n = 50, 4 operators, FP32 with row sums: 0.51 ms (2.2 TB/s); with slots read one by one while
// rounding, and divisions by R, 0.55; one thread per entry and another kernel for the sums 1.02 +
// 2.34 ms. 8 or 32 rows per block: 0.65 and 0.68 ms, 512 threads: 0.61 ms, all operators' loads in
// one loop with stepped instead of divided places: 0.62 ms.
//
// SUM (FP32 storage, row sums preserved): round each weight to nearest, then walk the slots in
// stencil order (centre first, then by distance, which is roughly descending magnitude) and
// move a weight by at most one FP32 ulp toward the remaining difference between the FP64 row
// sum and the exact sum of the FP32 values. Each stored weight stays within 1.5 ulp of its FP64
// value, and the row sum of the stored weights matches the FP64 row sum to about the ulp of the
// smallest weights instead of the ulp of the largest. Derivative rows sum to zero, so the
// rounding no longer adds (sum of the rounding errors) * u[centre] to every derivative: what is
// left scales with the field's variation across the stencil, not with its magnitude.
constexpr int PACK_THREADS = 256, PACK_SLOTS = 128, PACK_OPS = 4;

// The rounded weight of v, r the difference still to be made up.
__device__ __forceinline__ float round_toward_sum(double d, double& r) {
    float v = (float)d;
    if (v != 0.0f && std::isfinite(r)) {
        const float a = std::fabs(v);
        const double ulp = (double)nextafterf(a, INFINITY) - (double)a;
        if (std::isfinite(ulp)) {
            // ulp is a power of two between 2^-149 and 2^104: its inverse is exact, and so is r / ulp
            const double inv = __longlong_as_double((0x7feLL << 52) - __double_as_longlong(ulp));
            const double k = std::fmin(1.0, std::fmax(-1.0, std::rint(r * inv)));
            if (k != 0.0) {
                const float nv = (float)((double)v + k * ulp);
                r -= (double)nv - (double)v;
                v = nv;
            }
        }
    }
    return v;
}

template <typename WT, bool SUM>
__global__ void __launch_bounds__(PACK_THREADS) ell_pack_kernel(const int32_t* __restrict__ idx, WPtrs w, int n_ops,
                                                               int n_rows, int width, int R, int C,
                                                               int32_t* __restrict__ idx_t, WT* __restrict__ w_t) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int S = C | 1;  // row stride in LDS: odd, so that rows start in different banks
    double* sw = reinterpret_cast<double*>(smem);                       // [op][row][slot]
    int32_t* si = reinterpret_cast<int32_t*>(sw + (size_t)PACK_OPS * R * S);  // [row][slot]
    const int t = threadIdx.x, rs = __ffs(R) - 1;  // R is a power of two
    const int r0 = blockIdx.x * R;
    const int nr = max(0, min(R, n_rows - r0));  // rows past the end: index 0, weight 0
    const size_t dst0 = ell_row_base(r0, width);  // R divides ELL_TILE: the rows share a tile
    for (int g = 0; g < n_ops; g += PACK_OPS) {
        const int og = min(PACK_OPS, n_ops - g);
        const int q = t >> rs, rq = t & (R - 1);  // the weights this thread rounds: operator g + q, row rq
        const bool rounds = SUM && q < og && rq < nr;
        double s64 = 0.0, s32 = 0.0, rest = 0.0;
        // SUM needs the row sums before the first weight is rounded: a pass over the chunks for
        // them, and with more than one chunk a second pass that reads the slots again
        const int passes = SUM && width > C ? 2 : 1;
        for (int pass = 0; pass < passes; pass++) {
            const bool store = pass == passes - 1;
            for (int j0 = 0; j0 < width; j0 += C) {
                const int c = min(C, width - j0);
                for (int o = 0; o < og; o++) {
                    const double* src = w.p[g + o] + (size_t)r0 * width + j0;
#pragma unroll 4
                    for (int e = t; e < nr * c; e += PACK_THREADS) {
                        const int r = e / c, j = e - r * c;
                        sw[((size_t)o * R + r) * S + j] = src[(size_t)r * width + j];
                    }
                }
                if (g == 0 && store)
#pragma unroll 4
                    for (int e = t; e < nr * c; e += PACK_THREADS) {
                        const int r = e / c, j = e - r * c;
                        si[r * S + j] = idx[(size_t)(r0 + r) * width + j0 + j];
                    }
                __syncthreads();
                if (rounds) {
                    double* row = sw + ((size_t)q * R + rq) * S;
                    // 8 slots are read from LDS together: one after the other each waits out its latency
                    if (pass == 0) {
                        for (int b = 0; b < c; b += 8) {
                            double v[8];
#pragma unroll
                            for (int u = 0; u < 8; u++) v[u] = row[min(b + u, c - 1)];
#pragma unroll
                            for (int u = 0; u < 8; u++)
                                if (b + u < c) {
                                    s64 += v[u];
                                    s32 += (double)(float)v[u];
                                }
                        }
                        rest = s64 - s32;
                    }
                    if (store)
                        for (int b = 0; b < c; b += 8) {
                            double v[8];
#pragma unroll
                            for (int u = 0; u < 8; u++) v[u] = row[min(b + u, c - 1)];
#pragma unroll
                            for (int u = 0; u < 8; u++)
                                if (b + u < c) row[b + u] = (double)round_toward_sum(v[u], rest);
                        }
                }
                if (SUM) __syncthreads();
                if (store) {
                    // destination order: slot, row, operator
                    for (int e = t; e < c * R; e += PACK_THREADS) {
                        const int r = e & (R - 1), j = e >> rs;
                        const bool in = r < nr;
                        const size_t d = dst0 + (size_t)(j0 + j) * ELL_TILE + r;
                        const double* v = sw + (size_t)r * S + j;
                        const size_t step = (size_t)R * S;  // to the next operator
                        if (n_ops == 4) {
                            const WT p4[4] = {in ? (WT)v[0] : (WT)0, in ? (WT)v[step] : (WT)0, in ? (WT)v[2 * step] : (WT)0,
                                              in ? (WT)v[3 * step] : (WT)0};
                            store_pack<WT, 4>(w_t + d * 4, p4);
                        } else {
                            for (int o = 0; o < og; o++) w_t[d * n_ops + g + o] = in ? (WT)v[o * step] : (WT)0;
                        }
                        if (g == 0) idx_t[d] = in ? si[r * S + j] : 0;
                    }
                }
                __syncthreads();
            }
        }
    }
}

// Rows per block and LDS bytes of the packing kernel for chunks of C slots.
int pack_rows(int C, size_t* lds) {
    const size_t per_row = (size_t)(C | 1) * (PACK_OPS * sizeof(double) + sizeof(int32_t));
    int R = PACK_THREADS / PACK_OPS;  // a thread rounds one (operator, row)
    while (R > 4 && R * per_row > 32 * 1024) R /= 2;
    *lds = R * per_row;
    return R;
}

__global__ void ell_validate_kernel(const int32_t* __restrict__ idx, size_t total, int n_cols, int* __restrict__ bad) {
    size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= total) return;
    int v = idx[tid];
    if (v < 0 || v >= n_cols) atomicAdd(bad, 1);
}

template <typename WT, typename UT, typename AT, int NOPS, int FPT, int UB>
__global__ void __launch_bounds__(256) ell_spmm_kernel(const int32_t* __restrict__ idx_t, const WT* __restrict__ w_t,
                                                       const UT* __restrict__ u, UT* __restrict__ out,
                                                       const int32_t* __restrict__ order, int n_rows, int width, int F,
                                                       int n_tiles, int nb) {
    const int G = F / FPT;
    const int R = blockDim.x / G;
    int tile = xcd_tile(blockIdx.x, nb);
    if (tile >= n_tiles) return;
    int t = threadIdx.x;
    int rl = t / G;
    if (rl >= R) return;
    const int p = tile * R + rl;  // processing position (layout order)
    if (p >= n_rows) return;
    const int row = ell_row_at(order, p);
    int fofs = (t - rl * G) * FPT;
    AT acc[NOPS][FPT];
    ell_gather_dot<WT, UT, AT, NOPS, FPT, UB>(idx_t, w_t, u, p, width, F, fofs, acc);
#pragma unroll
    for (int o = 0; o < NOPS; o++) {
        UT r[FPT];
#pragma unroll
        for (int f = 0; f < FPT; f++) r[f] = (UT)acc[o][f];
        store_pack<UT, FPT>(out + ((size_t)o * n_rows + row) * F + fofs, r);
    }
}

// LDS-staged fused SpMM: one block per tile of the operator set's tile tables
// (rbfx_ell_build_local). The tile's distinct neighbour records are copied into LDS once, then
// every row gathers from there through 16-bit local indices; the summation order is that of
// ell_spmm_kernel, so the outputs are the same bit for bit. MX: FP32 multiply-adds on the
// matrix cores (16 fields on 4 lanes per row). FP32-accumulation instances with 4 fields per
// thread: six waves per SIMD (three 512-thread blocks per CU), as in rk4_stage_lds_kernel.
template <typename WT, typename UT, typename AT, int NOPS, int FPT, int UB, int SG, int PD, bool MX>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu((sizeof(UT) == 4 && sizeof(AT) == 4 && FPT == 4) ? 6 : 1))) ell_spmm_lds_kernel(const int32_t* __restrict__ loc_pos,
                                                           const int32_t* __restrict__ loc_off,
                                                           const int32_t* __restrict__ loc_nodes,
                                                           const uint16_t* __restrict__ loc_idx,
                                                           const WT* __restrict__ w_t, const UT* __restrict__ u,
                                                           UT* __restrict__ out, const int32_t* __restrict__ order,
                                                           int n_rows, int width, int F, int n_tiles, int nb) {
    extern __shared__ __align__(16) unsigned char smem[];
    UT* lds = reinterpret_cast<UT*>(smem);
    const int tile = xcd_tile(blockIdx.x, nb);
    if (tile >= n_tiles) return;  // uniform over the block
    const int k0 = loc_off[tile];
    const int t = threadIdx.x;
    const int rl = t / SG;
    const int p = loc_pos[tile] + rl;
    const bool live = p < loc_pos[tile + 1];
    const int fofs = (t - rl * SG) * FPT;
    AT d[NOPS][FPT];
    if constexpr (MX) {
        // the first index and weight batches are requested before the staging
        LdsMfmaGather<NOPS, UB, PD> g;
        if (live) g.start(loc_idx, (const float*)w_t, p, width, t - rl * SG);
        ell_stage_tile<UT>(u, F, loc_nodes + k0, loc_off[tile + 1] - k0, lds);
        __syncthreads();
        if (!live) return;  // after the only barrier
        g.finish((const float*)lds, fofs, d);
    } else {
        ell_stage_tile<UT>(u, F, loc_nodes + k0, loc_off[tile + 1] - k0, lds);
        __syncthreads();
        if (!live) return;  // after the only barrier
        ell_gather_dot_lds<WT, UT, AT, NOPS, FPT, UB, SG, PD>(loc_idx, w_t, lds, p, width, fofs, t - rl * SG, d);
    }
    const int row = ell_row_at(order, p);
#pragma unroll
    for (int o = 0; o < NOPS; o++) {
        UT r[FPT];
#pragma unroll
        for (int f = 0; f < FPT; f++) r[f] = (UT)d[o][f];
        store_pack<UT, FPT>(out + ((size_t)o * n_rows + row) * F + fofs, r);
    }
}

// One field, four lanes per row (share 6); lane o of a quad writes operator o's derivative.
template <typename WT, typename UT, typename AT, int NOPS>
__global__ void __launch_bounds__(64) ell_spmm_quad_kernel(const int32_t* __restrict__ idx_t, const WT* __restrict__ w_t,
                                                           const UT* __restrict__ u, UT* __restrict__ out,
                                                           const int32_t* __restrict__ order, int n_rows, int width, int nb) {
    const int p = xcd_tile(blockIdx.x, nb) * 16 + (int)threadIdx.x / 4, q = threadIdx.x % 4;
    if (p >= n_rows) return;  // whole quads
    const int row = ell_row_at(order, p);
    const AT d = ell_gather_dot_quad<WT, UT, AT, NOPS>(idx_t, w_t, u, p, width, q);
    if (q < NOPS) out[(size_t)q * n_rows + row] = (UT)d;
}

// Single operator `op` out of an interleaved set of n_ops (one field).
template <typename WT, typename UT, typename AT>
__global__ void __launch_bounds__(256) ell_spmv_strided_kernel(const int32_t* __restrict__ idx_t,
                                                               const WT* __restrict__ w_t, const UT* __restrict__ u,
                                                               UT* __restrict__ out, const int32_t* __restrict__ order,
                                                               int n_rows, int width, int n_ops, int op, int n_tiles,
                                                               int nb) {
    int tile = xcd_tile(blockIdx.x, nb);
    if (tile >= n_tiles) return;
    const int p = tile * blockDim.x + threadIdx.x;
    if (p >= n_rows) return;
    const int row = ell_row_at(order, p);
    AT acc = 0;
    const size_t base = ell_row_base(p, width);
    for (int j = 0; j < width; j++) {
        size_t e = base + (size_t)j * ELL_TILE;
        int nb_ = idx_t[e];
        acc = fma_acc<AT>((AT)w_t[e * n_ops + op], (AT)u[nb_], acc);
    }
    out[row] = (UT)acc;
}

// Row-order validation: every row must appear exactly once. count[] starts zeroed.
__global__ void ell_order_count_kernel(const int32_t* __restrict__ order, int n, int* __restrict__ count,
                                       int* __restrict__ bad) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    int r = order[p];
    if (r < 0 || r >= n) atomicAdd(bad, 1);
    else atomicAdd(&count[r], 1);
}

__global__ void ell_order_check_kernel(const int* __restrict__ count, int n, int* __restrict__ bad) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n && count[r] != 1) atomicAdd(bad, 1);
}

// moved collects the positions whose row is not the position itself (0: the identity order).
__global__ void ell_order_moved_kernel(const int32_t* __restrict__ order, int n, int* __restrict__ moved) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n && order[p] != p) atomicAdd(moved, 1);
}

// old_pos[row] = layout position of row in the current layout.
__global__ void ell_old_pos_kernel(const int32_t* __restrict__ old_order, int n, int32_t* __restrict__ old_pos) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n) old_pos[old_order ? old_order[p] : p] = p;
}

// New layout entry (position p, slot j) = old entry (old_pos[order[p]], j); pad positions keep
// index 0 and weight 0. One thread per destination entry, in destination order.
template <typename WT>
__global__ void ell_reorder_kernel(const int32_t* __restrict__ idx_o, const WT* __restrict__ w_o,
                                   const int32_t* __restrict__ order, const int32_t* __restrict__ old_pos, int n_rows,
                                   int n_pad, int width, int n_ops, int32_t* __restrict__ idx_n, WT* __restrict__ w_n) {
    size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (tid >= (size_t)n_pad * width) return;
    const size_t per_tile = (size_t)width * ELL_TILE;
    const int tile = (int)(tid / per_tile);
    const size_t rem = tid - (size_t)tile * per_tile;
    const int j = (int)(rem / ELL_TILE);
    const int p = tile * ELL_TILE + (int)(rem % ELL_TILE);
    if (p < n_rows) {
        size_t src = ell_row_base(old_pos[order[p]], width) + (size_t)j * ELL_TILE;
        idx_n[tid] = idx_o[src];
        for (int o = 0; o < n_ops; o++) w_n[tid * n_ops + o] = w_o[src * n_ops + o];
    } else {
        idx_n[tid] = 0;
        for (int o = 0; o < n_ops; o++) w_n[tid * n_ops + o] = (WT)0;
    }
}

inline int grid_blocks(int n_tiles) { return (n_tiles + 7) / 8 * 8; }

// LDS-staged SpMM launch (share 4; share 5 with the matrix-core core): the block is the tile.
template <typename WT, typename UT, typename AT, int NOPS>
int launch_spmm_lds(rbfx_ell* e, const EllTune& t, int F, const void* u, void* out) {
    if (e->lt <= 0) return rbfx_fail(e->ctx, RBFX_E_STATE, "spmm: LDS-staged shape without rbfx_ell_build_local");
    const int fpt = t.fpt, ub = t.ub, G = F / fpt;
    const int block = e->lt * G;
    const size_t lds = (size_t)e->k_max * F * sizeof(UT);
    const int n_tiles = e->n_ltiles, nb = grid_blocks(n_tiles);
    hipStream_t s = e->ctx->stream;
    const WT* wt = (const WT*)e->w_t;
#define RBFX_SPMM_LDS(FPT_, UB_, SG_, MX_)                                                                              if (fpt == FPT_ && ub == UB_ && G == SG_) {                                                                              ell_spmm_lds_kernel<WT, UT, AT, NOPS, FPT_, UB_, SG_, 2, MX_><<<nb, block, lds, s>>>(                                    e->loc_pos, e->loc_off, e->loc_nodes, e->loc_idx, wt, (const UT*)u, (UT*)out, e->order, e->n_rows,                  e->width, F, n_tiles, nb);                                                                                       RBFX_LAUNCH_CHECK(e->ctx, "ell_spmm_lds_kernel");                                                                   return RBFX_OK;                                                                                                  }
    if constexpr (NOPS >= 3) {
        if (t.share == 5) {
            if constexpr (std::is_same<WT, float>::value && std::is_same<UT, float>::value && std::is_same<AT, float>::value) {
                RBFX_SPMM_LDS(4, 4, 4, true) RBFX_SPMM_LDS(4, 8, 4, true)
            }
        } else {
            RBFX_SPMM_LDS(4, 8, 4, false) RBFX_SPMM_LDS(4, 4, 4, false) RBFX_SPMM_LDS(8, 8, 2, false)
            RBFX_SPMM_LDS(8, 4, 2, false)
        }
    }
#undef RBFX_SPMM_LDS
    return rbfx_fail(e->ctx, RBFX_E_INVALID, "spmm: no LDS-staged kernel for fields/thread %d, batch %d, group %d, share %d",
                     fpt, ub, G, t.share);
}

template <typename WT, typename UT, typename AT, int NOPS>
int launch_spmm_fpt(rbfx_ell* e, const EllTune& t, int F, const void* u, void* out) {
    if (t.share == 4 || t.share == 5) return launch_spmm_lds<WT, UT, AT, NOPS>(e, t, F, u, out);
    if (t.share == 6) {
        const int nb = grid_blocks((e->n_rows + 15) / 16);
        ell_spmm_quad_kernel<WT, UT, AT, NOPS><<<nb, 64, 0, e->ctx->stream>>>(e->idx_t, (const WT*)e->w_t, (const UT*)u, (UT*)out,
                                                                             e->order, e->n_rows, e->width, nb);
        RBFX_LAUNCH_CHECK(e->ctx, "ell_spmm_quad_kernel");
        return RBFX_OK;
    }
    const int fpt = t.fpt, block = t.block;
    int G = F / fpt;
    int R = block / G;
    if (R <= 0) return rbfx_fail(e->ctx, RBFX_E_INVALID, "spmm: %d fields with %d per thread exceed block %d", F, fpt, block);
    int n_tiles = (e->n_rows + R - 1) / R;
    int nb = grid_blocks(n_tiles);
    const int32_t* it = e->idx_t;
    const WT* wt = (const WT*)e->w_t;
    const UT* uu = (const UT*)u;
    UT* oo = (UT*)out;
    hipStream_t s = e->ctx->stream;
#define RBFX_SPMM_CASE(FPT_, UB_)                                                                                   \
    if (fpt == FPT_ && t.ub == UB_) {                                                                               \
        ell_spmm_kernel<WT, UT, AT, NOPS, FPT_, UB_><<<nb, block, 0, s>>>(it, wt, uu, oo, e->order, e->n_rows,     \
                                                                           e->width, F, n_tiles, nb);               \
        RBFX_LAUNCH_CHECK(e->ctx, "ell_spmm_kernel");                                                              \
        return RBFX_OK;                                                                                             \
    }
    RBFX_SPMM_CASE(1, 4) RBFX_SPMM_CASE(2, 4) RBFX_SPMM_CASE(4, 4) RBFX_SPMM_CASE(8, 4)
    RBFX_SPMM_CASE(1, 8) RBFX_SPMM_CASE(2, 8) RBFX_SPMM_CASE(4, 8) RBFX_SPMM_CASE(8, 8)
    RBFX_SPMM_CASE(1, 16)  // one field per thread (the SpMV): 16 slots per memory round trip
#undef RBFX_SPMM_CASE
    return rbfx_fail(e->ctx, RBFX_E_INVALID, "spmm: unsupported shape (fields/thread %d, batch %d)", fpt, t.ub);
}

template <typename WT, typename UT, typename AT>
int launch_spmm_ops(rbfx_ell* e, const EllTune& t, int F, const void* u, void* out) {
    switch (e->n_ops) {
        case 1: return launch_spmm_fpt<WT, UT, AT, 1>(e, t, F, u, out);
        case 2: return launch_spmm_fpt<WT, UT, AT, 2>(e, t, F, u, out);
        case 3: return launch_spmm_fpt<WT, UT, AT, 3>(e, t, F, u, out);
        case 4: return launch_spmm_fpt<WT, UT, AT, 4>(e, t, F, u, out);
        default: return rbfx_fail(e->ctx, RBFX_E_TOO_LARGE, "spmm: fused application supports 1..4 operators, set has %d", e->n_ops);
    }
}

int check_types(rbfx_ell* e, int field_type, int accum) {
    if (field_type != RBFX_F64 && field_type != RBFX_F32) return rbfx_fail(e->ctx, RBFX_E_INVALID, "bad field type %d", field_type);
    if (accum != RBFX_F64 && accum != RBFX_F32) return rbfx_fail(e->ctx, RBFX_E_INVALID, "bad accumulation type %d", accum);
    if (e->storage == RBFX_F64 && (field_type != RBFX_F64 || accum != RBFX_F64))
        return rbfx_fail(e->ctx, RBFX_E_INVALID, "FP64-stored operators take FP64 fields and FP64 accumulation");
    if (e->storage == RBFX_F32 && field_type == RBFX_F64 && accum == RBFX_F32)
        return rbfx_fail(e->ctx, RBFX_E_INVALID, "FP64 fields with FP32 accumulation is not offered");
    return RBFX_OK;
}

}  // namespace

// Launch shape of the fused kernels: a tuned entry wins, else the rules of default_shape (rbfx_tune.hip).
int rbfx_ell_pick(rbfx_ell* ell, int n_fields, int field_type, int accum, int kind, EllTune* t);

extern "C" {

int rbfx_ell_create(rbfx_ctx* ctx, int32_t n_rows, int32_t n_cols, int32_t width, const int32_t* d_idx, int32_t n_ops,
                    const uint32_t* dertype_bits, const double* const* d_w, int32_t storage, rbfx_ell** out) {
    if (!ctx || !out) return RBFX_E_INVALID;
    *out = nullptr;
    if (n_rows <= 0 || n_cols <= 0 || width <= 0 || !d_idx || n_ops <= 0 || n_ops > 16 || !d_w)
        return rbfx_fail(ctx, RBFX_E_INVALID, "ell_create: bad sizes (rows %d cols %d width %d ops %d)", n_rows, n_cols, width, n_ops);
    if (storage != RBFX_F64 && storage != RBFX_F32 && storage != RBFX_F32_RN)
        return rbfx_fail(ctx, RBFX_E_INVALID, "ell_create: bad storage %d", storage);
    const bool sum_preserving = storage == RBFX_F32;
    if (storage == RBFX_F32_RN) storage = RBFX_F32;
    for (int o = 0; o < n_ops; o++)
        if (!d_w[o]) return rbfx_fail(ctx, RBFX_E_INVALID, "ell_create: weight pointer %d is NULL", o);
    RBFX_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    rbfx_ell* e = new rbfx_ell();
    e->ctx = ctx;
    e->n_rows = n_rows;
    e->n_cols = n_cols;
    e->width = width;
    e->n_ops = n_ops;
    e->storage = storage;
    e->n_pad = (n_rows + ELL_ROW_PAD - 1) / ELL_ROW_PAD * ELL_ROW_PAD;
    for (int o = 0; o < n_ops; o++) e->types[o] = dertype_bits ? dertype_bits[o] : 0u;
    size_t slots = (size_t)e->n_pad * width;
    size_t wbytes = slots * n_ops * (storage == RBFX_F64 ? sizeof(double) : sizeof(float));
    int* d_bad = nullptr;
    hipError_t err;
    if ((err = rbfx_pool_alloc(ctx, &e->idx_t, slots * sizeof(int32_t))) != hipSuccess || (err = rbfx_pool_alloc(ctx, &e->w_t, wbytes)) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &d_bad, sizeof(int))) != hipSuccess) {
        rbfx_pool_free(ctx, e->idx_t);
        rbfx_pool_free(ctx, e->w_t);
        delete e;
        return rbfx_fail(ctx, RBFX_E_NOMEM, "ell_create: allocation failed: %s", hipGetErrorString(err));
    }
    // validate indices before anything gathers through them
    int bad = 0;
    size_t total_in = (size_t)n_rows * width;
    hipMemsetAsync(d_bad, 0, sizeof(int), ctx->stream);
    ell_validate_kernel<<<(unsigned)((total_in + 255) / 256), 256, 0, ctx->stream>>>(d_idx, total_in, n_cols, d_bad);
    hipMemcpyAsync(&bad, d_bad, sizeof(int), hipMemcpyDeviceToHost, ctx->stream);
    err = hipStreamSynchronize(ctx->stream);
    rbfx_pool_free(ctx, d_bad);
    if (err != hipSuccess || bad) {
        int code = err != hipSuccess ? RBFX_E_HIP : RBFX_E_INVALID;
        rbfx_ell_destroy(e);
        if (code == RBFX_E_HIP) return rbfx_fail(ctx, code, "ell_create: validation failed: %s", hipGetErrorString(err));
        return rbfx_fail(ctx, code, "ell_create: %d stencil indices outside [0,%d)", bad, n_cols);
    }
    WPtrs wp;
    std::memset(&wp, 0, sizeof(wp));
    for (int o = 0; o < n_ops; o++) wp.p[o] = d_w[o];
    const int C = std::min(width, PACK_SLOTS);
    size_t lds = 0;
    const int R = pack_rows(C, &lds);
    const unsigned blocks = (unsigned)(e->n_pad / R);
    if (storage == RBFX_F64)
        ell_pack_kernel<double, false><<<blocks, PACK_THREADS, lds, ctx->stream>>>(d_idx, wp, n_ops, n_rows, width, R, C,
                                                                                  e->idx_t, (double*)e->w_t);
    else if (sum_preserving)
        ell_pack_kernel<float, true><<<blocks, PACK_THREADS, lds, ctx->stream>>>(d_idx, wp, n_ops, n_rows, width, R, C,
                                                                                e->idx_t, (float*)e->w_t);
    else
        ell_pack_kernel<float, false><<<blocks, PACK_THREADS, lds, ctx->stream>>>(d_idx, wp, n_ops, n_rows, width, R, C,
                                                                                 e->idx_t, (float*)e->w_t);
    err = hipGetLastError();
    if (err == hipSuccess) err = hipStreamSynchronize(ctx->stream);
    if (err != hipSuccess) {
        rbfx_ell_destroy(e);
        return rbfx_fail(ctx, RBFX_E_HIP, "ell_create: pack failed: %s", hipGetErrorString(err));
    }
    *out = e;
    return RBFX_OK;
}

static void free_local(rbfx_ell* e) {
    rbfx_pool_free(e->ctx, e->loc_pos);
    rbfx_pool_free(e->ctx, e->loc_off);
    rbfx_pool_free(e->ctx, e->loc_nodes);
    rbfx_pool_free(e->ctx, e->loc_idx);
    e->loc_pos = e->loc_off = e->loc_nodes = nullptr;
    e->loc_idx = nullptr;
    e->lt = e->k_max = e->n_ltiles = 0;
}

void rbfx_ell_destroy(rbfx_ell* e) {
    if (!e) return;
    hipSetDevice(e->ctx->device);
    hipStreamSynchronize(e->ctx->stream);
    rbfx_pool_free(e->ctx, e->idx_t);
    rbfx_pool_free(e->ctx, e->w_t);
    rbfx_pool_free(e->ctx, e->order);
    free_local(e);
    delete e;
}

// The tile tables built on the host: stencils too wide, or lists too long, for the device build.
static int local_tables_host(rbfx_ell* e, int tile_rows, int max_nodes, LocalTables* T) {
    rbfx_ctx* ctx = e->ctx;
    const size_t entries = (size_t)e->n_pad * e->width;
    std::vector<int32_t> idx(entries);
    RBFX_HIP_CHECK(ctx, hipMemcpyAsync(idx.data(), e->idx_t, entries * sizeof(int32_t), hipMemcpyDeviceToHost, ctx->stream));
    RBFX_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    std::vector<int32_t> pos, off, nodes;
    std::vector<uint16_t> lidx;
    const int k_max = rbfx_build_local_tables(idx.data(), e->n_rows, e->n_pad, e->width, ELL_TILE, tile_rows, max_nodes,
                                              pos, off, nodes, lidx);
    if (k_max < 0)
        return rbfx_fail(ctx, RBFX_E_TOO_LARGE, "ell_build_local: a tile of %d rows has more than 65535 distinct nodes", tile_rows);
    int32_t *d_pos = nullptr, *d_off = nullptr, *d_nodes = nullptr;
    uint16_t* d_lidx = nullptr;
    hipError_t err;
    auto drop = [&]() {
        rbfx_pool_free(ctx, d_pos);
        rbfx_pool_free(ctx, d_off);
        rbfx_pool_free(ctx, d_nodes);
        rbfx_pool_free(ctx, d_lidx);
    };
    if ((err = rbfx_pool_alloc(ctx, &d_pos, pos.size() * sizeof(int32_t))) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &d_off, off.size() * sizeof(int32_t))) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &d_nodes, std::max<size_t>(1, nodes.size()) * sizeof(int32_t))) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &d_lidx, lidx.size() * sizeof(uint16_t))) != hipSuccess) {
        drop();
        return rbfx_fail(ctx, RBFX_E_NOMEM, "ell_build_local: %s", hipGetErrorString(err));
    }
    hipMemcpyAsync(d_pos, pos.data(), pos.size() * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream);
    hipMemcpyAsync(d_off, off.data(), off.size() * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream);
    hipMemcpyAsync(d_nodes, nodes.data(), nodes.size() * sizeof(int32_t), hipMemcpyHostToDevice, ctx->stream);
    hipMemcpyAsync(d_lidx, lidx.data(), lidx.size() * sizeof(uint16_t), hipMemcpyHostToDevice, ctx->stream);
    if ((err = hipStreamSynchronize(ctx->stream)) != hipSuccess) {
        drop();
        return rbfx_fail(ctx, RBFX_E_HIP, "ell_build_local: %s", hipGetErrorString(err));
    }
    T->pos = d_pos;
    T->off = d_off;
    T->nodes = d_nodes;
    T->idx = d_lidx;
    T->n_tiles = (int)pos.size() - 1;
    T->k_max = k_max;
    return RBFX_OK;
}

int rbfx_ell_build_local(rbfx_ell* e, int32_t tile_rows, int32_t max_nodes) {
    if (!e) return RBFX_E_INVALID;
    rbfx_ctx* ctx = e->ctx;
    if (tile_rows != 32 && tile_rows != 64 && tile_rows != 128)
        return rbfx_fail(ctx, RBFX_E_INVALID, "ell_build_local: tile_rows %d not 32, 64 or 128", tile_rows);
    if (max_nodes < 0 || (max_nodes > 0 && max_nodes < e->width))
        return rbfx_fail(ctx, RBFX_E_INVALID, "ell_build_local: max_nodes %d below the stencil width %d", max_nodes,
                         e->width);
    RBFX_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    int lds_attr = 0;
    if (hipDeviceGetAttribute(&lds_attr, hipDeviceAttributeMaxSharedMemoryPerBlock, ctx->device) != hipSuccess || lds_attr <= 0)
        lds_attr = 64 * 1024;
    LocalTables T;
    int rc = RBFX_OK;
    if (!rbfx_local_tables_device(e, tile_rows, max_nodes, (size_t)lds_attr, &T, &rc))
        rc = local_tables_host(e, tile_rows, max_nodes, &T);
    if (rc) return rc;
    free_local(e);
    e->loc_pos = T.pos;
    e->n_ltiles = T.n_tiles;
    e->loc_off = T.off;
    e->loc_nodes = T.nodes;
    e->loc_idx = T.idx;
    e->lt = tile_rows;
    e->k_max = T.k_max;
    e->lds_limit = lds_attr;
    e->layout_version++;
    return RBFX_OK;
}

int rbfx_ell_local_info(const rbfx_ell* e, int32_t* tile_rows, int32_t* k_max, int32_t* n_tiles) {
    if (!e) return RBFX_E_INVALID;
    if (tile_rows) *tile_rows = e->lt;
    if (k_max) *k_max = e->k_max;
    if (n_tiles) *n_tiles = e->n_ltiles;
    return RBFX_OK;
}

int rbfx_ell_set_row_order(rbfx_ell* e, const int32_t* d_order) {
    if (!e) return RBFX_E_INVALID;
    rbfx_ctx* ctx = e->ctx;
    if (!d_order) return rbfx_fail(ctx, RBFX_E_INVALID, "ell_set_row_order: order is NULL");
    RBFX_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    const int n = e->n_rows;
    const size_t entries = (size_t)e->n_pad * e->width;
    const size_t wsz = e->storage == RBFX_F64 ? sizeof(double) : sizeof(float);
    hipStream_t s = ctx->stream;
    int* d_count = nullptr;
    int32_t *d_old_pos = nullptr, *d_new_order = nullptr, *idx_n = nullptr;
    void* w_n = nullptr;
    hipError_t err;
    auto release = [&]() {
        hipStreamSynchronize(s);
        rbfx_pool_free(ctx, d_count);
        rbfx_pool_free(ctx, d_old_pos);
        rbfx_pool_free(ctx, d_new_order);
        rbfx_pool_free(ctx, idx_n);
        rbfx_pool_free(ctx, w_n);
    };
    if ((err = rbfx_pool_alloc(ctx, &d_count, sizeof(int) * ((size_t)n + 2))) != hipSuccess) {
        release();
        return rbfx_fail(ctx, RBFX_E_NOMEM, "ell_set_row_order: allocation failed: %s", hipGetErrorString(err));
    }
    // validate: a permutation of 0..n-1 (count[n] collects out-of-range entries and repeats;
    // count[n+1] the positions that move, 0 for the identity)
    int flags[2] = {0, 0};
    const unsigned g = (unsigned)((n + 255) / 256);
    hipMemsetAsync(d_count, 0, sizeof(int) * ((size_t)n + 2), s);
    ell_order_count_kernel<<<g, 256, 0, s>>>(d_order, n, d_count, d_count + n);
    ell_order_check_kernel<<<g, 256, 0, s>>>(d_count, n, d_count + n);
    ell_order_moved_kernel<<<g, 256, 0, s>>>(d_order, n, d_count + n + 1);
    hipMemcpyAsync(flags, d_count + n, sizeof(flags), hipMemcpyDeviceToHost, s);
    if ((err = hipStreamSynchronize(s)) != hipSuccess) {
        release();
        return rbfx_fail(ctx, RBFX_E_HIP, "ell_set_row_order: %s", hipGetErrorString(err));
    }
    const int bad = flags[0];
    if (bad) {
        release();
        return rbfx_fail(ctx, RBFX_E_INVALID, "ell_set_row_order: not a permutation of the %d rows", n);
    }
    if (flags[1] == 0 && !e->order) {  // node order, and the layout is in node order: nothing moves
        release();
        free_local(e);
        e->layout_version++;
        return RBFX_OK;
    }
    if ((err = rbfx_pool_alloc(ctx, &d_old_pos, sizeof(int32_t) * (size_t)n)) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &d_new_order, sizeof(int32_t) * (size_t)n)) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &idx_n, sizeof(int32_t) * entries)) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &w_n, wsz * entries * e->n_ops)) != hipSuccess) {
        release();
        return rbfx_fail(ctx, RBFX_E_NOMEM, "ell_set_row_order: allocation failed: %s", hipGetErrorString(err));
    }
    hipMemcpyAsync(d_new_order, d_order, sizeof(int32_t) * (size_t)n, hipMemcpyDeviceToDevice, s);
    ell_old_pos_kernel<<<g, 256, 0, s>>>(e->order, n, d_old_pos);
    const unsigned ge = (unsigned)((entries + 255) / 256);
    if (e->storage == RBFX_F64)
        ell_reorder_kernel<double><<<ge, 256, 0, s>>>(e->idx_t, (const double*)e->w_t, d_new_order, d_old_pos, n, e->n_pad,
                                                      e->width, e->n_ops, idx_n, (double*)w_n);
    else
        ell_reorder_kernel<float><<<ge, 256, 0, s>>>(e->idx_t, (const float*)e->w_t, d_new_order, d_old_pos, n, e->n_pad,
                                                     e->width, e->n_ops, idx_n, (float*)w_n);
    if ((err = hipGetLastError()) != hipSuccess || (err = hipStreamSynchronize(s)) != hipSuccess) {
        release();
        return rbfx_fail(ctx, RBFX_E_HIP, "ell_set_row_order: reorder failed: %s", hipGetErrorString(err));
    }
    rbfx_pool_free(ctx, e->idx_t);
    rbfx_pool_free(ctx, e->w_t);
    rbfx_pool_free(ctx, e->order);
    e->idx_t = idx_n;
    e->w_t = w_n;
    e->order = d_new_order;
    if (flags[1] == 0) {  // the identity: node order, which the kernels take without an order array
        rbfx_pool_free(ctx, e->order);
        e->order = nullptr;
    }
    free_local(e);  // the local tables describe the previous layout
    e->layout_version++;
    idx_n = nullptr;
    w_n = nullptr;
    d_new_order = nullptr;
    release();
    return RBFX_OK;
}

int rbfx_ell_info(const rbfx_ell* e, int32_t* n_rows, int32_t* width, int32_t* n_ops, int32_t* storage) {
    if (!e) return RBFX_E_INVALID;
    if (n_rows) *n_rows = e->n_rows;
    if (width) *width = e->width;
    if (n_ops) *n_ops = e->n_ops;
    if (storage) *storage = e->storage;
    return RBFX_OK;
}

int rbfx_spmm(rbfx_ell* e, int32_t n_fields, const void* d_u, void* d_out, int32_t field_type, int32_t accum) {
    if (!e) return RBFX_E_INVALID;
    if (n_fields <= 0 || !d_u || !d_out) return rbfx_fail(e->ctx, RBFX_E_INVALID, "spmm: bad arguments");
    int rc = check_types(e, field_type, accum);
    if (rc) return rc;
    EllTune t;
    rc = rbfx_ell_pick(e, n_fields, field_type, accum, 0, &t);
    if (rc) return rc;
    if (e->storage == RBFX_F64) return launch_spmm_ops<double, double, double>(e, t, n_fields, d_u, d_out);
    if (field_type == RBFX_F32 && accum == RBFX_F64) return launch_spmm_ops<float, float, double>(e, t, n_fields, d_u, d_out);
    if (field_type == RBFX_F32) return launch_spmm_ops<float, float, float>(e, t, n_fields, d_u, d_out);
    return launch_spmm_ops<float, double, double>(e, t, n_fields, d_u, d_out);
}

int rbfx_spmv(rbfx_ell* e, int32_t op, const void* d_u, void* d_out, int32_t field_type, int32_t accum) {
    if (!e) return RBFX_E_INVALID;
    if (op < 0 || op >= e->n_ops || !d_u || !d_out) return rbfx_fail(e->ctx, RBFX_E_INVALID, "spmv: bad arguments (op %d of %d)", op, e->n_ops);
    int rc = check_types(e, field_type, accum);
    if (rc) return rc;
    if (e->n_ops == 1) {
        EllTune t;
        rc = rbfx_ell_pick(e, 1, field_type, accum, 0, &t);
        if (rc) return rc;
        if (e->storage == RBFX_F64) return launch_spmm_fpt<double, double, double, 1>(e, t, 1, d_u, d_out);
        if (field_type == RBFX_F32 && accum == RBFX_F64) return launch_spmm_fpt<float, float, double, 1>(e, t, 1, d_u, d_out);
        if (field_type == RBFX_F32) return launch_spmm_fpt<float, float, float, 1>(e, t, 1, d_u, d_out);
        return launch_spmm_fpt<float, double, double, 1>(e, t, 1, d_u, d_out);
    }
    const int block = 256;
    int n_tiles = (e->n_rows + block - 1) / block;
    int nb = grid_blocks(n_tiles);
    hipStream_t s = e->ctx->stream;
    if (e->storage == RBFX_F64)
        ell_spmv_strided_kernel<double, double, double><<<nb, block, 0, s>>>(e->idx_t, (const double*)e->w_t, (const double*)d_u, (double*)d_out, e->order, e->n_rows, e->width, e->n_ops, op, n_tiles, nb);
    else if (field_type == RBFX_F32 && accum == RBFX_F64)
        ell_spmv_strided_kernel<float, float, double><<<nb, block, 0, s>>>(e->idx_t, (const float*)e->w_t, (const float*)d_u, (float*)d_out, e->order, e->n_rows, e->width, e->n_ops, op, n_tiles, nb);
    else if (field_type == RBFX_F32)
        ell_spmv_strided_kernel<float, float, float><<<nb, block, 0, s>>>(e->idx_t, (const float*)e->w_t, (const float*)d_u, (float*)d_out, e->order, e->n_rows, e->width, e->n_ops, op, n_tiles, nb);
    else
        ell_spmv_strided_kernel<float, double, double><<<nb, block, 0, s>>>(e->idx_t, (const float*)e->w_t, (const double*)d_u, (double*)d_out, e->order, e->n_rows, e->width, e->n_ops, op, n_tiles, nb);
    RBFX_LAUNCH_CHECK(e->ctx, "ell_spmv_strided_kernel");
    return RBFX_OK;
}

}  // extern "C"
