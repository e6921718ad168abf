// Tile tables for the LDS-staged gathers (rbfx_ell_build_local), built on the device.
//
// The tables are those of rbfx_build_local_tables (csrc/rbfx_knn.cpp), entry for entry: chunks of
// 64 * lt positions are cut greedily into tiles of at most lt consecutive positions with at most
// cap distinct stencil nodes, each tile lists its nodes in ascending order, and every entry of
// the layout holds its node's 16-bit place in its tile's list.
//   local_cut_kernel      one block per chunk walks its tiles: all entries of the next lt
//                         positions go into a hash table in LDS that keeps, per node, the first
//                         position that names it; the counts of new nodes per position, summed
//                         along the positions, say after how many of them the cap is reached
//   local_offsets_kernel  tile starts and list offsets from the chunks' counts
//   local_list_kernel     one block per tile: its distinct nodes through a hash table, sorted in
//                         LDS, then every entry's place through the same table
// Bounds: the cut is a chain of about 65 tiles per chunk (hash insertions and barriers, 49 chunks
// at 400k rows), the lists are LDS work with one pass over the indices. At 400,009 rows, n = 50,
// 128-row tiles of at most 768 nodes: cut 0.40 ms, lists 0.105 ms (the indices and places alone
// are 0.12 GB). The host build (OpenMP on 16 threads, the index array down and the tables up over
// PCIe) took about 95 ms there: set-up and first SpMM 105 -> 6.0 ms by this build alone, 1.26 ms with the
// packing and the kept memory that followed.
#include <algorithm>
#include <climits>
#include <vector>

#include "rbfx_ell_common.h"
#include "rbfx_ell_local.h"

namespace {

constexpr int CUT_THREADS = 1024;
constexpr int LIST_THREADS = 512;
constexpr uint32_t EMPTY = 0xffffffffu;  // node indices are non-negative int32
constexpr int HASH_MAX = 16384;          // slots: 8 bytes each in the cut, 6 in the lists

__device__ __forceinline__ int hash_first(uint32_t node, int H) {
    return (int)((node * 2654435761u) >> 15) & (H - 1);  // H a power of two, at most 2^17
}

// Slot of `node`, inserted if absent. Ends because the table always has an empty slot.
__device__ __forceinline__ int hash_insert(uint32_t* keys, int H, uint32_t node) {
    int s = hash_first(node, H);
    for (;;) {
        uint32_t k = keys[s];
        if (k == EMPTY) k = atomicCAS(&keys[s], EMPTY, node);
        if (k == node || k == EMPTY) return s;
        s = (s + 1) & (H - 1);
    }
}

// Slot of a node that the table holds.
__device__ __forceinline__ int hash_find(const uint32_t* keys, int H, uint32_t node) {
    int s = hash_first(node, H);
    while (keys[s] != node) s = (s + 1) & (H - 1);
    return s;
}

// Chunk c's tiles: start position t_pos[c * chunk + i] and node count t_cnt[c * chunk + i] of its
// i-th tile; c_info[3c ..] = {tiles, nodes of all its tiles, most nodes of one tile}.
__global__ void __launch_bounds__(CUT_THREADS) local_cut_kernel(const int32_t* __restrict__ idx_t, int n_rows, int width,
                                                               int lt, int cap, int chunk, int H,
                                                               int32_t* __restrict__ t_pos, int32_t* __restrict__ t_cnt,
                                                               int32_t* __restrict__ c_info) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint32_t* keys = reinterpret_cast<uint32_t*>(smem);
    int* first = reinterpret_cast<int*>(keys + H);
    __shared__ int fresh[128];  // nodes first named by position start + r
    __shared__ int s_len, s_cnt;
    const int t = threadIdx.x, c = blockIdx.x;
    const int p_lo = c * chunk, p_hi = min(n_rows, p_lo + chunk);
    const int sh = __ffs(lt) - 1;
    int n_t = 0, total = 0, most = 0;
    for (int p = p_lo; p < p_hi;) {
        const int rows = min(lt, p_hi - p);
        for (int s = t; s < H; s += CUT_THREADS) {
            keys[s] = EMPTY;
            first[s] = INT_MAX;
        }
        if (t < 128) fresh[t] = 0;
        __syncthreads();
        for (int e = t; e < (width << sh); e += CUT_THREADS) {
            const int r = e & (lt - 1), j = e >> sh;
            if (r < rows) {
                const int32_t node = idx_t[ell_row_base(p + r, width) + (size_t)j * ELL_TILE];
                atomicMin(&first[hash_insert(keys, H, (uint32_t)node)], r);
            }
        }
        __syncthreads();
        for (int s = t; s < H; s += CUT_THREADS)
            if (keys[s] != EMPTY) atomicAdd(&fresh[first[s]], 1);
        __syncthreads();
        if (t < 64) {  // one wave: two positions per lane, summed along the positions
            const int a = fresh[2 * t], b = fresh[2 * t + 1];
            int sum = a + b;
            for (int o = 1; o < 64; o <<= 1) {
                const int up = __shfl_up(sum, o);
                if (t >= o) sum += up;
            }
            const int before = sum - a - b;  // distinct nodes of the positions before this lane's
            // positions that fit: the counts never decrease, so they are the first ones
            const bool f0 = 2 * t < rows && (cap <= 0 || 2 * t == 0 || before + a <= cap);
            const bool f1 = 2 * t + 1 < rows && (cap <= 0 || sum <= cap);
            const int len = __popcll(__ballot(f0)) + __popcll(__ballot(f1));
            if (len - 1 == 2 * t) {
                s_len = len;
                s_cnt = before + a;
            } else if (len - 1 == 2 * t + 1) {
                s_len = len;
                s_cnt = sum;
            }
        }
        __syncthreads();
        const int len = s_len, cnt = s_cnt;
        if (t == 0) {
            t_pos[p_lo + n_t] = p;
            t_cnt[p_lo + n_t] = cnt;
        }
        n_t++;
        total += cnt;
        most = max(most, cnt);
        p += len;  // len >= 1: the first position always fits
        // the next round writes s_len only after barriers every thread passes
    }
    if (t == 0) {
        c_info[3 * c] = n_t;
        c_info[3 * c + 1] = total;
        c_info[3 * c + 2] = most;
    }
}

// One wave per chunk: pos and off of its tiles from c_base[2c ..] = {first tile, first list entry}.
__global__ void __launch_bounds__(64) local_offsets_kernel(const int32_t* __restrict__ t_pos,
                                                           const int32_t* __restrict__ t_cnt,
                                                           const int32_t* __restrict__ c_info,
                                                           const int32_t* __restrict__ c_base, int n_chunks, int chunk,
                                                           int n_rows, int32_t* __restrict__ pos,
                                                           int32_t* __restrict__ off) {
    const int c = blockIdx.x, lane = threadIdx.x;
    const int n_t = c_info[3 * c], tile0 = c_base[2 * c];
    int run = c_base[2 * c + 1];
    for (int i0 = 0; i0 < n_t; i0 += 64) {
        const int i = i0 + lane;
        const int cnt = i < n_t ? t_cnt[(size_t)c * chunk + i] : 0;
        int sum = cnt;
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(sum, o);
            if (lane >= o) sum += up;
        }
        if (i < n_t) {
            pos[tile0 + i] = t_pos[(size_t)c * chunk + i];
            off[tile0 + i] = run + sum - cnt;
        }
        run += __shfl(sum, 63);
    }
    if (c == n_chunks - 1 && lane == 0) {
        pos[tile0 + n_t] = n_rows;
        off[tile0 + n_t] = run;
    }
}

// Tile t's sorted node list and the places of its entries in it. H hash slots, P list entries
// (a power of two, at least the longest list).
__global__ void __launch_bounds__(LIST_THREADS) local_list_kernel(const int32_t* __restrict__ idx_t, int width, int lt,
                                                                 const int32_t* __restrict__ pos,
                                                                 const int32_t* __restrict__ off, int H, int P,
                                                                 int32_t* __restrict__ nodes,
                                                                 uint16_t* __restrict__ loc_idx) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint32_t* keys = reinterpret_cast<uint32_t*>(smem);
    uint32_t* list = keys + H;
    uint16_t* place = reinterpret_cast<uint16_t*>(list + P);
    __shared__ int s_n;
    const int t = threadIdx.x, tile = blockIdx.x;
    const int start = pos[tile], rows = pos[tile + 1] - start;
    const int k0 = off[tile], K = off[tile + 1] - k0;
    const int sh = __ffs(lt) - 1;
    for (int s = t; s < H; s += LIST_THREADS) keys[s] = EMPTY;
    for (int i = t; i < P; i += LIST_THREADS) list[i] = EMPTY;  // sorts behind every node
    if (t == 0) s_n = 0;
    __syncthreads();
    for (int e = t; e < (width << sh); e += LIST_THREADS) {
        const int r = e & (lt - 1), j = e >> sh;
        if (r < rows) hash_insert(keys, H, (uint32_t)idx_t[ell_row_base(start + r, width) + (size_t)j * ELL_TILE]);
    }
    __syncthreads();
    for (int s = t; s < H; s += LIST_THREADS) {
        const uint32_t k = keys[s];
        if (k != EMPTY) list[atomicAdd(&s_n, 1)] = k;  // K of them, K <= P
    }
    __syncthreads();
    int PP = 2;  // the power of two this tile's list needs
    while (PP < K) PP <<= 1;
    for (int k = 2; k <= PP; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = t; i < PP; i += LIST_THREADS) {
                const int q = i ^ j;
                if (q > i) {
                    const uint32_t a = list[i], b = list[q];
                    if ((a > b) == ((i & k) == 0)) {
                        list[i] = b;
                        list[q] = a;
                    }
                }
            }
            __syncthreads();
        }
    for (int i = t; i < K; i += LIST_THREADS) {
        const uint32_t node = list[i];
        nodes[k0 + i] = (int32_t)node;
        place[hash_find(keys, H, node)] = (uint16_t)i;
    }
    __syncthreads();
    for (int e = t; e < (width << sh); e += LIST_THREADS) {
        const int r = e & (lt - 1), j = e >> sh;
        if (r < rows) {
            const size_t q = ell_row_base(start + r, width) + (size_t)j * ELL_TILE;
            loc_idx[q] = place[hash_find(keys, H, (uint32_t)idx_t[q])];
        }
    }
}

int pow2_at_least(int v, int lo) {
    int p = lo;
    while (p < v) p <<= 1;
    return p;
}

}  // namespace

bool rbfx_local_tables_device(rbfx_ell* e, int lt, int cap, size_t lds_limit, LocalTables* T, int* rc) {
    rbfx_ctx* ctx = e->ctx;
    hipStream_t st = ctx->stream;
    *rc = RBFX_OK;
    // The cut keeps every entry of lt positions in its table (an eighth of the slots stays
    // empty): up to 112 slots per stencil with 128-row tiles, 224 and 448 with 64 and 32.
    const long long entries = (long long)lt * e->width;
    if (entries > HASH_MAX / 8 * 7) return false;
    const int Hc = pow2_at_least((int)(entries * 8 / 7), 1024);
    const size_t cut_lds = (size_t)Hc * 8;
    if (cut_lds + 1024 > lds_limit) return false;
    const int chunk = 64 * lt, n = e->n_rows;
    const int n_chunks = (int)(((long long)n + chunk - 1) / chunk);
    int32_t* scratch = nullptr;  // t_pos, t_cnt (a tile per row at most), c_info, c_base
    const size_t ints = 2 * (size_t)n + 5 * (size_t)n_chunks;
    auto fail = [&](hipError_t err, int code) {
        hipStreamSynchronize(st);
        rbfx_pool_free(ctx, scratch);
        rbfx_pool_free(ctx, T->pos);
        rbfx_pool_free(ctx, T->off);
        rbfx_pool_free(ctx, T->nodes);
        rbfx_pool_free(ctx, T->idx);
        *T = LocalTables();
        *rc = rbfx_fail(ctx, code, "ell_build_local: %s", hipGetErrorString(err));
        return true;
    };
    hipError_t err;
    if ((err = rbfx_pool_alloc(ctx, &scratch, ints * sizeof(int32_t))) != hipSuccess) return fail(err, RBFX_E_NOMEM);
    int32_t *t_pos = scratch, *t_cnt = t_pos + n, *c_info = t_cnt + n, *c_base = c_info + 3 * (size_t)n_chunks;
    local_cut_kernel<<<n_chunks, CUT_THREADS, cut_lds, st>>>(e->idx_t, n, e->width, lt, cap, chunk, Hc, t_pos, t_cnt, c_info);
    std::vector<int32_t> info(3 * (size_t)n_chunks), base(2 * (size_t)n_chunks);
    if ((err = hipGetLastError()) != hipSuccess ||
        (err = hipMemcpyAsync(info.data(), c_info, info.size() * sizeof(int32_t), hipMemcpyDeviceToHost, st)) != hipSuccess ||
        (err = hipStreamSynchronize(st)) != hipSuccess)
        return fail(err, RBFX_E_HIP);
    int tiles = 0, most = 0;
    long long nodes = 0;
    for (int c = 0; c < n_chunks; c++) {
        base[2 * (size_t)c] = tiles;
        base[2 * (size_t)c + 1] = (int32_t)nodes;
        tiles += info[3 * (size_t)c];
        nodes += info[3 * (size_t)c + 1];
        most = std::max(most, info[3 * (size_t)c + 2]);
    }
    // The lists keep the longest one in a table of twice its length (at most HASH_MAX slots)
    // beside the sorted copy; lists above 8192 nodes do not fit the LDS and are left to the host.
    const int P = pow2_at_least(most, 64), H = std::min(HASH_MAX, pow2_at_least(2 * most, 128));
    const size_t list_lds = (size_t)H * 6 + (size_t)P * 4;
    if (most > HASH_MAX / 2 || list_lds + 1024 > lds_limit) {
        rbfx_pool_free(ctx, scratch);
        return false;
    }
    const size_t all = (size_t)e->n_pad * e->width;
    if ((err = rbfx_pool_alloc(ctx, &T->pos, ((size_t)tiles + 1) * sizeof(int32_t))) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &T->off, ((size_t)tiles + 1) * sizeof(int32_t))) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &T->nodes, (size_t)std::max<long long>(1, nodes) * sizeof(int32_t))) != hipSuccess ||
        (err = rbfx_pool_alloc(ctx, &T->idx, all * sizeof(uint16_t))) != hipSuccess)
        return fail(err, RBFX_E_NOMEM);
    if ((err = hipMemcpyAsync(c_base, base.data(), base.size() * sizeof(int32_t), hipMemcpyHostToDevice, st)) != hipSuccess)
        return fail(err, RBFX_E_HIP);
    local_offsets_kernel<<<n_chunks, 64, 0, st>>>(t_pos, t_cnt, c_info, c_base, n_chunks, chunk, n, T->pos, T->off);
    // pad rows (they share the last layout tile with real ones) keep place 0
    const size_t last = ell_row_base(n - 1, e->width) / ((size_t)ELL_TILE * e->width) * ((size_t)ELL_TILE * e->width);
    if ((err = hipGetLastError()) != hipSuccess ||
        (err = hipMemsetAsync(T->idx + last, 0, (all - last) * sizeof(uint16_t), st)) != hipSuccess)
        return fail(err, RBFX_E_HIP);
    local_list_kernel<<<tiles, LIST_THREADS, list_lds, st>>>(e->idx_t, e->width, lt, T->pos, T->off, H, P, T->nodes, T->idx);
    if ((err = hipGetLastError()) != hipSuccess || (err = hipStreamSynchronize(st)) != hipSuccess)
        return fail(err, RBFX_E_HIP);
    rbfx_pool_free(ctx, scratch);
    T->n_tiles = tiles;
    T->k_max = most;
    return true;
}
