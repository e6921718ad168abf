// Internal declarations shared by the HIP translation units of librbfx.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "rbfx.h"

// FP64 add and multiply that round on their own. hipcc contracts a * b + c into a fused
// multiply-add by default, also across inlined calls (this HIP version's __dadd_rn and
// __dmul_rn are plain + and *); operations written under contract(off) carry no contraction
// permission, so these two stay separate wherever they are inlined.
__device__ __forceinline__ double dadd_nc(double a, double b) {
#pragma clang fp contract(off)
    return a + b;
}
__device__ __forceinline__ double dmul_nc(double a, double b) {
#pragma clang fp contract(off)
    return a * b;
}

struct rbfx_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t t0 = nullptr, t1 = nullptr;
    int n_cu = 0;
    int clock_khz = 0;
    char name[256] = {0};
    std::string err;
    // Device memory kept for the next object (rbfx_pool_alloc): blocks not in use, oldest first, and the
    // sizes of those handed out.
    struct Block {
        void* p;
        size_t bytes;
    };
    std::mutex pool_mu;
    std::vector<Block> idle;
    std::unordered_map<void*, size_t> lent;
    size_t idle_bytes = 0, idle_max = 0;
};

// Records a formatted message on ctx (or the global slot) and returns code.
int rbfx_fail(rbfx_ctx* ctx, int code, const char* fmt, ...);

#define RBFX_HIP_CHECK(ctx, call)                                                             \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return rbfx_fail((ctx), RBFX_E_HIP, "%s failed: %s (%s:%d)", #call,                \
                             hipGetErrorString(e_), __FILE__, __LINE__);                      \
    } while (0)

// Checks the last launch on this thread.
#define RBFX_LAUNCH_CHECK(ctx, what)                                                          \
    do {                                                                                      \
        hipError_t e_ = hipGetLastError();                                                    \
        if (e_ != hipSuccess)                                                                 \
            return rbfx_fail((ctx), RBFX_E_HIP, "launch of %s failed: %s", (what),            \
                             hipGetErrorString(e_));                                          \
    } while (0)

// hipMalloc that, when memory runs out, gives the idle blocks of the device's contexts back and tries again.
hipError_t rbfx_malloc(rbfx_ctx* ctx, void** p, size_t bytes);

// Device memory of objects that are built and dropped again and again (operator sets, tile tables, the
// Stokes factor, the search's scratch). Blocks of at least 1 MiB stay with the context when they
// are freed and serve the next request of up to their size and at least 4/5 of it; contents are
// whatever the last user left. Everything that touches such memory is work on the context's
// stream, so a block's next use comes after its last one without a wait. At most 1/64 of the
// device's memory and 32 blocks are kept; they are given back with the context, by
// rbfx_release_idle, or when an allocation of any context on the device fails.
hipError_t rbfx_pool_alloc_bytes(rbfx_ctx* ctx, void** p, size_t bytes);
void rbfx_pool_free(rbfx_ctx* ctx, void* p);
template <typename T>
hipError_t rbfx_pool_alloc(rbfx_ctx* ctx, T** p, size_t bytes) {
    void* v = nullptr;
    const hipError_t e = rbfx_pool_alloc_bytes(ctx, &v, bytes);
    *p = static_cast<T*>(v);
    return e;
}

// Pieces of one allocation, each on 256 bytes: carve once without memory for the size, then with it.
struct Carver {
    unsigned char* base = nullptr;
    size_t used = 0;
    template <typename T>
    void take(T** p, size_t n) {
        if (base) *p = reinterpret_cast<T*>(base + used);
        used += (n * sizeof(T) + 255) / 256 * 256;
    }
};

static inline unsigned popcount32(uint32_t x) { return (unsigned)__builtin_popcount(x); }
