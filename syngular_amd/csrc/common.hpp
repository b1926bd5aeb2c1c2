// Shared helpers for the gfx950 kernels of syngular_amd.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "../../include/syngular_amd.h"

namespace syn {

// Thread-local message of the last failure (returned by syn_last_error).
void set_error(const char *fmt, ...);

inline int hip_check(hipError_t e, const char *what) {
    if (e != hipSuccess) {
        set_error("%s: %s", what, hipGetErrorString(e));
        return SYN_EHIP;
    }
    return SYN_OK;
}

#define SYN_LAUNCH_CHECK(what)                                   \
    do {                                                         \
        hipError_t _e = hipGetLastError();                       \
        if (_e != hipSuccess) return ::syn::hip_check(_e, what); \
    } while (0)

// Number of XCDs on MI355X.  Consecutive work-group ids are dealt round-robin
// to the XCDs; remapping so that each XCD receives a contiguous range of
// logical blocks keeps neighbouring tiles (which share operand panels) in the
// same L2.
constexpr int kXcds = 8;

__device__ __forceinline__ int64_t xcd_remap(int64_t bid, int64_t nblocks) {
    if (nblocks < 2 * kXcds) return bid;
    int64_t q = nblocks / kXcds, r = nblocks % kXcds;
    int64_t x = bid % kXcds, j = bid / kXcds;
    return x * q + (x < r ? x : r) + j;
}

// Items are sorted by block_start; find the item that owns logical block b.
template <typename Item>
__device__ __forceinline__ int find_item(const Item *items, int n, int64_t b) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (items[mid].block_start <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Item table of a launch: in device memory, or by value in the kernel's
// arguments when it comes from the host and has few items.  A table of one to a
// few dozen items otherwise costs a pinned allocation, a copy command of 3 us
// on the stream and the gap before the kernel that waits for it.  Two sizes, so
// that a single item does not carry kInlineBytes of arguments.
//
// A device table reaches its kernel as a __restrict__ pointer (KernelTable):
// only so does the compiler read items through the scalar unit and keep their
// fields in scalar registers.  Inside a struct argument it took them for memory
// that the kernel's own stores may change: a product of 8192 x 4096 x 2048
// 2459 us, mixed 1550, against 2060 and 1165.
constexpr size_t kInlineBytes = SYN_INLINE_BYTES;
template <typename Item>
using DeviceTable = const Item *;
template <typename Item, int N>
struct InlineTable {
    Item it[N];
};
template <typename Tab>
struct KernelTableOf {
    typedef Tab type;
};
template <typename Item>
struct KernelTableOf<const Item *> {
    typedef const Item *__restrict__ type;
};
template <typename Tab>
using KernelTable = typename KernelTableOf<Tab>::type;

template <typename Item>
__device__ __forceinline__ const Item *items_of(const Item *p) {
    return p;
}
template <typename Item, int N>
__device__ __forceinline__ const Item *items_of(const InlineTable<Item, N> &t) {
    return t.it;
}
template <typename Item>
constexpr int kInlineItems = (int)(kInlineBytes / sizeof(Item));

// launch(table) with the items as an InlineTable; the caller has checked n
template <typename Item, typename F>
inline int launch_inline(const Item *items, int n, F launch) {
    if (n == 1) {
        InlineTable<Item, 1> t;
        memcpy(t.it, items, sizeof(Item));
        return launch(t);
    }
    InlineTable<Item, kInlineItems<Item>> t;
    memcpy(t.it, items, (size_t)n * sizeof(Item));
    memset((void *)(t.it + n), 0, (kInlineItems<Item> - n) * sizeof(Item));
    return launch(t);
}
// SYN_EINVAL when a host table cannot go by value
template <typename Item>
inline int inline_check(const Item *items, int n, const char *who) {
    if (n < 0 || n > kInlineItems<Item> || (n && !items)) {
        set_error("%s: %d items (a host table holds at most %d)", who, n, kInlineItems<Item>);
        return SYN_EINVAL;
    }
    return SYN_OK;
}

// Work-group barrier that orders LDS only: global stores issued before it
// stay in flight.  For phases whose global writes no thread of the
// work-group reads back (a plain __syncthreads waits for them to land).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Host-side helpers shared by the multi-step routines (gemm.hip).
int gemm_f64_launch(syn_gemm_item P, hipStream_t s, bool mixed = false);
int gemm_f64_split_launch(syn_gemm_item P, hipStream_t s, double *ws, int64_t ws_cap);
// two independent FP64 problems in one launch (one tile size for both)
int gemm_f64_pair_launch(syn_gemm_item P0, syn_gemm_item P1, hipStream_t s);
syn_gemm_item make_gemm(const double *A, int64_t lda, int ta, const double *B, int64_t ldb, int tb, double *C,
                        int64_t ldc, int64_t m, int64_t n, int64_t k, double alpha, double beta, int tri = 0);

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

}  // namespace syn
