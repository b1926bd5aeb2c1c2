// Grouped FP64 GEMM launches: C = alpha * op(A) * op(B) + beta * C for a table
// of independent problems of any shape, tiles as in gemm_tile.hpp.
#include "gemm_tile.hpp"

#include <algorithm>
#include "prof.hpp"

namespace syn {

// Tile order of a single problem.  Work-groups are dealt to the XCDs round
// robin (id % 8), and each XCD has its own L2.  XCD x gets whole tile rows
// (or columns), zig-zag paired within every 16: rows x and 15 - x, then 16 + x
// and 31 - x, ...  A whole row reuses its A panel in one L2, and when the
// work of a tile grows or shrinks along the rows (a triangular hint) each XCD
// gets the same sum of long and short rows.  Columns are dealt instead when
// the hint makes the work depend on the column (op(B) triangular).  Shapes
// that do not split into such groups keep contiguous ranges per XCD.
__device__ __forceinline__ int64_t tile_of_block(int64_t bid, int64_t total, int64_t tiles_n, int tri) {
    const int64_t tiles_m = total / tiles_n;
    const bool by_col = (tri & (8 | 16)) && !(tri & (1 | 2 | 4));
    const int64_t lines = by_col ? tiles_n : tiles_m, len = by_col ? tiles_m : tiles_n;
    if (lines % (2 * kXcds) != 0 || total < 2 * kXcds) return xcd_remap(bid, total);
    const int64_t x = bid % kXcds, j = bid / kXcds, u = j / len, g = u / 2;
    const int64_t line = 2 * kXcds * g + ((u & 1) ? 2 * kXcds - 1 - x : x), pos = j % len;
    return by_col ? pos * tiles_n + line : line * tiles_n + pos;
}

template <int BM, int BN, int BK, int WM, int WN, typename CT, typename Tab>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, 2) void gemm_f64_grouped(KernelTable<Tab> tab, int n_items, int64_t total) {
    const syn_gemm_item *__restrict__ items = items_of(tab);
    if (n_items == 1) {
        gemm_f64_tile<BM, BN, BK, WM, WN, CT>(items[0],
                                              tile_of_block(blockIdx.x, total, items[0].tiles_n, items[0].tri));
        return;
    }
    const int64_t bid = xcd_remap(blockIdx.x, total);
    const syn_gemm_item &P = items[find_item(items, n_items, bid)];
    gemm_f64_tile<BM, BN, BK, WM, WN, CT>(P, bid - P.block_start);
}

// Persistent form of the grouped launch: a fixed grid of work-groups (a
// multiple of the 8 XCDs) walks the logical tiles b = blockIdx.x + i * grid,
// so every tile of a work-group stays on its XCD and the XCD keeps the same
// contiguous tile range as the one-tile-per-work-group launch.  For launches
// of many small tiles (thousands of chains' products) it saves the per-tile
// work-group start and drain; a tile computes exactly what it computes there.
template <int BM, int BN, int BK, int WM, int WN, typename CT = double>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, 2) void gemm_f64_grouped_persistent(
    const syn_gemm_item *__restrict__ items, int n_items, int64_t total) {
    for (int64_t b = blockIdx.x; b < total; b += gridDim.x) {
        if (b != (int64_t)blockIdx.x) __syncthreads();   // LDS of the previous tile is free
        const int64_t bid = xcd_remap(b, total);
        const syn_gemm_item &P = items[find_item(items, n_items, bid)];
        gemm_f64_tile<BM, BN, BK, WM, WN, CT>(P, bid - P.block_start);
    }
}

template <int BM, int BN, int BK, int WM, int WN, typename CT = double>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, 2) void gemm_f64_single(syn_gemm_item P) {
    const int64_t total = (int64_t)gridDim.x;
    gemm_f64_tile<BM, BN, BK, WM, WN, CT>(P, tile_of_block(blockIdx.x, total, P.tiles_n, P.tri));
}

// Two independent problems in one launch: work-groups [0, tiles0) take the
// first, the rest the second (each in its own tile order).  For short
// dependent chains of small products (the recursive Cholesky-inverse) this
// saves a launch and lets the two run side by side.
template <int BM, int BN, int BK, int WM, int WN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, 2) void gemm_f64_pair(syn_gemm_item P0, int64_t tiles0,
                                                                             syn_gemm_item P1, int64_t tiles1) {
    const int64_t bid = blockIdx.x;
    if (bid < tiles0)
        gemm_f64_tile<BM, BN, BK, WM, WN, double>(P0, tile_of_block(bid, tiles0, P0.tiles_n, P0.tri));
    else
        gemm_f64_tile<BM, BN, BK, WM, WN, double>(P1, tile_of_block(bid - tiles0, tiles1, P1.tiles_n, P1.tri));
}

// Launches of few 64 x 64 tiles, four work-groups a tile (gemm_f64_quad).
// Up to half of the 256 compute units busy with 64 x 64 tiles the quadrants
// are faster at every K (us, 64 x 64 tiles / quadrants): 1 tile K = 16 4.7 /
// 4.6, 256 16.9 / 8.0, 1024 57 / 24; 64 tiles of 256 18.3 / 9.5, 128 of 64
// 8.0 / 6.5, of 256 19.4 / 12.8.  256 tiles: 16 6.2 / 7.8, 64 9.1 / 9.2, 256
// 21.6 / 19.9; 512 of 256 29.5 / 33.2.
constexpr int kQuadK = 32;
constexpr int64_t kQuadMax = 128;

template <typename CT, typename Tab>
__global__ __launch_bounds__(256, 2) void gemm_quad_grouped(KernelTable<Tab> tab, int n_items, int64_t total) {
    const syn_gemm_item *__restrict__ items = items_of(tab);
    const int64_t b = xcd_remap(blockIdx.x, 4 * total), t = b >> 2;
    const syn_gemm_item &P = items[find_item(items, n_items, t)];
    gemm_f64_quad<kQuadK, CT>(P, t - P.block_start, (int)(b & 3));
}

template <typename CT>
__global__ __launch_bounds__(256, 2) void gemm_quad_single(syn_gemm_item P) {
    const int64_t b = xcd_remap(blockIdx.x, (int64_t)gridDim.x);
    gemm_f64_quad<kQuadK, CT>(P, b >> 2, (int)(b & 3));
}

__global__ __launch_bounds__(256, 2) void gemm_quad_pair(syn_gemm_item P0, int64_t tiles0, syn_gemm_item P1) {
    const int64_t b = xcd_remap(blockIdx.x, (int64_t)gridDim.x), t = b >> 2;
    if (t < tiles0)
        gemm_f64_quad<kQuadK, double>(P0, t, (int)(b & 3));
    else
        gemm_f64_quad<kQuadK, double>(P1, t - tiles0, (int)(b & 3));
}

// Split-K form of a single problem: work-group b computes K slice
// b / tiles of tile b % tiles; slice 0 writes C (with beta), slice s > 0
// writes the partial product into ws + (s - 1) m ws_ld, and
// gemm_splitk_reduce adds the partials into C.  Used where the tiles alone
// would leave most of the chip idle for a last partial round (a Gram
// matrix's lower triangle: 528 tiles of 128 on 512 work-group slots).
template <int BM, int BN, int BK, int WM, int WN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, 2) void gemm_f64_splitk(syn_gemm_item P, int64_t tiles,
                                                                               int64_t kc, double *ws,
                                                                               int64_t ws_ld) {
    const int64_t bid = blockIdx.x;
    const int64_t slice = bid / tiles, tloc = bid - slice * tiles;
    const int64_t t = tile_of_block(tloc, tiles, P.tiles_n, P.tri);
    const int64_t klo = slice * kc;
    const int64_t khi = klo + kc < P.k ? klo + kc : P.k;
    if (slice > 0) {
        P.C = ws + (slice - 1) * P.m * ws_ld;
        P.ldc = ws_ld;
        P.beta = 0.0;
    }
    gemm_f64_tile<BM, BN, BK, WM, WN, double>(P, t, klo, khi);
}

__global__ __launch_bounds__(256) void gemm_splitk_reduce(double *C, int64_t ldc, const double *ws, int64_t ws_ld,
                                                          int64_t m, int64_t n, int extra, int lower) {
    const int64_t total = m * n;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int64_t i = e / n, j = e - i * n;
        if (lower && j > i) continue;
        double v = C[i * ldc + j];
        for (int q = 0; q < extra; ++q) v += ws[q * m * ws_ld + i * ws_ld + j];
        C[i * ldc + j] = v;
    }
}

// One GEMM launched with its descriptor passed by value (no device table):
// used by the library's own multi-step routines (Cholesky, CholeskyQR, ...).
int gemm_f64_pair_launch(syn_gemm_item P0, syn_gemm_item P1, hipStream_t s) {
    const bool live0 = P0.m > 0 && P0.n > 0 && !(P0.k <= 0 && P0.beta == 1.0);
    const bool live1 = P1.m > 0 && P1.n > 0 && !(P1.k <= 0 && P1.beta == 1.0);
    if (!live0 || !live1) {
        if (live0) return gemm_f64_launch(P0, s);
        if (live1) return gemm_f64_launch(P1, s);
        return SYN_OK;
    }
    // one tile size for both, chosen by the larger output
    const int64_t area = std::max(P0.m * P0.n, P1.m * P1.n);
    const int tile = (area >= (int64_t)256 * 128 * 128) ? 1 : 0;
    const int64_t bm = tile ? 128 : 64;
    P0.tiles_n = (P0.n + bm - 1) / bm;
    P1.tiles_n = (P1.n + bm - 1) / bm;
    P0.block_start = P1.block_start = 0;
    const int64_t t0 = ((P0.m + bm - 1) / bm) * P0.tiles_n, t1 = ((P1.m + bm - 1) / bm) * P1.tiles_n;
    double fl = 0.0;
    for (const syn_gemm_item *P : {&P0, &P1}) {
        double f = 2.0 * (double)P->m * (double)P->n * (double)P->k;
        const int nbits = __builtin_popcount((unsigned)P->tri);
        if (nbits == 1) f *= 0.5;
        if (nbits >= 2) f /= 3.0;
        fl += f;
    }
    ProfScope ps(tile ? kTagGemmPair128 : kTagGemmPair64, fl, s);
    if (!tile && t0 + t1 <= kQuadMax)
        hipLaunchKernelGGL(gemm_quad_pair, dim3((unsigned)(4 * (t0 + t1))), dim3(256), 0, s, P0, t0, P1);
    else if (tile)
        hipLaunchKernelGGL((gemm_f64_pair<128, 128, 16, 64, 64>), dim3((unsigned)(t0 + t1)), dim3(256), 0, s, P0, t0,
                           P1, t1);
    else
        hipLaunchKernelGGL((gemm_f64_pair<64, 64, 16, 32, 32>), dim3((unsigned)(t0 + t1)), dim3(256), 0, s, P0, t0,
                           P1, t1);
    SYN_LAUNCH_CHECK("gemm_f64_pair_launch");
    return SYN_OK;
}

int gemm_f64_launch(syn_gemm_item P, hipStream_t s, bool mixed) {
    if (P.m <= 0 || P.n <= 0) return SYN_OK;
    if (P.k <= 0 && P.beta == 1.0) return SYN_OK;
    const int tile = (P.m * P.n >= (int64_t)256 * 128 * 128) ? 1 : 0;
    const int64_t bm = tile ? 128 : 64;
    P.tiles_n = (P.n + bm - 1) / bm;
    const int64_t tiles = ((P.m + bm - 1) / bm) * P.tiles_n;
    P.block_start = 0;
    // algorithmic flops: a structural-zero hint halves the product (a third
    // for triangle x triangle)
    double fl = 2.0 * (double)P.m * (double)P.n * (double)P.k;
    const int nbits = __builtin_popcount((unsigned)P.tri);
    if (nbits == 1) fl *= 0.5;
    if (nbits >= 2) fl /= 3.0;
    if (mixed) {
        ProfScope ps(tile ? kTagGemmMixed128 : kTagGemmMixed64, fl, s);
        if (!tile && tiles <= kQuadMax)
            hipLaunchKernelGGL(gemm_quad_single<float>, dim3((unsigned)(4 * tiles)), dim3(256), 0, s, P);
        else if (tile)
            hipLaunchKernelGGL((gemm_f64_single<128, 128, 16, 64, 64, float>), dim3((unsigned)tiles), dim3(256), 0,
                               s, P);
        else
            hipLaunchKernelGGL((gemm_f64_single<64, 64, 16, 32, 32, float>), dim3((unsigned)tiles), dim3(256), 0, s,
                               P);
        SYN_LAUNCH_CHECK("gemm_f64_launch (mixed)");
        return SYN_OK;
    }
    ProfScope ps(tile ? kTagGemmSingle128 : kTagGemmSingle64, fl, s);
    if (!tile && tiles <= kQuadMax)
        hipLaunchKernelGGL(gemm_quad_single<double>, dim3((unsigned)(4 * tiles)), dim3(256), 0, s, P);
    else if (tile)
        hipLaunchKernelGGL((gemm_f64_single<128, 128, 16, 64, 64>), dim3((unsigned)tiles), dim3(256), 0, s, P);
    else
        hipLaunchKernelGGL((gemm_f64_single<64, 64, 16, 32, 32>), dim3((unsigned)tiles), dim3(256), 0, s, P);
    SYN_LAUNCH_CHECK("gemm_f64_launch");
    return SYN_OK;
}

// One problem split along K when its tiles alone would leave work-group
// slots idle in the last round (a Gram matrix's lower triangle: 528 tiles of
// 128 on 512 slots).  ws holds ws_cap doubles for the partial products (the K slices
// after the first).  With 2 work-groups per CU the chip holds 2 * CUs tiles
// at a time; for `live` computed tiles (the lower triangle for tri bit 1),
// s slices take ceil(live s / slots) rounds of 1/s of the work; s <= 4 and
// every slice keeps at least 256 of K.
int gemm_f64_split_launch(syn_gemm_item P, hipStream_t s, double *ws, int64_t ws_cap) {
    if (P.m <= 0 || P.n <= 0) return SYN_OK;
    if (P.k <= 0 && P.beta == 1.0) return SYN_OK;
    const int tile = (P.m * P.n >= (int64_t)256 * 128 * 128) ? 1 : 0;
    if (ws == nullptr || P.k < 512) return gemm_f64_launch(P, s);
    static int slots = 0;
    if (slots == 0) {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
        slots = 2 * cus;
    }
    const int64_t bm = tile ? 128 : 64;
    const int64_t tm = (P.m + bm - 1) / bm, tn = (P.n + bm - 1) / bm;
    int64_t live = 0;
    if (P.tri & 1)
        for (int64_t r = 0; r < tm; ++r) live += (r + 1 < tn ? r + 1 : tn);
    else
        live = tm * tn;
    int best = 1;
    double best_cost = (double)((live + slots - 1) / slots);
    for (int sl = 2; sl <= 4; ++sl) {
        const int64_t kc = ((P.k + sl - 1) / sl + 15) / 16 * 16;
        if (kc < 256 || (int64_t)(sl - 1) * P.m * P.n > ws_cap) break;
        const double cost = (double)((live * sl + slots - 1) / slots) / sl;
        if (cost < best_cost - 1e-9) {
            best_cost = cost;
            best = sl;
        }
    }
    if (best == 1) return gemm_f64_launch(P, s);
    const int64_t kc = ((P.k + best - 1) / best + 15) / 16 * 16;
    P.tiles_n = tn;
    P.block_start = 0;
    const int64_t tiles = tm * tn;
    double fl = 2.0 * (double)P.m * (double)P.n * (double)P.k;
    const int nbits = __builtin_popcount((unsigned)P.tri);
    if (nbits == 1) fl *= 0.5;
    if (nbits >= 2) fl /= 3.0;
    ProfScope ps(tile ? kTagGemmSplitK128 : kTagGemmSplitK64, fl, s);
    if (tile)
        hipLaunchKernelGGL((gemm_f64_splitk<128, 128, 16, 64, 64>), dim3((unsigned)(tiles * best)), dim3(256), 0, s,
                           P, tiles, kc, ws, P.n);
    else
        hipLaunchKernelGGL((gemm_f64_splitk<64, 64, 16, 32, 32>), dim3((unsigned)(tiles * best)), dim3(256), 0, s,
                           P, tiles, kc, ws, P.n);
    SYN_LAUNCH_CHECK("gemm_f64_split_launch");
    int64_t blocks = (P.m * P.n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(gemm_splitk_reduce, dim3((unsigned)blocks), dim3(256), 0, s, (double *)P.C, P.ldc,
                       (const double *)ws, P.n, P.m, P.n, best - 1, (P.tri & 1) ? 1 : 0);
    SYN_LAUNCH_CHECK("gemm_f64_split_launch reduce");
    return SYN_OK;
}

syn_gemm_item make_gemm(const double *A, int64_t lda, int ta, const double *B, int64_t ldb, int tb, double *C,
                        int64_t ldc, int64_t m, int64_t n, int64_t k, double alpha, double beta, int tri) {
    syn_gemm_item P;
    memset(&P, 0, sizeof(P));
    P.A = A;
    P.B = B;
    P.C = C;
    P.m = m;
    P.n = n;
    P.k = k;
    P.lda = lda;
    P.ldb = ldb;
    P.ldc = ldc;
    P.alpha = alpha;
    P.beta = beta;
    P.transA = ta;
    P.transB = tb;
    P.tri = tri;
    return P;
}

}  // namespace syn

namespace syn {

// Grouped launches of more tiles than this many work-group slots run
// persistent (kPersistentGrid work-groups: 512 CUs' worth of two each would
// be 512; four per CU for the 64-tile kernels).
constexpr int64_t kPersistentMin = 4096;
constexpr int64_t kPersistentGrid = 1024;

// A table by value has few items: its launches of 4096 tiles and more are of
// large problems, whose tiles gain nothing from the persistent form.
template <typename CT, typename Tab>
static int launch_grouped(Tab tab, int n_items, int64_t total, int tile, hipStream_t s, const char *who) {
    constexpr bool kDevice = __is_same(Tab, DeviceTable<syn_gemm_item>);
    const bool pers = kDevice && total >= kPersistentMin && n_items > 1;
    const unsigned grid = (unsigned)(pers ? kPersistentGrid : total);
    bool quad = false;
    if constexpr (!__is_same(CT, bf16s)) {
        quad = tile == 0 && total <= kQuadMax;
        if (quad)
            hipLaunchKernelGGL((gemm_quad_grouped<CT, Tab>), dim3((unsigned)(4 * total)), dim3(256), 0, s, tab, n_items,
                               total);
    }
    if constexpr (kDevice) {
        if (pers && tile == 0)
            hipLaunchKernelGGL((gemm_f64_grouped_persistent<64, 64, 16, 32, 32, CT>), dim3(grid), dim3(256), 0, s,
                               tab, n_items, total);
        else if (pers)
            hipLaunchKernelGGL((gemm_f64_grouped_persistent<128, 128, 16, 64, 64, CT>), dim3(grid), dim3(256), 0, s,
                               tab, n_items, total);
    }
    if (!pers && !quad) {
        if (tile == 0)
            hipLaunchKernelGGL((gemm_f64_grouped<64, 64, 16, 32, 32, CT, Tab>), dim3(grid), dim3(256), 0, s, tab,
                               n_items, total);
        else
            hipLaunchKernelGGL((gemm_f64_grouped<128, 128, 16, 64, 64, CT, Tab>), dim3(grid), dim3(256), 0, s, tab,
                               n_items, total);
    }
    SYN_LAUNCH_CHECK(who);
    return SYN_OK;
}

// the three compute types' entry points: items on the device, or on the host
// and passed by value
template <typename CT>
static int gemm_entry(const syn_gemm_item *items, int n_items, int64_t total_blocks, int tile, void *stream, int tag64,
                      int tag128, bool host, const char *who) {
    if (n_items < 0 || total_blocks < 0) {
        set_error("%s: negative item or block count", who);
        return SYN_EINVAL;
    }
    if (host)
        if (int rc = inline_check(items, n_items, who)) return rc;
    if (n_items == 0 || total_blocks == 0) return SYN_OK;
    if (total_blocks > 0x7fffffffLL) {
        set_error("%s: %lld tiles exceed the grid limit", who, (long long)total_blocks);
        return SYN_EINVAL;
    }
    hipStream_t s = (hipStream_t)stream;
    if (tile != 0 && tile != 1) {
        set_error("%s: unknown tile configuration %d", who, tile);
        return SYN_EINVAL;
    }
    ProfScope ps(tile == 1 ? tag128 : tag64, -1.0, s);
    if (!host) return launch_grouped<CT>(DeviceTable<syn_gemm_item>{items}, n_items, total_blocks, tile, s, who);
    return launch_inline(items, n_items, [&](const auto &tab) {
        return launch_grouped<CT>(tab, n_items, total_blocks, tile, s, who);
    });
}

}  // namespace syn

extern "C" int syn_gemm_f64(const syn_gemm_item *items, int n_items, int64_t total_blocks, int tile, void *stream) {
    using namespace syn;
    return gemm_entry<double>(items, n_items, total_blocks, tile, stream, kTagGemmGrouped64, kTagGemmGrouped128, false, "syn_gemm_f64");
}

extern "C" int syn_gemm_f64_host(const syn_gemm_item *items, int n_items, int64_t total_blocks, int tile, void *stream) {
    using namespace syn;
    return gemm_entry<double>(items, n_items, total_blocks, tile, stream, kTagGemmGrouped64, kTagGemmGrouped128, true, "syn_gemm_f64_host");
}

extern "C" int syn_gemm_mixed_f64(const syn_gemm_item *items, int n_items, int64_t total_blocks, int tile, void *stream) {
    using namespace syn;
    return gemm_entry<float>(items, n_items, total_blocks, tile, stream, kTagGemmMixed64, kTagGemmMixed128, false, "syn_gemm_mixed_f64");
}

extern "C" int syn_gemm_mixed_f64_host(const syn_gemm_item *items, int n_items, int64_t total_blocks, int tile, void *stream) {
    using namespace syn;
    return gemm_entry<float>(items, n_items, total_blocks, tile, stream, kTagGemmMixed64, kTagGemmMixed128, true, "syn_gemm_mixed_f64_host");
}

extern "C" int syn_gemm_bf16_f64(const syn_gemm_item *items, int n_items, int64_t total_blocks, int tile, void *stream) {
    using namespace syn;
    return gemm_entry<bf16s>(items, n_items, total_blocks, tile, stream, kTagGemmBf1664, kTagGemmBf16128, false, "syn_gemm_bf16_f64");
}

extern "C" int syn_gemm_bf16_f64_host(const syn_gemm_item *items, int n_items, int64_t total_blocks, int tile, void *stream) {
    using namespace syn;
    return gemm_entry<bf16s>(items, n_items, total_blocks, tile, stream, kTagGemmBf1664, kTagGemmBf16128, true, "syn_gemm_bf16_f64_host");
}
