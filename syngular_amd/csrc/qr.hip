// Batched Householder QR, one work-group per matrix.
//
// Used wherever the reference calls numpy.linalg.qr on a site unfolding: the
// QR-truncation ">>" sweep, decompose, and left/right orthonormalisation.
// The leading nb = min(n, keep) columns are factored (the later columns only
// enter R = Q^T A, which the caller forms with the GEMM), then the first kq
// columns of the complete orthogonal factor are accumulated backwards,
// Q = H_0 H_1 ... H_{p-1} [I; 0]  (Golub & Van Loan, Alg. 5.1.2 / 5.2.1).
//
// Parallel layout: the 64 lanes of a wave own 64 consecutive columns and the
// 8 waves own 8 contiguous row segments, so every global access of the
// row-major W and Q is coalesced along a row; the per-column partial dot
// products of the segments are combined through LDS.  The working copy of
// the leading block lives in LDS when it fits and in the caller's workspace
// (L2-resident at these sizes) otherwise.
//
// That column-by-column form is for matrices of more than 512 rows or 96
// factored columns; the others go by panels of 32 columns in registers
// (hh_tile.hpp) with the compact WY products on the MFMA.
#include "common.hpp"
#include "hh_tile.hpp"
#include "prof.hpp"

#include <algorithm>

namespace syn {

constexpr int kQrThreads = 512;
constexpr int kQrWaves = kQrThreads / 64;
constexpr int kColWaves = 4;
constexpr int64_t kQrLdsDoubles = (96 * 1024) / 8;

template <int NW>
__device__ __forceinline__ void seg_bounds(int64_t lo, int64_t hi, int w, int64_t &a, int64_t &b) {
    const int64_t len = hi > lo ? hi - lo : 0;
    const int64_t per = (len + NW - 1) / NW;
    a = lo + per * w;
    b = a + per;
    if (a > hi) a = hi;
    if (b > hi) b = hi;
}

// Apply H = I - tau v v^T (v = [1; M[j+1:, j]] taken from V) to columns
// [c_lo, c_hi) of M (rows j..m-1).  V and M may alias (factorisation step).
template <int NW>
__device__ __forceinline__ void apply_reflector(const double *V, int64_t ldv, int64_t j, double tau, double *M,
                                                int64_t ldm, int64_t m, int64_t c_lo, int64_t c_hi,
                                                double (*red)[64]) {
    // rows loaded together: column j is not among those written, but the
    // compiler cannot know, and row by row each would wait for the last store
    // (8 matrices of 128 x 64, segments of up to 32 rows: 409 us by four, 437 by
    // eight, more by sixteen; taller segments not measured)
    constexpr int U = 4;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int64_t r0, r1;
    seg_bounds<NW>(j + 1, m, w, r0, r1);
    for (int64_t c0 = c_lo; c0 < c_hi; c0 += 64) {
        const int64_t c = c0 + lane;
        const bool act = c < c_hi;
        double part = 0.0;
        if (act) {
            const double *vp = V + r0 * ldv + j, *mp = M + r0 * ldm + c;
            int left = (int)(r1 - r0);
            for (; left >= U; left -= U, vp += U * ldv, mp += U * ldm) {
                double v[U], x[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    v[u] = vp[u * ldv];
                    x[u] = mp[u * ldm];
                }
#pragma unroll
                for (int u = 0; u < U; ++u) part = fma(v[u], x[u], part);
            }
            for (; left > 0; --left, vp += ldv, mp += ldm) part = fma(*vp, *mp, part);
        }
        red[w][lane] = part;
        __syncthreads();
        double dot = 0.0;
        if (act) {
            dot = M[j * ldm + c];
#pragma unroll
            for (int q = 0; q < NW; ++q) dot += red[q][lane];
        }
        const double f = tau * dot;
        __syncthreads();  // every wave has read red[] and M[j, c] before row j changes
        if (act) {
            if (w == 0) M[j * ldm + c] -= f;
            const double *vp = V + r0 * ldv + j;
            double *mp = M + r0 * ldm + c;
            int left = (int)(r1 - r0);
            for (; left >= U; left -= U, vp += U * ldv, mp += U * ldm) {
                double v[U], x[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    v[u] = vp[u * ldv];
                    x[u] = mp[u * ldm];
                }
#pragma unroll
                for (int u = 0; u < U; ++u) mp[u * ldm] = fma(-f, v[u], x[u]);
            }
            for (; left > 0; --left, vp += ldv, mp += ldm) *mp = fma(-f, *vp, *mp);
        }
    }
}

template <int NW, bool IN_LDS>
__device__ __forceinline__ void qr_one(const syn_qr_item &P, double *lds_w) {
    constexpr int kTaus = 128;   // reflector scales kept in LDS; the rest is read back
    __shared__ double red[NW][64], taus[kTaus];
    const int64_t m = P.m, n = P.n, keep = P.keep;
    const int64_t nb = n < keep ? n : keep;
    const int64_t kq = keep < m ? keep : m;
    const int64_t p = m < nb ? m : nb;
    double *W = IN_LDS ? lds_w : P.work;
    const int tid = threadIdx.x;

    if (m * nb < 0x7fffffff) {
        for (unsigned e = tid; e < (unsigned)(m * nb); e += 64 * NW) {
            const unsigned i = e / (unsigned)nb, j = e - i * (unsigned)nb;
            W[e] = P.a[i * P.rs + j * P.cs];
        }
    } else {
        for (int64_t e = tid; e < m * nb; e += 64 * NW) {
            const int64_t i = e / nb, j = e - i * nb;
            W[e] = P.a[i * P.rs + j * P.cs];
        }
    }
    __syncthreads();

    for (int64_t j = 0; j < p; ++j) {
        double part = 0.0;
        for (int64_t i = j + 1 + tid; i < m; i += (64 * NW)) {
            const double v = W[i * nb + j];
            part = fma(v, v, part);
        }
        part = row_sum(lk_sum(part));   // wave_sum's pairs, without its trips through LDS
        if ((tid & 63) == 0) red[tid >> 6][0] = part;
        __syncthreads();
        // every thread works out the reflector: no second exchange
        double xn2 = 0.0;
#pragma unroll
        for (int q = 0; q < NW; ++q) xn2 += red[q][0];
        const double alpha = W[j * nb + j];
        double tau = 0.0, scal = 0.0, beta = alpha;
        if (xn2 > 0.0) {
            beta = -copysign(sqrt(fma(alpha, alpha, xn2)), alpha);
            tau = (beta - alpha) / beta;
            scal = 1.0 / (alpha - beta);
        }
        if (tid == 0) {
            if (j < kTaus) taus[j] = tau;
            P.tau[j] = tau;
        }
        if (tau != 0.0) {
            for (int64_t i = j + 1 + tid; i < m; i += (64 * NW)) W[i * nb + j] *= scal;
            __syncthreads();
            if (tid == 0) W[j * nb + j] = beta;   // all have read alpha
            apply_reflector<NW>(W, nb, j, tau, W, nb, m, j + 1, nb, red);
        }
        __syncthreads();
    }

    // Q is accumulated row-major in P.q (or, for q_trans, in the workspace
    // tail and transposed on the way out).
    double *Q = P.q_trans ? P.work + m * nb : P.q;
    const int64_t ldq = P.q_trans ? kq : P.ldq;
    for (int64_t e = tid; e < m * kq; e += (64 * NW)) {
        const int64_t i = e / kq, c = e - i * kq;
        Q[i * ldq + c] = (i == c) ? 1.0 : 0.0;
    }
    __syncthreads();
    for (int64_t j = p - 1; j >= 0; --j) {
        const double tau = j < kTaus ? taus[j] : P.tau[j];
        if (tau != 0.0) apply_reflector<NW>(W, nb, j, tau, Q, ldq, m, j, kq, red);
        __syncthreads();
    }
    if (P.q_trans) {
        for (int64_t e = tid; e < m * kq; e += (64 * NW)) {
            const int64_t c = e / m, i = e - c * m;
            P.q[c * P.ldq + i] = Q[i * ldq + c];
        }
    }
}

// Panels of kHhCols columns factored in registers, W (the leading block) in
// the workspace: each panel's reflectors are applied to the columns right of
// it, and at the end, from the last panel back, to [I; 0], 16 columns per
// wave.  A column costs about a microsecond of dependent steps (two barriers)
// instead of a pass over the matrix by rows.  One matrix through ops.qr_many,
// before and after: 64 x 32 198 / 74 us, 128 x 64 656 / 181, 256 x 64 2018 /
// 245, 96 x 90 772 / 226, 512 x 24 1086 / 172.
constexpr int64_t kTileRows = 512, kTileCols = 96;
constexpr int kTilePanels = (int)kTileCols / kHhCols;
template <int NW, int ROWS, int PANELS, bool SMALL>
struct QrTileSmem {
    HhSmem<NW, ROWS, SMALL> hh;
    double T[PANELS][kHhCols * kHhCols];
};

template <int RT, int NW, typename Smem>
__device__ __forceinline__ void qr_tile(const syn_qr_item &P, Smem &sm) {
    constexpr int NT = 64 * NW;
    const int m = (int)P.m, nb = (int)(P.n < P.keep ? P.n : P.keep), kq = (int)(P.keep < P.m ? P.keep : P.m);
    const int p = m < nb ? m : nb, tid = threadIdx.x, wv = tid >> 6;
    double *W = P.work;
    for (int e = tid; e < m * nb; e += NT) {
        const int i = e / nb, j = e - i * nb;
        W[e] = P.a[i * P.rs + j * P.cs];
    }
    __syncthreads();
    for (int j0 = 0; j0 < p; j0 += kHhCols) {
        const int b = p - j0 < kHhCols ? p - j0 : kHhCols;
        double *Wp = W + (int64_t)j0 * nb + j0, *T = sm.T[j0 / kHhCols];
        hh_panel_regs<RT, NW>(Wp, nb, m - j0, b, T, kHhCols, P.tau + j0, nullptr, 0, sm.hh);
        for (int c = j0 + b + 16 * wv; c < p; c += 16 * NW)
            hh_apply_wave(Wp, nb, m - j0, b, T, kHhCols, true, W + (int64_t)j0 * nb + c, nb, p - c < 16 ? p - c : 16);
        __syncthreads();
    }
    double *Q = P.q_trans ? P.work + (int64_t)m * nb : P.q;
    const int64_t ldq = P.q_trans ? kq : P.ldq;
    for (int e = tid; e < m * kq; e += NT) {
        const int i = e / kq, c = e - i * kq;
        Q[i * ldq + c] = (i == c) ? 1.0 : 0.0;
    }
    __syncthreads();
    for (int j0 = (p - 1) / kHhCols * kHhCols; j0 >= 0; j0 -= kHhCols) {
        const int b = p - j0 < kHhCols ? p - j0 : kHhCols;
        for (int c = j0 + 16 * wv; c < kq; c += 16 * NW)
            hh_apply_wave(W + (int64_t)j0 * nb + j0, nb, m - j0, b, sm.T[j0 / kHhCols], kHhCols, false,
                          Q + j0 * ldq + c, ldq, kq - c < 16 ? kq - c : 16);
        __syncthreads();
    }
    if (P.q_trans) {
        for (int e = tid; e < m * kq; e += NT) {
            const int c = e / m, i = e - c * m;
            P.q[c * P.ldq + i] = Q[i * ldq + c];
        }
    }
}

// lds_cap: doubles of dynamic LDS the launch holds; a matrix whose leading
// block fits works in LDS, a larger one in its workspace.
template <int NW>
__device__ __forceinline__ void qr_columns(const syn_qr_item &P, double *lds_w, int64_t lds_cap) {
    const int64_t nb = P.n < P.keep ? P.n : P.keep;
    if (P.m * nb <= lds_cap)
        qr_one<NW, true>(P, lds_w);
    else
        qr_one<NW, false>(P, lds_w);
}

// Matrices of any shape and form.  One work-group fits a compute unit (107 KB of
// LDS with the static part, 200 registers a thread), so a launch of more matrices
// than the chip has units takes the two kernels below for what they are for.
// (Rows as in the blocked QR's panels: with the 512 that it needs, the other
// places in LDS cost a two-site gate at chi = 64 3 of 247 us.)
typedef QrTileSmem<kQrWaves, 1024, kTilePanels, false> QrAnySmem;
template <typename Tab>
__global__ __launch_bounds__(kQrThreads) void qr_kernel(KernelTable<Tab> tab, int64_t lds_cap) {
    extern __shared__ double lds_w[];
    const syn_qr_item &P = items_of(tab)[blockIdx.x];
    const int64_t nb = P.n < P.keep ? P.n : P.keep;
    if (P.columns == SYN_QR_COLUMNS) {
        if (threadIdx.x >= 64 * kColWaves) return;   // whole waves: the others' barriers do not wait for them
        qr_columns<kColWaves>(P, lds_w, lds_cap);
    } else if (P.m <= kTileRows && nb <= kTileCols) {
        QrAnySmem &sm = *(QrAnySmem *)lds_w;
        if (P.m <= 128)
            qr_tile<1, kQrWaves>(P, sm);
        else if (P.m <= 256)
            qr_tile<2, kQrWaves>(P, sm);
        else
            qr_tile<4, kQrWaves>(P, sm);
    } else
        qr_columns<kQrWaves>(P, lds_w, lds_cap);
}

// The column-by-column form by four waves, whatever the shape, with the LDS
// that the launch's matrices need.  The mixed sweep asks for it: it rounds its
// factors to FP32, where another order of the FP64 sums, no less exact, now and
// then ends on the neighbouring FP32 number, so this order is part of that
// form's results.
template <typename Tab>
__global__ __launch_bounds__(64 * kColWaves) void qr_columns_kernel(KernelTable<Tab> tab, int64_t lds_cap) {
    extern __shared__ double lds_w[];
    qr_columns<kColWaves>(items_of(tab)[blockIdx.x], lds_w, lds_cap);
}

// Matrices of up to 16 NW rows (NW 1, 2, 4): the panel form by NW waves, the same
// bits as by eight, whose other waves hold no rows.
template <int NW, typename Tab>
__global__ __launch_bounds__(64 * NW, 3) void qr_rows_kernel(KernelTable<Tab> tab) {
    constexpr int ROWS = 16 * NW, PANELS = (ROWS + kHhCols - 1) / kHhCols;
    __shared__ QrTileSmem<NW, ROWS, PANELS, true> sm;
    const syn_qr_item &P = items_of(tab)[blockIdx.x];
    if (P.m <= ROWS && (P.n < P.keep ? P.n : P.keep) <= kTileCols)
        qr_tile<1, NW>(P, sm);
    else   // not a matrix of the class: right, if slow
        qr_one<NW, false>(P, nullptr);
}

template <typename Kernel>
static int qr_lds(Kernel *kern, size_t most, const char *who) {
    return hip_check(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most), who);
}

// every launch holds what the panel form needs; the other form its lds_cap
template <typename Tab>
static int qr_launch(Tab tab, int n_items, int64_t lds_doubles, hipStream_t s) {
    static bool attr_set = false;
    if (!attr_set) {
        const size_t most = std::max(sizeof(QrAnySmem), (size_t)kQrLdsDoubles * sizeof(double));
        if (int rc = qr_lds(qr_kernel<Tab>, most, "syn_qr_f64: hipFuncSetAttribute")) return rc;
        attr_set = true;
    }
    const size_t lds = std::max(sizeof(QrAnySmem), (size_t)lds_doubles * sizeof(double));
    ProfScope ps(kTagQr, 0.0, s);
    hipLaunchKernelGGL(qr_kernel<Tab>, dim3(n_items), dim3(kQrThreads), lds, s, tab, lds_doubles);
    SYN_LAUNCH_CHECK("syn_qr_f64 launch");
    return SYN_OK;
}

}  // namespace syn

extern "C" int syn_qr_f64(const syn_qr_item *items, int n_items, void *stream) {
    using namespace syn;
    if (n_items < 0) {
        set_error("syn_qr_f64: negative item count");
        return SYN_EINVAL;
    }
    if (n_items == 0) return SYN_OK;
    return qr_launch(DeviceTable<syn_qr_item>{items}, n_items, kQrLdsDoubles, (hipStream_t)stream);
}

extern "C" int syn_qr_f64_host(const syn_qr_item *items, int n_items, void *stream) {
    return syn_qr_sized_f64_host(items, n_items, syn::kQrLdsDoubles, stream);
}

extern "C" int syn_qr_sized_f64(const syn_qr_item *items, int n_items, int64_t lds_doubles, void *stream) {
    using namespace syn;
    if (n_items < 0 || lds_doubles < 0 || lds_doubles > kQrLdsDoubles) {
        set_error("syn_qr_sized_f64: bad item count %d or LDS size %lld (at most %lld doubles)", n_items,
                  (long long)lds_doubles, (long long)kQrLdsDoubles);
        return SYN_EINVAL;
    }
    if (n_items == 0) return SYN_OK;
    return qr_launch(DeviceTable<syn_qr_item>{items}, n_items, lds_doubles, (hipStream_t)stream);
}

extern "C" int syn_qr_sized_f64_host(const syn_qr_item *items, int n_items, int64_t lds_doubles, void *stream) {
    using namespace syn;
    if (int rc = inline_check(items, n_items, "syn_qr_sized_f64_host")) return rc;
    if (lds_doubles < 0 || lds_doubles > kQrLdsDoubles) {
        set_error("syn_qr_sized_f64_host: bad LDS size %lld (at most %lld doubles)", (long long)lds_doubles,
                  (long long)kQrLdsDoubles);
        return SYN_EINVAL;
    }
    if (n_items == 0) return SYN_OK;
    return launch_inline(items, n_items,
                         [&](const auto &tab) { return qr_launch(tab, n_items, lds_doubles, (hipStream_t)stream); });
}

// tables of many matrices, so from device memory only
extern "C" int syn_qr_columns_f64(const syn_qr_item *items, int n_items, int64_t lds_doubles, void *stream) {
    using namespace syn;
    if (n_items < 0 || (n_items && !items) || lds_doubles < 0 || lds_doubles > kQrLdsDoubles) {
        set_error("syn_qr_columns_f64: bad item count %d or LDS size %lld (at most %lld doubles)", n_items,
                  (long long)lds_doubles, (long long)kQrLdsDoubles);
        return SYN_EINVAL;
    }
    if (n_items == 0) return SYN_OK;
    typedef DeviceTable<syn_qr_item> Tab;
    static bool attr_set = false;
    if (!attr_set) {
        if (int rc = qr_lds(qr_columns_kernel<Tab>, (size_t)kQrLdsDoubles * sizeof(double),
                            "syn_qr_columns_f64: hipFuncSetAttribute"))
            return rc;
        attr_set = true;
    }
    hipStream_t s = (hipStream_t)stream;
    ProfScope ps(kTagQr, 0.0, s);
    hipLaunchKernelGGL(qr_columns_kernel<Tab>, dim3(n_items), dim3(64 * kColWaves), (size_t)lds_doubles * sizeof(double),
                       s, Tab{items}, lds_doubles);
    SYN_LAUNCH_CHECK("syn_qr_columns_f64 launch");
    return SYN_OK;
}

extern "C" int syn_qr_rows_f64(const syn_qr_item *items, int n_items, int64_t rows, void *stream) {
    using namespace syn;
    if (n_items < 0 || (n_items && !items) || rows < 1 || rows > 64) {
        set_error("syn_qr_rows_f64: bad item count %d or rows %lld (at most 64)", n_items, (long long)rows);
        return SYN_EINVAL;
    }
    if (n_items == 0) return SYN_OK;
    typedef DeviceTable<syn_qr_item> Tab;
    hipStream_t s = (hipStream_t)stream;
    ProfScope ps(kTagQr, 0.0, s);
    if (rows <= 16)
        hipLaunchKernelGGL((qr_rows_kernel<1, Tab>), dim3(n_items), dim3(64), 0, s, Tab{items});
    else if (rows <= 32)
        hipLaunchKernelGGL((qr_rows_kernel<2, Tab>), dim3(n_items), dim3(128), 0, s, Tab{items});
    else
        hipLaunchKernelGGL((qr_rows_kernel<4, Tab>), dim3(n_items), dim3(256), 0, s, Tab{items});
    SYN_LAUNCH_CHECK("syn_qr_rows_f64 launch");
    return SYN_OK;
}
