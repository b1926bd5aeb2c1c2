// Householder panel of up to 32 columns in registers, shared by the
// one-work-group QR (qr.hip) and the blocked QR's panel kernel (hhblock.hip).
//
// The panel's rows are dealt to the NW waves in tiles of 16 (tile t of wave
// w: rows 16 (w + NW t) ..), columns to the 16 lanes li of a tile, two tiles
// wide: lane (li, lk) holds rows lk + 4 r of columns li and 16 + li.  A
// column costs two barriers: its entries and partial norms go through LDS,
// then each wave's partial dot products with every column.  What bounds it is
// that chain (LDS round trips, one square root and two divisions), about a
// microsecond a column, not the arithmetic.  (Sums over the waves are shared
// out over the lanes: 600 x 600 keeping 300 1.72 -> 1.52 ms, 256 x 64 275 ->
// 245 us.)
#pragma once
#include "common.hpp"

namespace syn {

typedef double hv4d __attribute__((ext_vector_type(4)));

constexpr int kHhCols = 32;

// sum over the four rows of 16 lanes, in every lane
__device__ __forceinline__ double lk_sum(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const auto l32 = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)u, false, false);
    const auto h32 = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
    const double s = __builtin_bit_cast(double, (uint64_t)h32[0] << 32 | l32[0]) +
                     __builtin_bit_cast(double, (uint64_t)h32[1] << 32 | l32[1]);
    const uint64_t w = __builtin_bit_cast(uint64_t, s);
    const auto l16 = __builtin_amdgcn_permlane16_swap((unsigned)w, (unsigned)w, false, false);
    const auto h16 = __builtin_amdgcn_permlane16_swap((unsigned)(w >> 32), (unsigned)(w >> 32), false, false);
    return __builtin_bit_cast(double, (uint64_t)h16[0] << 32 | l16[0]) +
           __builtin_bit_cast(double, (uint64_t)h16[1] << 32 | l16[1]);
}

// Sum over the 16 lanes of a DPP row, in every lane: row rotations in the
// vector unit, a few dozen cycles where a cross-lane exchange through LDS takes
// about sixty a step.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_f64<0x128>(v);   // row_ror:8, 4, 2, 1
    v += dpp_f64<0x124>(v);
    v += dpp_f64<0x122>(v);
    return v + dpp_f64<0x121>(v);
}

// For a panel of at most ROWS rows.  SMALL: the waves' parts of V^T V take the
// place of what the columns needed, for a barrier, so that more work-groups fit a
// compute unit.  A launch of one matrix keeps them apart (a two-site gate at chi =
// 300 takes 1.60 ms with them together, 1.58 apart).
template <int NW, int ROWS, bool SMALL = false>
struct HhSmem {
    double xs[ROWS];                     // the column being reflected
    double red[NW];                      // partial squared norms
    double part[NW][kHhCols];            // partial dot products
    double tau[kHhCols];
    double S[3][16][17];                 // V^T V, upper triangle by tiles (0,0), (0,1), (1,1)
    double Sp[NW][3][256];               // each wave's part of it
};
template <int NW, int ROWS>
struct HhSmem<NW, ROWS, true> {
    union {
        struct {
            double xs[ROWS];
            double red[NW];
            double part[NW][kHhCols];
        };
        double Sp[NW][3][256];
    };
    double tau[kHhCols];
    double S[3][16][17];
};

// Factors the m x b panel at A (row-major, leading dimension lda; m <= 16 NW
// RT <= ROWS, b <= 32) in place: R on and above the diagonal, v below (LAPACK dgeqrf:
// beta = -sign(alpha) norm, tau = 0 and v = e1 for a column already zero below
// the diagonal).  T (ld ldt): the upper triangular factor of I - V T V^T,
// zeros below, tau to tau_out.  Vx, when given (leading dimension ldv), gets
// V with its unit diagonal and zeros above.  Every thread of the work-group
// (64 NW) calls it; ends with a barrier.
template <int RT, int NW, int ROWS, bool SMALL>
__device__ __forceinline__ void hh_panel_regs(double *A, int64_t lda, int m, int b, double *T, int64_t ldt,
                                              double *tau_out, double *Vx, int64_t ldv, HhSmem<NW, ROWS, SMALL> &sm) {
    static_assert(16 * NW * RT <= ROWS, "rows of the panel");
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, lk = lane >> 4;
    double a[RT][2][4];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * (wv + NW * t) + lk + 4 * r, j = 16 * c + li;
                a[t][c][r] = (i < m && j < b) ? A[i * lda + j] : 0.0;
            }
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
        for (int jl = 0; jl < 16 && 16 * ct + jl < b; ++jl) {
            const int j = 16 * ct + jl;
            double sq = 0.0;
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * (wv + NW * t) + lk + 4 * r;
                    if (li == jl) sm.xs[i] = a[t][ct][r];
                    if (i > j) sq = fma(a[t][ct][r], a[t][ct][r], sq);
                }
            sq = lk_sum(sq);
            if (lane == jl) sm.red[wv] = sq;
            lds_barrier();
            const double xn2 = row_sum(li < NW ? sm.red[li & (NW - 1)] : 0.0);
            const double alpha = sm.xs[j];
            double tau = 0.0, scal = 0.0, beta = alpha;
            if (xn2 > 0.0) {
                beta = -copysign(sqrt(fma(alpha, alpha, xn2)), alpha);
                tau = (beta - alpha) / beta;
                scal = 1.0 / (alpha - beta);
            }
            if (tid == 0) sm.tau[j] = tau;
            if (tau == 0.0) {
                // no reflector: a NaN in the column stays in it
#pragma unroll
                for (int t = 0; t < RT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (li == jl && 16 * (wv + NW * t) + lk + 4 * r > j) a[t][ct][r] = 0.0;
                lds_barrier();   // all have read xs and red
                continue;
            }
            double v[RT][4], d0 = 0.0, d1 = 0.0;
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * (wv + NW * t) + lk + 4 * r;
                    const double x = i > j ? sm.xs[i] * scal : i == j ? 1.0 : 0.0;
                    v[t][r] = x;
                    if (li == jl && i >= j) a[t][ct][r] = i > j ? x : beta;
                    d0 = fma(x, a[t][0][r], d0);
                    d1 = fma(x, a[t][1][r], d1);
                }
            d0 = lk_sum(d0);
            d1 = lk_sum(d1);
            if (lk == 0) {
                sm.part[wv][li] = d0;
                sm.part[wv][16 + li] = d1;
            }
            lds_barrier();
            // a quarter of the waves' parts per row of lanes: all of them in
            // every lane made LDS reads a third of a column of 16 waves
            double f0 = 0.0, f1 = 0.0;
#pragma unroll
            for (int q = 0; q < NW; q += 4) {
                if constexpr (NW < 4) {
                    if (lk >= NW) continue;
                }
                f0 += sm.part[q + lk][li];
                f1 += sm.part[q + lk][16 + li];
            }
            f0 = lk_sum(f0);
            f1 = lk_sum(f1);
            f0 = li > j ? tau * f0 : 0.0;
            f1 = 16 + li > j ? tau * f1 : 0.0;
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    a[t][0][r] = fma(-v[t][r], f0, a[t][0][r]);
                    a[t][1][r] = fma(-v[t][r], f1, a[t][1][r]);
                }
        }
    }
    // the panel, V, and V^T V on the MFMA (a lane's V entries are both
    // operands: row lk + 4 r is the contraction index, column li the other)
    hv4d s00 = {0.0, 0.0, 0.0, 0.0}, s01 = s00, s11 = s00;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * (wv + NW * t) + lk + 4 * r;
            double v[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int j = 16 * c + li;
                const bool in = i < m && j < b;
                v[c] = !in || i < j ? 0.0 : i == j ? 1.0 : a[t][c][r];
                if (in) A[i * lda + j] = a[t][c][r];
                if (in && Vx) Vx[i * ldv + j] = v[c];
            }
            s00 = __builtin_amdgcn_mfma_f64_16x16x4f64(v[0], v[0], s00, 0, 0, 0);
            s01 = __builtin_amdgcn_mfma_f64_16x16x4f64(v[0], v[1], s01, 0, 0, 0);
            s11 = __builtin_amdgcn_mfma_f64_16x16x4f64(v[1], v[1], s11, 0, 0, 0);
        }
    if (SMALL) lds_barrier();   // all have read the last column's part
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int e = (lk + 4 * r) * 16 + li;
        sm.Sp[wv][0][e] = s00[r];
        sm.Sp[wv][1][e] = s01[r];
        sm.Sp[wv][2][e] = s11[r];
    }
    lds_barrier();
    for (int e = tid; e < 768; e += 64 * NW) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < NW; ++q) s += sm.Sp[q][e >> 8][e & 255];
        sm.S[e >> 8][(e & 255) >> 4][e & 15] = s;
    }
    lds_barrier();
    // T[a][j] = -tau_j sum_{a <= l < j} T[a][l] S[l][j], T[j][j] = tau_j: a
    // row depends on itself only, one lane each
    if (tid < kHhCols) {
        double row[kHhCols];
#pragma unroll
        for (int j = 0; j < kHhCols; ++j) {
            const double tj = j < b ? sm.tau[j] : 0.0;
            double s = 0.0;
#pragma unroll
            for (int l = 0; l < j; ++l)
                s = fma(row[l], l < 16 ? (j < 16 ? sm.S[0][l][j] : sm.S[1][l][j - 16]) : sm.S[2][l - 16][j - 16], s);
            row[j] = tid == j ? tj : tid < j ? -tj * s : 0.0;
            if (tid < b && j < b) T[tid * ldt + j] = row[j];
        }
    }
    if (tid < b && tau_out) tau_out[tid] = sm.tau[tid];
    __syncthreads();
}

// C <- (I - V op(T) V^T) C for 16 columns of C (m rows, leading dimension
// ldc; nc <= 16 of them live) by one wave: V (m x b, b <= 32) is the panel
// stored as R over v (leading dimension lda, unit diagonal implied), T its
// factor; op transposes T when tt (the factorisation's own update).  The
// products chain in registers: a result's rows are the lanes' lk + 4 r, the
// contraction layout of the next.
__device__ __forceinline__ void hh_apply_wave(const double *V, int64_t ldv, int m, int b, const double *T, int ldt,
                                              bool tt, double *C, int64_t ldc, int nc) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const bool cin = li < nc;
    auto vat = [&](int i, int j) -> double {
        if (i >= m || j >= b || i < j) return 0.0;
        return i == j ? 1.0 : V[i * ldv + j];
    };
    hv4d y[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll 4
    for (int i0 = 0; i0 < m; i0 += 4) {
        const int i = i0 + lk;
        const double c = (cin && i < m) ? C[i * ldc + li] : 0.0;
        y[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(vat(i, li), c, y[0], 0, 0, 0);
        y[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(vat(i, 16 + li), c, y[1], 0, 0, 0);
    }
    hv4d z[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll
    for (int rho = 0; rho < 2; ++rho)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = 16 * rho + 4 * r + lk;
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                const int i = 16 * o + li;
                const double t = (k < b && i < b) ? (tt ? T[k * ldt + i] : T[i * ldt + k]) : 0.0;
                z[o] = __builtin_amdgcn_mfma_f64_16x16x4f64(t, y[rho][r], z[o], 0, 0, 0);
            }
        }
    for (int i0 = 0; i0 < m; i0 += 16) {
        hv4d c;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = i0 + lk + 4 * r;
            c[r] = (cin && i < m) ? C[i * ldc + li] : 0.0;
        }
#pragma unroll
        for (int rho = 0; rho < 2; ++rho)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(-vat(i0 + li, 16 * rho + 4 * r + lk), z[rho][r], c, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = i0 + lk + 4 * r;
            if (cin && i < m) C[i * ldc + li] = c[r];
        }
    }
}

}  // namespace syn
