// Output tile of the FP64 GEMM on CDNA4 matrix cores (v_mfma_f64_16x16x4f64).
//
// C = alpha * op(A) * op(B) + beta * C for a table of independent problems of
// any shape.  A work-group of 4 waves owns one BM x BN output tile; each wave
// owns a WM x WN sub-tile held as (WM/16) x (WN/16) MFMA accumulators.  Operand
// tiles are staged through LDS stored k-major ([k][i] and [k][j]) so that the
// 16 lanes that feed one MFMA row read 16 consecutive doubles; rows are padded
// by one double to spread the transposed stores over the banks.  The K loop is
// double-buffered: the next global tile is loaded into registers while the
// current LDS tile feeds the MFMAs.  Each operand orientation is a separate
// instance (no per-element branches), which keeps a 128 x 128 tile within the
// register budget of two work-groups per compute unit, so one work-group's
// barrier and load waits are covered by the other's MFMAs.
//
// MFMA f64 16x16x4 operand layout (lane l of 64):
//   A: A[i = l%16][k = l/16]     B: B[k = l/16][j = l%16]
//   D: reg r of lane l holds D[i = l/16 + 4*r][j = l%16]  (checked against
//      NumPy on the device: rows 4g+r and g+4r differ unless g == r)
#pragma once
#include "common.hpp"

namespace syn {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// Compute types: double (v_mfma_f64_16x16x4f64) or float, the mixed form
// (operands rounded to FP32 when staged into LDS, v_mfma_f32_16x16x4f32 with
// FP32 accumulation; the result is stored as FP64).  The two MFMAs take the
// same operand layout; the output rows of lane l, register r are
// l/16 + 4r (f64) and 4(l/16) + r (f32).
template <typename CT>
struct Mfma;
template <>
struct Mfma<double> {
    typedef v4d acc_t;
    static __device__ __forceinline__ acc_t zero() { return v4d{0.0, 0.0, 0.0, 0.0}; }
    static __device__ __forceinline__ acc_t mac(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int r) { return lk + 4 * r; }
};
template <>
struct Mfma<float> {
    typedef v4f acc_t;
    static __device__ __forceinline__ acc_t zero() { return v4f{0.0f, 0.0f, 0.0f, 0.0f}; }
    static __device__ __forceinline__ acc_t mac(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};

// BF16 compute type (the precision form's contractions): operands rounded
// to bfloat16 (round to nearest even) when staged into LDS, stored as their
// 16-bit patterns, v_mfma_f32_16x16x16_bf16 with FP32 accumulation.  One
// MFMA covers K = 16: lane l holds A[i = l%16][k = 4(l/16) + v] and
// B[k = 4(l/16) + v][j = l%16] for v = 0..3; the output rows are those of
// the f32 MFMA, 4(l/16) + r.
struct bf16s {
    unsigned short bits;
};
typedef short v4s __attribute__((ext_vector_type(4)));
template <>
struct Mfma<bf16s> {
    typedef v4f acc_t;
    static __device__ __forceinline__ acc_t zero() { return v4f{0.0f, 0.0f, 0.0f, 0.0f}; }
    static __device__ __forceinline__ acc_t mac4(v4s a, v4s b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};

// FP64 -> staged operand: FP64, FP32 (round to nearest) or BF16 (FP32 first,
// then round to nearest even on the upper 16 bits; the inputs are finite).
template <typename CT>
__device__ __forceinline__ CT stage(double x) {
    return (CT)x;
}
template <>
__device__ __forceinline__ bf16s stage<bf16s>(double x) {
    unsigned u = __builtin_bit_cast(unsigned, (float)x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return bf16s{(unsigned short)(u >> 16)};
}

template <int BM, int BN, int BK, typename CT>
struct GemmSmem {
    CT As[2][BK][BM + 1];
    CT Bs[2][BK][BN + 1];
};

template <int BM, int BN, int BK, int WM, int WN, bool TA, bool TB, typename CT>
__device__ __forceinline__ void gemm_f64_tile_at(const syn_gemm_item &P, int64_t row0, int64_t col0,
                                                 GemmSmem<BM, BN, BK, CT> &sm, int64_t klo, int64_t khi) {
    constexpr int NW = (BM / WM) * (BN / WN);
    constexpr int NT = NW * 64;
    constexpr int TI = WM / 16, TJ = WN / 16;
    constexpr int EA = BM * BK / NT, EB = BK * BN / NT;
    static_assert(EA * NT == BM * BK && EB * NT == BK * BN, "tile/threads mismatch");
    auto &As = sm.As;
    auto &Bs = sm.Bs;

    const int tri = P.tri;
    const int64_t m = P.m, n = P.n, lda = P.lda, ldb = P.ldb;
    if (row0 >= m || col0 >= n) return;  // a size known on the device only: the launch covers its largest
    // K band of the structurally non-zero products for this tile
    int64_t kmin = 0, k = P.k;
    if (tri & 2) k = k < row0 + BM ? k : row0 + BM;
    if (tri & 8) k = k < col0 + BN ? k : col0 + BN;
    if (tri & 4) kmin = row0;
    if (tri & 16) kmin = kmin > col0 ? kmin : col0;
    if (kmin < klo) kmin = klo;   // this work-group's K slice (split-K); klo is a multiple of BK
    if (k > khi) k = khi;
    kmin = (kmin / BK) * BK;
    constexpr bool ta = TA, tb = TB;
    const double *__restrict__ A = (const double *)P.A;
    const double *__restrict__ B = (const double *)P.B;
    // The guarded loads below take these.  Where the item is a kernel argument the
    // compiler knows A and B to be global memory, and its guarded global loads wait
    // for each other (409 waits in place of 260); as flat loads they do not.  FP64
    // 704 x 740 x 2048 209 us with the former, 143 with the latter.
    const double *Ag = A, *Bg = B;
    asm("" : "+s"(Ag), "+s"(Bg));

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm0 = (w / (BN / WN)) * WM, wn0 = (w % (BN / WN)) * WN;

    double ra[EA], rb[EB];
    // Interior tiles (all BM rows, BN columns and BK steps of the K tile in
    // range) load through buffer instructions: element s of a thread sits at
    // base(k0) + voff + s * stride, with voff one VGPR computed once, s *
    // stride a scalar offset and the K tile's base in the scalar descriptor,
    // so the steady state spends no vector instructions on addresses or
    // bounds (the guarded form below costs about two per MFMA).  Offsets are
    // 32-bit: the path is taken for leading dimensions below 2^20 doubles,
    // which keeps every offset of a tile under 2^31.
    static_assert(NT % BK == 0 && NT % BM == 0 && NT % BN == 0, "thread/tile shapes");
    constexpr int kStepA = ta ? NT / BM : NT / BK;   // rows of the stored A per element step
    constexpr int kStepB = tb ? NT / BK : NT / BN;   // rows of the stored B per element step
    const bool ld_small = lda < (1 << 20) && ldb < (1 << 20);
    const int voff_a = ta ? ((tid / BM) * (int)lda + tid % BM) * 8 : ((tid / BK) * (int)lda + tid % BK) * 8;
    const int voff_b = tb ? ((tid / BK) * (int)ldb + tid % BK) * 8 : ((tid / BN) * (int)ldb + tid % BN) * 8;
    const int sstr_a = kStepA * (int)lda * 8, sstr_b = kStepB * (int)ldb * 8;
    auto load_fast = [&](int64_t k0) {
        const double *pa = ta ? A + k0 * lda + row0 : A + row0 * lda + k0;
        const double *pb = tb ? B + col0 * ldb + k0 : B + k0 * ldb + col0;
        const __amdgpu_buffer_rsrc_t sa = __builtin_amdgcn_make_buffer_rsrc((void *)pa, (short)0, 0x7fffffff, 0x00020000);
        const __amdgpu_buffer_rsrc_t sb = __builtin_amdgcn_make_buffer_rsrc((void *)pb, (short)0, 0x7fffffff, 0x00020000);
#pragma unroll
        for (int s = 0; s < EA; ++s)
            ra[s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(sa, voff_a, s * sstr_a, 0));
#pragma unroll
        for (int s = 0; s < EB; ++s)
            rb[s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(sb, voff_b, s * sstr_b, 0));
    };
    const bool tile_in = row0 + BM <= m && col0 + BN <= n && ld_small;
    auto load = [&](int64_t k0) {
        if (tile_in && k0 + BK <= k) {
            load_fast(k0);
            return;
        }
#pragma unroll
        for (int s = 0; s < EA; ++s) {
            int e = tid + NT * s;
            int r, c;
            if constexpr (!ta) { r = e / BK; c = e % BK; } else { c = e / BM; r = e % BM; }
            int64_t gi = row0 + r, gk = k0 + c;
            if constexpr (ta)
                ra[s] = (gi < m && gk < k) ? Ag[gk * lda + gi] : 0.0;
            else
                ra[s] = (gi < m && gk < k) ? Ag[gi * lda + gk] : 0.0;
        }
#pragma unroll
        for (int s = 0; s < EB; ++s) {
            int e = tid + NT * s;
            int j, c;
            if constexpr (!tb) { c = e / BN; j = e % BN; } else { j = e / BK; c = e % BK; }
            int64_t gj = col0 + j, gk = k0 + c;
            if constexpr (tb)
                rb[s] = (gj < n && gk < k) ? Bg[gj * ldb + gk] : 0.0;
            else
                rb[s] = (gj < n && gk < k) ? Bg[gk * ldb + gj] : 0.0;
        }
    };
    // Element s of a thread lands at a fixed LDS base plus a compile-time
    // multiple of s (the same (row, k) map as the loads: e = tid + NT s), so
    // the stores take immediate offsets instead of per-element arithmetic.
    constexpr int kLdsStepA = ta ? (NT / BM) * (BM + 1) : NT / BK;
    constexpr int kLdsStepB = tb ? NT / BK : (NT / BN) * (BN + 1);
    const int lds_a = ta ? (tid / BM) * (BM + 1) + tid % BM : (tid % BK) * (BM + 1) + tid / BK;
    const int lds_b = tb ? (tid % BK) * (BN + 1) + tid / BK : (tid / BN) * (BN + 1) + tid % BN;
    auto store = [&](int buf) {
        CT *sa = &As[buf][0][0] + lds_a;
        CT *sb = &Bs[buf][0][0] + lds_b;
#pragma unroll
        for (int s = 0; s < EA; ++s) sa[s * kLdsStepA] = stage<CT>(ra[s]);
#pragma unroll
        for (int s = 0; s < EB; ++s) sb[s * kLdsStepB] = stage<CT>(rb[s]);
    };

    typedef Mfma<CT> M;
    typename M::acc_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = M::zero();

    const int64_t nk = k > kmin ? (k - kmin + BK - 1) / BK : 0;
    load(kmin);
    store(0);
    __syncthreads();
    const int li = lane & 15, lk = lane >> 4;
    for (int64_t kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
        if (kt + 1 < nk) load(kmin + (kt + 1) * BK);
        if constexpr (__is_same(CT, bf16s)) {
            static_assert(BK % 16 == 0, "the bf16 MFMA takes K = 16");
#pragma unroll
            for (int kk = 0; kk < BK / 16; ++kk) {
                v4s a[TI], b[TJ];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
#pragma unroll
                    for (int i = 0; i < TI; ++i) a[i][v] = (short)As[cur][kk * 16 + 4 * lk + v][wm0 + i * 16 + li].bits;
#pragma unroll
                    for (int j = 0; j < TJ; ++j) b[j][v] = (short)Bs[cur][kk * 16 + 4 * lk + v][wn0 + j * 16 + li].bits;
                }
#pragma unroll
                for (int i = 0; i < TI; ++i)
#pragma unroll
                    for (int j = 0; j < TJ; ++j) acc[i][j] = M::mac4(a[i], b[j], acc[i][j]);
            }
            if (kt + 1 < nk) store(cur ^ 1);
            __syncthreads();
            continue;
        } else {
        // the operands of step kk + 1 are read from LDS while the MFMAs of
        // step kk run
        CT a[2][TI], b[2][TJ];
        auto read_ops = [&](int kk, int h) {
#pragma unroll
            for (int i = 0; i < TI; ++i) a[h][i] = As[cur][kk * 4 + lk][wm0 + i * 16 + li];
#pragma unroll
            for (int j = 0; j < TJ; ++j) b[h][j] = Bs[cur][kk * 4 + lk][wn0 + j * 16 + li];
        };
        read_ops(0, 0);
#pragma unroll
        for (int kk = 0; kk < BK / 4; ++kk) {
            if (kk + 1 < BK / 4) read_ops(kk + 1, (kk + 1) & 1);
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int j = 0; j < TJ; ++j) acc[i][j] = M::mac(a[kk & 1][i], b[kk & 1][j], acc[i][j]);
        }
        if (kt + 1 < nk) store(cur ^ 1);
        __syncthreads();
        }
    }

    double *__restrict__ C = (double *)P.C;
    const int64_t ldc = P.ldc;
    const double alpha = P.alpha, beta = P.beta;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int64_t gi = row0 + wm0 + i * 16 + M::row(lk, r);
                int64_t gj = col0 + wn0 + j * 16 + li;
                if (gi < m && gj < n) {
                    double v = alpha * (double)acc[i][j][r];
                    if (beta != 0.0) v += beta * C[gi * ldc + gj];
                    C[gi * ldc + gj] = v;
                }
            }
}

template <int BM, int BN, int BK, int WM, int WN, bool TA, bool TB, typename CT>
__device__ __forceinline__ void gemm_f64_tile_t(const syn_gemm_item &P, int64_t t, GemmSmem<BM, BN, BK, CT> &sm,
                                                int64_t klo, int64_t khi) {
    const int64_t row0 = (t / P.tiles_n) * BM, col0 = (t % P.tiles_n) * BN;
    if ((P.tri & 1) && col0 >= row0 + BM) return;  // tile strictly above the diagonal of C
    gemm_f64_tile_at<BM, BN, BK, WM, WN, TA, TB, CT>(P, row0, col0, sm, klo, khi);
}

// The operand orientation is fixed at compile time in each instance, so the
// loads carry no per-element branches and the register budget fits two
// work-groups per compute unit.
template <int BM, int BN, int BK, int WM, int WN, typename CT>
__device__ __forceinline__ void gemm_f64_tile(const syn_gemm_item &P, int64_t t, int64_t klo = 0,
                                              int64_t khi = INT64_MAX) {
    __shared__ GemmSmem<BM, BN, BK, CT> sm;
    if (!P.transA) {
        if (!P.transB)
            gemm_f64_tile_t<BM, BN, BK, WM, WN, false, false, CT>(P, t, sm, klo, khi);
        else
            gemm_f64_tile_t<BM, BN, BK, WM, WN, false, true, CT>(P, t, sm, klo, khi);
    } else {
        if (!P.transB)
            gemm_f64_tile_t<BM, BN, BK, WM, WN, true, false, CT>(P, t, sm, klo, khi);
        else
            gemm_f64_tile_t<BM, BN, BK, WM, WN, true, true, CT>(P, t, sm, klo, khi);
    }
}

// Quadrant quad (0..3) of 64 x 64 tile t as a 32 x 32 tile of its own, one
// 16 x 16 block a wave, 32 of K a step.  For launches whose tiles leave compute
// units idle: a wave of the 64 x 64 tile runs 16 MFMAs and a barrier every 16
// of K (0.8 us measured), a wave of the quadrant 8 every 32 (0.65 us).  The
// MFMAs of an output element are the same in the same order, so a launch may
// take either form and gives the same bits.  (A third form that loads the
// MFMA operands from global memory without LDS measured the same up to 64
// tiles and less beyond; a second K tile in flight changed nothing.)
template <int BK, typename CT>
__device__ __forceinline__ void gemm_f64_quad(const syn_gemm_item &P, int64_t t, int quad) {
    __shared__ GemmSmem<32, 32, BK, CT> sm;
    const int64_t row64 = (t / P.tiles_n) * 64, col64 = (t % P.tiles_n) * 64;
    if ((P.tri & 1) && col64 >= row64 + 64) return;
    const int64_t row0 = row64 + 32 * (quad >> 1), col0 = col64 + 32 * (quad & 1);
    if (!P.transA) {
        if (!P.transB)
            gemm_f64_tile_at<32, 32, BK, 16, 16, false, false, CT>(P, row0, col0, sm, 0, INT64_MAX);
        else
            gemm_f64_tile_at<32, 32, BK, 16, 16, false, true, CT>(P, row0, col0, sm, 0, INT64_MAX);
    } else {
        if (!P.transB)
            gemm_f64_tile_at<32, 32, BK, 16, 16, true, false, CT>(P, row0, col0, sm, 0, INT64_MAX);
        else
            gemm_f64_tile_at<32, 32, BK, 16, 16, true, true, CT>(P, row0, col0, sm, 0, INT64_MAX);
    }
}

}  // namespace syn
