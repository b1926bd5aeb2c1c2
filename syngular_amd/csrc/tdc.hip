// Direct phase of the blocked Gram eigen-solver: tridiagonal reduction and
// divide and conquer.
//
// A Gram matrix G is reduced to tridiagonal form T = H^T G H by Householder
// reflectors (Golub & Van Loan 8.3.1, in the panel form of LAPACK's dlatrd),
// T is diagonalised by divide and conquer (Cuppen 1981; deflation, secular
// equation and the recomputed z of Gu & Eisenstat 1995), the eigenvectors of
// T are transformed back to rt = (H Q)^T with compact WY blocks, and G is
// replaced by rt G rt^T, diagonal to rounding.  The Jacobi sweeps that follow
// (tjacobi.hip) start from there: their end-of-sweep test is what accepts the
// result, and a matrix with an entry that still passes it is rotated until
// none does, so the phase changes how many sweeps a call takes (usually none)
// and not what its result satisfies.
//
// Why: a block Jacobi sweep rewrites G and rt in every one of its n / 16
// steps and a call takes 7..14 sweeps, about 4 n^3 flops each; the reduction
// costs 4/3 n^3, the divide and conquer 8/3 n^3 at most and the products
// 6 n^3, once.  Calls measured with the sweeps alone and with this phase, in
// ms: one matrix of order 64 0.78 / 0.33, 128 1.5 / 0.54, 256 3.3 / 1.19, 512
// 7.1 / 2.5, 1024 21 / 6.2, 2048 80 / 17.9; 2000 of order 64 5.3 / 1.6, 1000 of
// 128 15.5 / 2.7, 800 of 256 88 / 10.3, 8 of 512 9.6 / 2.7.
// Residuals fall with the number of rotations: rt^T diag(s^2) rt - G from
// 1e-13 to 1e-15 of the largest eigenvalue.
//
// Buffers of a problem: G's strict upper triangle holds the reflectors (row
// j: v_j from column j + 1; the lower triangle and the diagonal keep G and
// restore it), x (n x n) the reduced matrix and then the merges' eigenvector
// matrices U, y (n x n) the permuted rows of a merge and G rt^T, vec the
// vectors, node records and T factors.
#include "gemm_tile.hpp"
#include "hh_tile.hpp"
#include "prof.hpp"
#include "rotation.hpp"
#include "tdc.hpp"

#include <algorithm>
#include <mutex>

namespace syn {

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v2du __attribute__((ext_vector_type(2), aligned(8)));

// Vector region of a problem (2048 * half >= 64 n doubles, tjacobi.hpp):
// rows of n doubles, then the 32 x 32 T factors of the reflector blocks.
// in Tdc::fail, beside 0 and 1: a work-group waited too long for another; no
// entry of the matrix passes the rotation test
constexpr int kGaveUp = 2, kDiagonal = 3;
struct Tdc {
    int n;
    int64_t ldg, ldr;
    double *g, *rt, *x, *y;
    double *d, *e, *tau;       // tridiagonal form and reflector scales
    double *dd;                // eigenvalues of the current nodes, by row
    double *dl, *zl, *zh;      // poles, z and recomputed z of the undeflated part
    double *tr;                // roots relative to their origin pole
    int *org, *src;            // origin pole of a root; source row of a position
    int *meta, *nrot;          // undeflated count and rotations of a node (at its first row)
    int *rp;                   // row pairs of the rotations
    double *rcs;               // their cosines and sines
    double *rho;               // rank-one weight of a node (at its first row)
    int *fail;                 // not 0: the direct phase does not apply to this matrix
    double *tf;                // T factors
};

__device__ __forceinline__ Tdc tdc_view(const syn_gbj_item &P) {
    Tdc t;
    const int64_t n = P.nv, half = tj_dims<16>(n).half;
    t.n = (int)n;
    t.ldg = P.ldg;
    t.ldr = P.ldr;
    t.g = P.g;
    t.rt = P.rt;
    t.x = P.w + tj_g2_off<16>(half, n);
    t.y = P.w + tj_floor_off<16>(half) + 1;
    double *w = P.w;
    t.d = w;
    t.e = w + n;
    t.tau = w + 2 * n;
    t.dd = w + 3 * n;
    t.dl = w + 4 * n;
    t.zl = w + 5 * n;
    t.zh = w + 6 * n;
    t.tr = w + 7 * n;
    t.org = (int *)(w + 8 * n);
    t.src = t.org + n;
    t.meta = (int *)(w + 9 * n);
    t.nrot = t.meta + n;
    t.rp = (int *)(w + 10 * n);
    t.rcs = w + 11 * n;
    t.rho = w + 13 * n;
    t.fail = (int *)(w + 14 * n);
    t.tf = w + 16 * n;
    return t;
}

// Leaves of the divide and conquer (a power of two, at most kLeaf rows each);
// leaf i starts at row i n / leaves, so sizes differ by one at most.
constexpr int kLeaf = 16;
__host__ __device__ __forceinline__ int tdc_leaves(int64_t n) {
    int l = 1;
    while ((n + l - 1) / l > kLeaf) l *= 2;
    return l;
}
__device__ __forceinline__ int leaf_start(int n, int leaves, int i) { return (int)((int64_t)i * n / leaves); }

// Rows of node t of a level (level 1 merges pairs of leaves); false when the
// problem has no such node or takes no direct phase.
__device__ __forceinline__ bool tdc_node(const Tdc &T, int level, int t, int &lo, int &mid, int &hi) {
    const int L = tdc_leaves(T.n);
    if (t >= (L >> level) || *T.fail) return false;
    lo = leaf_start(T.n, L, t << level);
    mid = leaf_start(T.n, L, (t << level) + (1 << (level - 1)));
    hi = leaf_start(T.n, L, (t + 1) << level);
    return true;
}

__device__ __forceinline__ double rcp_nr(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}

__device__ __forceinline__ double rsq_nr(double x) {
    double y = __builtin_amdgcn_rsq(x);
    y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
    return fma(0.5 * y, fma(-x * y, y, 1.0), y);
}

__device__ __forceinline__ void opaque(int &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ double lane_f64(double v, int lane) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
// sum over the wave, in every lane
__device__ __forceinline__ double all_sum(double v) {
    v = row_sum(v);
    return (lane_f64(v, 0) + lane_f64(v, 16)) + (lane_f64(v, 32) + lane_f64(v, 48));
}

// ---------------------------------------------------------------------------
// Reduction to tridiagonal form T = H^T G H, the matrix in registers.
//
// Step j reflects column j below its diagonal: v (v_j+1 = 1), tau, then
// p = tau A v, w = p - (tau/2 p.v) v and A <- A - v w^T - w v^T.  A pass over
// the registers applies step j - 1's v and w and multiplies the result by
// step j's v at once: column j alone is brought up to date first, from p, v
// and its value before the pass.  So a step is one exchange of p and of the
// next column, a few short vector operations that every wave (one
// work-group) or work-group (several) does for itself, and the pass.
// ---------------------------------------------------------------------------

// Reflector of a column: alpha = its entry at j + 1, xn2 = the squared norm
// below.  H alpha = beta e1 (LAPACK's sign), v = column * scal below j + 1.  A
// column below 1e-145 (the matrix is scaled to order one) counts as zero.
__device__ __forceinline__ void reflector(double alpha, double xn2, double &beta, double &tau, double &scal) {
    beta = alpha;
    tau = scal = 0.0;
    if (xn2 > 1e-290) {
        const double h = fma(alpha, alpha, xn2), r = rsq_nr(h), s = h * r, aa = fabs(alpha);
        beta = -copysign(s, alpha);
        tau = fma(aa, r, 1.0);
        scal = copysign(rcp_nr(aa + s), alpha);
    }
}

// Power-of-two scale that brings a Gram matrix to order one (its largest
// entry is on the diagonal); 0 for a zero, tiny, huge or non-finite diagonal,
// which the Jacobi sweeps take as they did.  Non-finite entries elsewhere end
// in the leaves' iteration limit.
__device__ __forceinline__ double gram_scale(const Tdc &T) {
    double mx = 0.0, bad = 0.0;
    for (int i = threadIdx.x & 63; i < T.n; i += 64) {
        const double v = fabs(T.g[i * T.ldg + i]);
        mx = fmax(mx, v);
        if (!(v <= 1e280)) bad = 1.0;
    }
    for (int off = 32; off > 0; off >>= 1) {
        mx = fmax(mx, __shfl_xor(mx, off, 64));
        bad = fmax(bad, __shfl_xor(bad, off, 64));
    }
    return bad != 0.0 || !(mx > 1e-280) ? 0.0 : ldexp(1.0, -ilogb(mx));
}

// largest of n entries, in every lane of a wave
__device__ __forceinline__ double gram_top(const double *d, int n) {
    double mx = 0.0;
    for (int i = threadIdx.x & 63; i < n; i += 64) mx = fmax(mx, fabs(d[i]));
    for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
    return mx;
}

// Orders up to 16 NB, one work-group of NB waves per matrix.  The matrix is
// symmetric: of its NB x NB tiles of 16 x 16, wave I keeps the diagonal one,
// those an even distance left of it and those an odd distance right of it, so
// each pair of blocks has one tile and 256 rows fit the register file of one
// compute unit.  Blocks die from the first on, and this deal leaves every live
// wave half of the live blocks at any time (the NB / 2 blocks before a wave's
// own, dealt first, kept the last wave at all its tiles for half of the
// steps).  Lane (li, lk) holds rows lk + 4 r and column li of its tiles.  A
// tile adds to the product's rows of block I (summed over the wave's tiles,
// then over li) and, as its transpose, of block J (summed over r, then over lk
// for four tiles at once, then over the waves by wave 0).
//
// A step is wave 0's short vector work and the pass over the tiles by all.
// Wave 0 publishes v and w as soon as it has them, and the others update their
// tiles while it works out the next column and its reflector.  Tiles go four at
// a time without a branch between them, so that their loads overlap, and the
// sums over lanes are taken for four values at once.  Bound by latency and, at
// 16 waves, by LDS reads and vector issue about equally (cycles of a step of
// order 256: 600 for p, 1900 for the reflector beside the update, 2800 for the
// product).  Against tiles one by one, dealt as the NB / 2 blocks before a
// wave's own, and wave 0's work ahead of the whole pass: one matrix of order
// 256 870 -> 663 us, 192 444 -> 382, 128 222 -> 188.  The update on the MFMA
// (one 16 x 16 x 4, half of its contraction zeros) measured 762 and 198 at 256
// and 128 without the wave sums below, two block rows a wave 1020 and 270.
template <int NB>
struct TdTiles {
    static constexpr int KT = NB / 2 + 1, KS = NB / 2, KG = (KT + 2) / 4;
    // block of tile k of wave I: its own, those right of it, then from the
    // nearest on those left of it, so the dead ones are the last (NB, whose
    // entries stay zero: the wave has no such tile)
    static __device__ __forceinline__ int block(int I, int k) {
        const int right = (NB - I) / 2, J = k <= right ? I + 2 * k - 1 : I - 2 * (k - right);
        return k == 0 ? I : J < 0 ? NB : J;
    }
    // tiles of wave I beside its own with a block from jb on
    static __device__ __forceinline__ int live(int I, int jb) { return (NB - I) / 2 + (I - jb) / 2; }
    // place of wave I among those that add to block J
    static __device__ __forceinline__ int slot(int I, int J) {
        return I > J ? (I - J) / 2 - 1 : (NB - 1 - J) / 2 + (J - I - 1) / 2;
    }
};

// Half of a sum over the four rows of 16 lanes, of two values at once: the
// partners of a pair of halves (or of rows) add what both hold of value a in
// the first of them and of value b in the second.
template <bool HALVES>
__device__ __forceinline__ double swap_add(double a, double b) {
    const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
    if constexpr (HALVES) {
        const auto l = __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
        return __builtin_bit_cast(double, (uint64_t)h[0] << 32 | l[0]) +
               __builtin_bit_cast(double, (uint64_t)h[1] << 32 | l[1]);
    } else {
        const auto l = __builtin_amdgcn_permlane16_swap((unsigned)ua, (unsigned)ub, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
        return __builtin_bit_cast(double, (uint64_t)h[0] << 32 | l[0]) +
               __builtin_bit_cast(double, (uint64_t)h[1] << 32 | l[1]);
    }
}

// Sums over the 16 lanes of a row of four values at once, value li / 4 in
// lane li.
__device__ __forceinline__ double row_sum4(double s0, double s1, double s2, double s3) {
    const bool up = (threadIdx.x & 8) != 0, hi = (threadIdx.x & 4) != 0;
    const double a = (up ? s2 : s0) + dpp_f64<0x128>(up ? s0 : s2);   // row_ror:8
    const double b = (up ? s3 : s1) + dpp_f64<0x128>(up ? s1 : s3);
    double y = (hi ? b : a) + dpp_f64<0x141>(hi ? a : b);             // row_half_mirror
    y += dpp_f64<0xb1>(y);                                            // quad_perm:[1,0,3,2]
    return y + dpp_f64<0x4e>(y);                                      // quad_perm:[2,3,0,1]
}

template <int NB>
__global__ __launch_bounds__(64 * NB) void td_reduce_kernel(const syn_gbj_item *__restrict__ items, int nlo, int nhi,
                                                              double tol) {
    typedef TdTiles<NB> Tl;
    constexpr int N = 16 * NB, KT = Tl::KT, KS = Tl::KS, KG = Tl::KG, E = N / 64;
    __shared__ v2d vw[N + 16];                  // v and w of the step before
    __shared__ double us[N + 16], rowp[N], colx[N];
    __shared__ double colp[NB][KS][16];
    if (items[blockIdx.x].nv <= nlo || items[blockIdx.x].nv > nhi) return;
    const Tdc T = tdc_view(items[blockIdx.x]);
    const int n = T.n, tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int I = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: tile indices and their tests too
    const double sc = gram_scale(T);
    if (tid == 0) *T.fail = sc == 0.0;
    if (sc == 0.0) return;
    for (int i = tid; i < N; i += 64 * NB) rowp[i] = i < n ? T.g[i * T.ldg + i] * sc : 0.0;
    double a[KT][4];
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        const int J = Tl::block(I, k);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * I + lk + 4 * r, c = 16 * J + li;
            a[k][r] = (J < NB && i < n && c < n) ? T.g[i * T.ldg + c] * sc : 0.0;
        }
    }
    // nothing to rotate: the matrix stays as it is (below)
    __syncthreads();
    const double floor_abs = __DBL_EPSILON__ * gram_top(rowp, N);
    bool hit = false;
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        const int J = Tl::block(I, k);
        if (J >= NB) continue;
        const double dc = rowp[16 * J + li];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            hit = hit || ((k > 0 || lk + 4 * r != li) && rotates(a[k][r], rowp[16 * I + lk + 4 * r], dc, tol, floor_abs));
    }
    if (!__syncthreads_or(hit)) {
        if (tid == 0) *T.fail = kDiagonal;
        return;
    }
    for (int i = tid; i < N + 16; i += 64 * NB) {
        vw[i] = v2d{0.0, 0.0};
        us[i] = 0.0;
        if (i >= N) continue;
        rowp[i] = 0.0;
        colx[i] = i < n ? T.g[i] * sc : 0.0;
    }
    for (int i = tid; i < NB * KS * 16; i += 64 * NB) (&colp[0][0][0])[i] = 0.0;
    // every entry is in registers before reflectors overwrite the upper triangle
    __syncthreads();
    double tau = 0.0;   // in wave 0: of the previous step
    for (int j = 0; j < n - 1; ++j) {
        double c[E];
        // the lane's coordinates anew in every step: the LDS addresses are an
        // addition each, and kept across steps they would not fit
        int lane = tid & 63, li = lane & 15, lk = lane >> 4;
        opaque(lane);
        opaque(li);
        opaque(lk);
        if (I == 0) {
            // p of step j - 1 (u still its v) and w
            double p[E], u[E], s = 0.0;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = lane + 64 * e, B = i >> 4;
                if (NB > 12) __builtin_amdgcn_sched_barrier(0);   // 1024 threads: loads kept few
                double y = rowp[i];
                if (NB <= 12)
#pragma unroll
                    for (int k = 0; k < KS; ++k) y += colp[B][k][i & 15];
                p[e] = i >= j ? tau * y : 0.0;
                c[e] = colx[i];
                u[e] = us[i];
                s = fma(p[e], u[e], s);
            }
            const double kk = 0.5 * tau * all_sum(s);
#pragma unroll
            for (int e = 0; e < E; ++e) vw[lane + 64 * e] = v2d{u[e], fma(-kk, u[e], p[e])};
        }
        lds_barrier();
        if (I == 0) {
            __builtin_amdgcn_s_setprio(3);   // the others have a pass to hide in
            // column j and its reflector
            const v2d xj = vw[j];
            double xn2 = 0.0;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const v2d x = vw[lane + 64 * e];
                c[e] = fma(-x[1], xj[0], fma(-x[0], xj[1], c[e]));
                if (lane + 64 * e > j + 1) xn2 = fma(c[e], c[e], xn2);
                us[lane + 64 * e] = c[e];   // the column: v is its multiple by scal
            }
            __builtin_amdgcn_wave_barrier();
            const double dj = us[j], alpha = us[j + 1];
            __builtin_amdgcn_wave_barrier();
            xn2 = all_sum(xn2);
            double beta, scal;
            reflector(alpha, xn2, beta, tau, scal);
            if (lane == 0) {
                T.d[j] = dj;
                T.e[j] = j < n - 2 ? beta : alpha;
                T.tau[j] = tau;
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = lane + 64 * e;
                const double x = i <= j ? 0.0 : i == j + 1 ? 1.0 : c[e] * scal;
                us[i] = x;
                if (i > j && i < n) T.g[j * T.ldg + i] = x;
            }
        }
        if (I == 0) __builtin_amdgcn_s_setprio(0);
        if (j == n - 2) break;
        const int jb = (j + 1) >> 4, jl = (j + 1) & 15;
        const bool row_live = 16 * I + 15 > j;
        const int live = Tl::live(I, jb);   // of the tiles beside the own one
        // A <- A - v w^T - w v^T.  Four tiles at a time without a branch between
        // them (dead ones among them meet zeros), so that their loads overlap.
        if (row_live) {
            v2d x[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = vw[16 * I + lk + 4 * r];
            const v2d y0 = vw[16 * I + li];
#pragma unroll
            for (int r = 0; r < 4; ++r) a[0][r] = fma(-x[r][1], y0[0], fma(-x[r][0], y0[1], a[0][r]));
#pragma unroll
            for (int g = 0; g < KG; ++g) {
                if (live <= 4 * g) continue;
#pragma unroll
                for (int h = 0; h < 4; h += 2) {
                    if (NB > 12) __builtin_amdgcn_sched_barrier(0);
                    v2d y[2];
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                        if (1 + 4 * g + h + q < KT) y[q] = vw[16 * Tl::block(I, 1 + 4 * g + h + q) + li];
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const int k = 1 + 4 * g + h + q;
                        if (k >= KT) continue;
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            a[k][r] = fma(-x[r][1], y[q][0], fma(-x[r][0], y[q][1], a[k][r]));
                    }
                }
            }
            // the next column: a tile's column, or the row that is its transpose
            if (I == jb) {
#pragma unroll
                for (int k = 0; k < KT; ++k) {
                    const int J = Tl::block(I, k);
                    if (J >= NB) continue;
                    if (k == 0) {
                        if (li == jl)
#pragma unroll
                            for (int r = 0; r < 4; ++r) colx[16 * I + lk + 4 * r] = a[k][r];
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (lk + 4 * r == jl) colx[16 * J + li] = a[k][r];
                    }
                }
            } else {
#pragma unroll
                for (int k = 1; k < KT; ++k)
                    if (Tl::block(I, k) == jb && li == jl)
#pragma unroll
                        for (int r = 0; r < 4; ++r) colx[16 * I + lk + 4 * r] = a[k][r];
            }
        }
        lds_barrier();
        // y = A u; a wave whose rows have just died clears what it added
        if (row_live || 16 * I + 15 == j) {
            double ui[4], s[4];
            const double u0 = us[16 * I + li];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                ui[r] = us[16 * I + lk + 4 * r];
                s[r] = a[0][r] * u0;
            }
#pragma unroll
            for (int g = 0; g < KG; ++g) {
                if (row_live && live <= 4 * g) continue;   // its blocks need no sums any more
                double sum[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {   // tiles h and h + 2 of the four
                    if (NB > 12) __builtin_amdgcn_sched_barrier(0);
                    double t[2] = {0.0, 0.0}, uj[2];
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                        if (1 + 4 * g + h + 2 * q < KT) uj[q] = us[16 * Tl::block(I, 1 + 4 * g + h + 2 * q) + li];
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const int k = 1 + 4 * g + h + 2 * q < KT ? 1 + 4 * g + h + 2 * q : 0;
                        if (k == 0) continue;
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            s[r] = fma(a[k][r], uj[q], s[r]);
                            t[q] = fma(a[k][r], ui[r], t[q]);
                        }
                    }
                    sum[h] = swap_add<true>(t[0], t[1]);   // lane rows 0, 1: tile h; 2, 3: tile h + 2
                }
                // lane row lk holds the sums of tile 1 + 4 g + lk
                const double y = swap_add<false>(sum[0], sum[1]);
                const int kl = 1 + 4 * g + lk, Jl = Tl::block(I, kl);
                if (kl < KT && Jl < NB) colp[Jl][Tl::slot(I, Jl)][li] = y;
            }
            const double y = row_sum4(s[0], s[1], s[2], s[3]);   // of s[li / 4]
            if ((li & 3) == 0) rowp[16 * I + lk + li] = y;
        }
        lds_barrier();
        // the largest orders: a wave sums its own block's parts, wave 0 would
        // read all of them one block after the other
        if (NB > 12) {
            if (row_live) {
                double y = lk == 0 ? rowp[16 * I + li] : 0.0;
#pragma unroll
                for (int k = 0; k < KS; k += 4) y += colp[I][k + lk][li];
                y = lk_sum(y);
                if (lk == 0) rowp[16 * I + li] = y;
            }
            lds_barrier();
        }
    }
    // the last diagonal entry takes the last step's v and w
    if (I == (n - 1) >> 4 && li == ((n - 1) & 15)) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (16 * I + lk + 4 * r == n - 1) T.d[n - 1] = fma(-2.0 * vw[n - 1][1], vw[n - 1][0], a[0][r]);
    }
}

// Orders up to 64 P, several work-groups per matrix: work-group g of S holds
// columns S (8 q + wave) + g, lane l of a wave rows l + 64 p, so a column's
// sum stays within its wave.  p and the next column travel through global
// memory as the doubles themselves, in words that hold kEmpty until they are
// written (one 64-bit relaxed atomic each): a reader polls the word itself,
// and no fence or flag orders anything.  Three buffers by step: whoever has
// read all of step j knows that all others have read all of step j - 1 (they
// published step j after it), and empties its own words of step j - 1's buffer
// before it publishes step j + 1, so they are empty when anyone polls them for
// step j + 2.  For that every work-group publishes in every step: the last S
// columns, one of each, go on when their rows are dead.
//
// A work-group can wait for one that has no compute unit yet only in its first
// exchange: past it, all of the matrix are running and stay so.  SpinTurn keeps
// other launches of this kernel from holding the units, and a launch's
// work-groups start in order, so the first unfinished matrix always gets its
// units, and that first wait lasts as long as the matrices ahead or another
// stream's kernels do.  Every wait is bounded all the same, that one by kArrive
// polls and the others by kSpin: past the limit the work-group gives up, the
// matrix counts as failed and the Jacobi sweeps take it.  (One limit of kSpin for
// all waits and launches side by side: 3 matrices of order 1500 in a call 50 ms,
// now 24; four streams of such calls at once: 5 of 48 calls gave up, up to 230 ms
// each, now none, up to 81.)
//
// Order 2048 (128 work-groups) is bound by the exchange, 128 readers of every
// word (3.0 of a step's 6.6 us; the vectors 1.5, the pass 0.8), the smaller
// ones by the chain of poll, sums and barriers (order 512: 0.7, 1.0, 0.5 and
// 0.6 to publish).  With halves of doubles beside a step number (twice the
// bytes, four loads an entry, all repeated until the last was there), five
// barriers a step, the pass two rows at a time and the last diagonal entry
// taken from the registers inside the loop (which kept a second copy of the
// matrix alive: 250 bytes of scratch a lane), one matrix of order 300, 512,
// 1024 and 2048 took 1.31, 2.16, 5.5 and 28.1 ms; now 1.01, 1.7, 4.6, 13.5.
constexpr int kMultiThreads = 512;
constexpr int kMultiWaves = kMultiThreads / 64;
constexpr int kSpin = 1 << 14;    // polls of one step
constexpr int kArrive = 1 << 21;  // of the first, a second or so
constexpr unsigned kGroupedMax = 16;
constexpr uint64_t kEmpty = ~(uint64_t)0;   // a NaN no operation makes

// words of the exchange: buffer, vector (p, column), entry; in x, which the
// reduction does not use otherwise
__device__ __forceinline__ uint64_t *xword(const Tdc &T, int buf, int which, int i) {
    return (uint64_t *)T.x + (int64_t)(buf * 2 + which) * T.n + i;
}
__device__ __forceinline__ void put_word(uint64_t *w, uint64_t u) {
    __hip_atomic_store(w, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish(uint64_t *w, double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    put_word(w, u == kEmpty ? u >> 1 : u);   // an input's NaN may look like that
}
__device__ __forceinline__ uint64_t peek(const uint64_t *w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// work-groups of a matrix
template <int Q>
__host__ __device__ __forceinline__ int multi_groups(int64_t n) {
    return (int)((n + kMultiWaves * Q - 1) / (kMultiWaves * Q));
}

__global__ __launch_bounds__(256) void td_clear_kernel(const syn_gbj_item *__restrict__ items, int nlo, int nhi, int fail) {
    // fail: kDiagonal until td_test_kernel finds an entry to rotate
    if (items[blockIdx.x].nv <= nlo || items[blockIdx.x].nv > nhi) return;
    const Tdc T = tdc_view(items[blockIdx.x]);
    for (int i = blockIdx.y * 256 + threadIdx.x; i < 6 * T.n; i += gridDim.y * 256) ((uint64_t *)T.x)[i] = kEmpty;
    if (blockIdx.y == 0 && threadIdx.x == 0) *T.fail = fail;
}

// The rotation test of the sweeps (tj_check_kernel), rows dealt to grid.y.  A
// matrix without an entry to rotate, as at a bond that no gate has touched, is left
// to them as it is: through the whole phase one of order 130 took 538 us and one of
// 300 1463, by the sweeps alone 184 and 338, and with this test 215 and 252.  (The
// reductions in one work-group test their registers, for about a microsecond.)
__global__ __launch_bounds__(256) void td_test_kernel(const syn_gbj_item *__restrict__ items, int nlo, int nhi, double tol) {
    __shared__ double d[kTdcMax];
    if (items[blockIdx.x].nv <= nlo || items[blockIdx.x].nv > nhi) return;
    const Tdc T = tdc_view(items[blockIdx.x]);
    const int n = T.n;
    for (int i = threadIdx.x; i < n; i += 256) d[i] = T.g[i * T.ldg + i];
    __syncthreads();
    const double floor_abs = __DBL_EPSILON__ * gram_top(d, n);
    for (int i = blockIdx.y; i < n; i += gridDim.y) {
        bool hit = false;
        for (int k = threadIdx.x; k < n; k += 256)
            hit = hit || (i != k && rotates_any(T.g[i * T.ldg + k], d[i], d[k], tol, floor_abs));
        if (hit) *T.fail = 0;
        if (__syncthreads_or(hit)) return;
    }
}

template <int P, int Q>
__global__ __launch_bounds__(kMultiThreads) void td_reduce_multi_kernel(const syn_gbj_item *__restrict__ items,
                                                                        int n_items, int nlo, int nhi, int S, int grouped,
                                                                        int arrive, int spin) {
    constexpr int N = 64 * P, NW = kMultiWaves, E = (N + kMultiThreads - 1) / kMultiThreads;
    __shared__ v2d vw[N];                         // v and w of the step before
    __shared__ double us[N], red[NW], red2[NW], sp, sd, sa;
    __shared__ int gone;
    // a matrix's work-groups follow each other in the launch, on one XCD
    // (every eighth work-group) when grouped: those already running never
    // wait for one behind another matrix's
    const int k = grouped ? blockIdx.x >> 3 : blockIdx.x, item = grouped ? k / S * 8 + (blockIdx.x & 7) : k / S;
    const int g = k % S;
    if (item >= n_items || items[item].nv <= nlo || items[item].nv > nhi) return;
    const Tdc T = tdc_view(items[item]);
    const int n = T.n;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tail = n - S;   // the columns that are published to the end
    if (*T.fail == kDiagonal) return;
    const double sc = gram_scale(T);
    if (sc == 0.0) {
        if (g == 0 && tid == 0) *T.fail = 1;
        return;
    }
    double a[P][Q];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int i = lane + 64 * p, c = S * (NW * q + wv) + g;
            a[p][q] = (i < n && c < n) ? T.g[c * T.ldg + i] * sc : 0.0;
        }
    double v[E], c[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = 0.0;
    double tau = 0.0;
    if (tid == 0) gone = 0;
    for (int i = tid; i < N; i += kMultiThreads) us[i] = 0.0;
    lds_barrier();
    int buf = 0;
    for (int j = 0; j < n - 1; ++j, buf = buf == 2 ? 0 : buf + 1) {
        const int next = buf == 2 ? 0 : buf + 1, before = buf == 0 ? 2 : buf - 1;   // steps j + 1, j - 1
        // the thread's place anew in every step: addresses kept across steps
        // would not fit
        int me = tid;
        opaque(me);
        // p of step j - 1 and column j before it (entries from j on)
        double p[E], s = 0.0;
        bool ok = true;
        if (j == 0) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = me + kMultiThreads * e;
                p[e] = 0.0;
                c[e] = i < n ? T.g[i * T.ldg] * sc : 0.0;   // row 0's owner may be past this step
            }
        } else {
            // every entry that is not there is asked for again, together
            uint64_t wp[E], wc[E];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = me + kMultiThreads * e;
                wp[e] = i < n && (i >= j || i >= tail) ? kEmpty : 0;
                wc[e] = i < n && i >= j ? kEmpty : 0;
            }
            // the first time once they are all there: a loop of its own
            for (int left = j == 1 ? arrive : 0; left > 0; --left) {
                bool there = true;
                for (int i = me ? me : kMultiThreads; i < n; i += kMultiThreads)   // nothing comes for row 0
                    there = there && peek(xword(T, buf, 0, i)) != kEmpty && peek(xword(T, buf, 1, i)) != kEmpty;
                if (there) break;
                __builtin_amdgcn_s_sleep(8);
            }
            for (int left = spin;;) {
                ok = true;
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int i = me + kMultiThreads * e;
                    if (wp[e] == kEmpty) wp[e] = peek(xword(T, buf, 0, i));
                    if (wc[e] == kEmpty) wc[e] = peek(xword(T, buf, 1, i));
                }
#pragma unroll
                for (int e = 0; e < E; ++e) ok = ok && wp[e] != kEmpty && wc[e] != kEmpty;
                if (ok || --left <= 0) break;
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                p[e] = me + kMultiThreads * e >= j ? __builtin_bit_cast(double, wp[e]) : 0.0;
                c[e] = __builtin_bit_cast(double, wc[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            s = fma(p[e], v[e], s);
            if (me + kMultiThreads * e == j) sp = p[e];
        }
        if (!ok) gone = 1;
        s = all_sum(s);
        if (lane == 0) red[wv] = s;
        lds_barrier();
        if (gone) {
            if (tid == 0) *T.fail = kGaveUp;
            return;
        }
        // all have read step j - 1's words: the wave's own are empty again
        if (lane < Q) {
            const int cc = S * (NW * lane + wv) + g;
            if (cc < n) {
                put_word(xword(T, before, 0, cc), kEmpty);
                put_word(xword(T, before, 1, cc), kEmpty);
            }
        }
        double kk = 0.0;
#pragma unroll
        for (int q = 0; q < NW; ++q) kk += red[q];
        kk *= 0.5 * tau;
        const double vj = us[j], wj = fma(-kk, vj, sp);   // us: still step j - 1's v
        double xn2 = 0.0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = me + kMultiThreads * e;
            const double w = fma(-kk, v[e], p[e]);
            c[e] = fma(-w, vj, fma(-v[e], wj, c[e]));
            if (i > j + 1) xn2 = fma(c[e], c[e], xn2);
            if (i < N) vw[i] = v2d{v[e], w};
            if (i == j) sd = c[e];
            if (i == j + 1) sa = c[e];
        }
        xn2 = all_sum(xn2);
        if (lane == 0) red2[wv] = xn2;
        lds_barrier();
        xn2 = 0.0;
#pragma unroll
        for (int q = 0; q < NW; ++q) xn2 += red2[q];
        const double alpha = sa;
        double beta, scal;
        reflector(alpha, xn2, beta, tau, scal);
        if (tid == 0 && g == 0) {
            T.d[j] = sd;
            T.e[j] = j < n - 2 ? beta : alpha;
            T.tau[j] = tau;
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = me + kMultiThreads * e;
            v[e] = i <= j ? 0.0 : i == j + 1 ? 1.0 : c[e] * scal;
            if (i < N) us[i] = v[e];
            // row j of the upper triangle was read by its owner alone
            if (j % S == g && i > j && i < n) T.g[j * T.ldg + i] = v[e];
        }
        lds_barrier();
        // 64s of rows loaded together (order 512: 1.34 ms one by one, 1.42 by
        // four; 2048: 14.6 and 13.5)
        constexpr int G = P > 8 ? 4 : 1;
        double y[Q];
        v2d x[Q];
        const int lane = me & 63;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int cc = S * (NW * q + wv) + g;
            y[q] = 0.0;
            x[q] = cc < n ? vw[cc] : v2d{0.0, 0.0};
        }
#pragma unroll
        for (int p0 = 0; p0 < P; p0 += G) {
            if (P > 8) __builtin_amdgcn_sched_barrier(0);   // row loads not all in flight at once
            if (64 * (p0 + G) <= j + 1) continue;
            v2d r[G];
            double u[G];
#pragma unroll
            for (int h = 0; h < G; ++h) {
                r[h] = vw[lane + 64 * (p0 + h)];
                u[h] = us[lane + 64 * (p0 + h)];
            }
#pragma unroll
            for (int h = 0; h < G; ++h)
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    a[p0 + h][q] = fma(-r[h][1], x[q][0], fma(-r[h][0], x[q][1], a[p0 + h][q]));
                    y[q] = fma(a[p0 + h][q], u[h], y[q]);
                }
        }
        // the words emptied above are there before anything of step j + 1 is
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint64_t *xcol = xword(T, next, 1, lane);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            if (S * (NW * q + wv) + g != j + 1) continue;
#pragma unroll
            for (int p2 = 0; p2 < P; ++p2)
                if (lane + 64 * p2 > j && lane + 64 * p2 < n) publish(xcol + 64 * p2, a[p2][q]);
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int cc = S * (NW * q + wv) + g;
            const double t = tau * all_sum(y[q]);
            if (lane == 0 && (cc > j || cc >= tail) && cc < n) publish(xword(T, next, 0, cc), t);
        }
    }
    // the last diagonal entry is the column that step n - 1 would take (its v
    // and w are zero)
    if (g == 0 && tid == 0) {
        uint64_t u = kEmpty;
        for (int left = spin; u == kEmpty && left > 0; --left) u = peek(xword(T, buf, 1, n - 1));
        T.d[n - 1] = __builtin_bit_cast(double, u);
        if (u == kEmpty) *T.fail = kGaveUp;
    }
}

// ---------------------------------------------------------------------------
// Leaves: implicit QL (Golub & Van Loan 8.3.3) of the tridiagonal block of at
// most kLeaf rows, one wave each; the eigenvectors leave as the rows of rt,
// eigenvalues ascending.  The rotations form one serial chain of about 200
// for 16 rows: the diagonals live in two registers, entry i in lane i of each
// row of lanes, read and written by lane number, so a link is its dozen
// dependent operations and one reciprocal square root (with the diagonals in
// LDS, a round trip each, the leaf took 120 us); lane c carries component c
// of the vector the chain is at, the others are in LDS off the chain.  The
// split points' rank-one terms are subtracted here: node boundaries take |e|
// off the diagonal on both sides.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void set_entry(double &v, int i, double x) {
    if ((int)(threadIdx.x & 15) == i) v = x;
}

__global__ __launch_bounds__(64) void td_leaf_kernel(const syn_gbj_item *__restrict__ items) {
    __shared__ double q[kLeaf][64];
    const Tdc T = tdc_view(items[blockIdx.x]);
    const int L = tdc_leaves(T.n), t = blockIdx.y, c = threadIdx.x, i = c & 15;
    if (t >= L || *T.fail) return;
    const int lo = leaf_start(T.n, L, t), hi = leaf_start(T.n, L, t + 1), m = hi - lo;
    double dv = i < m ? T.d[lo + i] : 0.0, ev = i + 1 < m ? T.e[lo + i] : 0.0;
    if (lo > 0 && i == 0) dv -= fabs(T.e[lo - 1]);
    if (hi < T.n && i == m - 1) dv -= fabs(T.e[hi - 1]);
    for (int k = 0; k < kLeaf; ++k) q[k][c] = k == c ? 1.0 : 0.0;
    bool ok = true;
    for (int l = 0; l < m && ok; ++l) {
        for (int it = 0;; ++it) {
            // the first negligible off-diagonal entry from l on (the last
            // entry is zero, so there is one)
            const double dn = dpp_f64<0x101>(dv);   // row_shl:1, the next entry
            const bool small = fabs(ev) <= 1.2e-16 * (fabs(dv) + fabs(dn)) + 1e-22 || i >= m - 1;
            const int mm = __builtin_ctz((unsigned)(__ballot(small) & 0xffffu) >> l << l);
            if (mm == l) break;
            if (it == 60) {
                ok = false;
                break;
            }
            const double dl = lane_f64(dv, l), el = lane_f64(ev, l);
            double g = (lane_f64(dv, l + 1) - dl) / (2.0 * el);
            const double r0 = sqrt(fma(g, g, 1.0));
            double dnext = lane_f64(dv, mm);
            g = dnext - dl + el / (g + copysign(r0, g));
            double s = 1.0, co = 1.0, p = 0.0, z1 = q[mm][c];
            int k = mm - 1;
            for (; k >= l; --k) {
                const double ek = lane_f64(ev, k), dk = lane_f64(dv, k), z0 = q[k][c];
                const double f = s * ek, b = co * ek, r2 = fma(f, f, g * g);
                if (!(r2 > 1e-290)) break;   // both vanish: the block splits here
                const double ir = rsq_nr(r2);
                set_entry(ev, k + 1, r2 * ir);
                s = f * ir;
                co = g * ir;
                g = dnext - p;
                const double r = fma(dk - g, s, 2.0 * co * b);
                p = s * r;
                set_entry(dv, k + 1, g + p);
                g = fma(co, r, -b);
                q[k + 1][c] = fma(s, z0, co * z1);
                z1 = fma(co, z0, -s * z1);
                dnext = dk;
            }
            // the entry the chain stopped at: l, or where it split
            q[k + 1][c] = z1;
            set_entry(dv, k + 1, dnext - p);
            set_entry(ev, k + 1, k >= l ? 0.0 : g);
            set_entry(ev, mm, 0.0);
        }
    }
    if (!ok && c == 0) *T.fail = 1;
    // ascending order, ties by index
    int rk = 0;
    for (int k = 0; k < m; ++k) {
        const double o = lane_f64(dv, k);
        rk += o < dv || (o == dv && k < i);
    }
    for (int k = 0; k < m; ++k) {
        const int r = __builtin_amdgcn_readlane(rk, k);
        if (c < m) T.rt[(int64_t)(lo + r) * T.ldr + lo + c] = q[k][c];
    }
    if (c < m) T.dd[lo + rk] = dv;
    if (c == 0) T.meta[lo] = m;
}

// ---------------------------------------------------------------------------
// Merge of two solved halves: D + rho z z^T with z the last row of the first
// half's Q and the first row of the second's.  This kernel orders the poles
// (each half brings its roots and its deflated values, two ascending lists
// each), deflates (a negligible z entry, or two poles whose rotation would
// leave a negligible off-diagonal entry), and writes the row order, the
// rotations, the undeflated poles and z.
// ---------------------------------------------------------------------------
constexpr int kPrepThreads = 256;
__host__ __device__ constexpr int64_t prep_lds(int64_t k) { return 2 * k + 3 * ((k + 1) / 2) + 16; }   // doubles

__device__ __forceinline__ int lower_count(const double *a, int lo, int hi, double v, bool with_equal) {
    const int base = lo;
    while (lo < hi) {
        const int m = (lo + hi) >> 1;
        if (a[m] < v || (with_equal && a[m] == v))
            lo = m + 1;
        else
            hi = m;
    }
    return lo - base;
}

__global__ __launch_bounds__(kPrepThreads) void td_prep_kernel(const syn_gbj_item *__restrict__ items, int level) {
    extern __shared__ double sm[];
    __shared__ double red[2][kPrepThreads / 64];
    __shared__ int scan[kPrepThreads], sh[4];
    const Tdc T = tdc_view(items[blockIdx.x]);
    int lo, mid, hi;
    if (!tdc_node(T, level, blockIdx.y, lo, mid, hi)) return;
    const int k = hi - lo, n1 = mid - lo, tid = threadIdx.x;
    double *ds = sm, *zs = sm + k;
    int *sidx = (int *)(zs + k), *nt = sidx + k, *dfl = nt + k;   // 3 k ints
    const int K1 = T.meta[lo], K2 = T.meta[mid];
    const double e = T.e[mid - 1], rho = 2.0 * fabs(e);
    const int b[5] = {0, K1, n1, n1 + K2, k};
    for (int i = tid; i < k; i += kPrepThreads) zs[i] = T.dd[lo + i];
    __syncthreads();
    double zmax = 0.0, dmax = 0.0;
    // ranks among the four lists (their values staged in zs)
    for (int i = tid; i < k; i += kPrepThreads) {
        const double v = zs[i];
        const int own = i < b[1] ? 0 : i < b[2] ? 1 : i < b[3] ? 2 : 3;
        int rk = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) rk += q == own ? i - b[q] : lower_count(zs, b[q], b[q + 1], v, q < own);
        ds[rk] = v;
        sidx[rk] = i;
        dmax = fmax(dmax, fabs(v));
    }
    __syncthreads();
    for (int i = tid; i < k; i += kPrepThreads) {
        const int r = sidx[i];
        const double z = r < n1 ? T.rt[(int64_t)(lo + r) * T.ldr + mid - 1]
                                : copysign(1.0, e) * T.rt[(int64_t)(lo + r) * T.ldr + mid];
        zs[i] = z * 0.70710678118654752440;
        zmax = fmax(zmax, fabs(zs[i]));
    }
    for (int off = 32; off > 0; off >>= 1) {
        zmax = fmax(zmax, __shfl_xor(zmax, off, 64));
        dmax = fmax(dmax, __shfl_xor(dmax, off, 64));
    }
    if ((tid & 63) == 0) {
        red[0][tid >> 6] = zmax;
        red[1][tid >> 6] = dmax;
    }
    if (tid < 4) sh[tid] = 0;
    __syncthreads();
    for (int q = 0; q < kPrepThreads / 64; ++q) {
        zmax = fmax(zmax, red[0][q]);
        dmax = fmax(dmax, red[1][q]);
    }
    const double tol = 8.0 * 1.1102230246251565e-16 * fmax(dmax, zmax);
    // the entries that stay, in order (nt), and the negligible ones (dfl)
    const int per = (k + kPrepThreads - 1) / kPrepThreads, i0 = tid * per, i1 = i0 + per < k ? i0 + per : k;
    int cnt = 0;
    for (int i = i0; i < i1; ++i) cnt += rho * fabs(zs[i]) > tol;
    scan[tid] = cnt;
    __syncthreads();
    for (int off = 1; off < kPrepThreads; off <<= 1) {
        const int a = tid >= off ? scan[tid - off] : 0;
        __syncthreads();
        scan[tid] += a;
        __syncthreads();
    }
    const int n_nt = scan[kPrepThreads - 1];
    int at = scan[tid] - cnt;
    for (int i = i0; i < i1; ++i) {
        if (rho * fabs(zs[i]) > tol)
            nt[at++] = i;
        else
            dfl[i - at] = i;
    }
    __syncthreads();
    // two neighbouring poles so close that a rotation deflates one of them
    for (int q = tid; q + 1 < n_nt; q += kPrepThreads) {
        const double s = zs[nt[q]], c = zs[nt[q + 1]], t = ds[nt[q + 1]] - ds[nt[q]];
        if (fabs(t * c * s) <= tol * fma(c, c, s * s)) sh[0] = 1;
    }
    __syncthreads();
    if (tid == 0) {
        int K = n_nt, nr = 0, nd = k - n_nt;
        if (sh[0]) {
            K = 0;
            int pj = nt[0];
            for (int q = 1; q < n_nt; ++q) {
                const int j = nt[q];
                const double s0 = zs[pj], c0 = zs[j], t = ds[j] - ds[pj], h2 = fma(c0, c0, s0 * s0);
                if (fabs(t * c0 * s0) <= tol * h2) {
                    const double ih = 1.0 / sqrt(h2), c = c0 * ih, s = -s0 * ih;
                    zs[j] = h2 * ih;
                    zs[pj] = 0.0;
                    const double dp = ds[pj], dj = ds[j];
                    ds[j] = fma(dp * s, s, dj * c * c);
                    ds[pj] = fma(dp * c, c, dj * s * s);
                    T.rp[2 * (lo + nr)] = pj;
                    T.rp[2 * (lo + nr) + 1] = j;
                    T.rcs[2 * (lo + nr)] = c;
                    T.rcs[2 * (lo + nr) + 1] = s;
                    ++nr;
                    dfl[nd++] = pj;
                } else {
                    nt[K++] = pj;   // K <= q: behind the entries still to come
                }
                pj = j;
            }
            nt[K++] = pj;
        }
        sh[1] = K;
        sh[2] = nr;
    }
    __syncthreads();
    const int K = sh[1], nr = sh[2], nd = k - K;
    // positions: undeflated first, then the deflated ones ascending
    for (int q = tid; q < K; q += kPrepThreads) {
        T.dl[lo + q] = ds[nt[q]];
        T.zl[lo + q] = zs[nt[q]];
        T.src[lo + q] = sidx[nt[q]];
    }
    for (int q = tid; q < nd; q += kPrepThreads) {
        const double v = ds[dfl[q]];
        int rk = 0;
        for (int u = 0; u < nd; ++u) {
            const double o = ds[dfl[u]];
            rk += o < v || (o == v && u < q);
        }
        T.dd[lo + K + rk] = v;
        T.src[lo + K + rk] = sidx[dfl[q]];
    }
    __syncthreads();
    // the rotations act on source rows
    for (int q = tid; q < nr; q += kPrepThreads) {
        T.rp[2 * (lo + q)] = sidx[T.rp[2 * (lo + q)]];
        T.rp[2 * (lo + q) + 1] = sidx[T.rp[2 * (lo + q) + 1]];
    }
    if (tid == 0) {
        T.meta[lo] = K;
        T.nrot[lo] = nr;
        T.rho[lo] = rho;
    }
}

// Rows of a node into their merge order (rt -> y, the half a row does not
// reach zero), after the deflating rotations.  A work-group takes 64 columns
// of the node: the rotations act on rows, so its columns are its own.
__global__ __launch_bounds__(256) void td_copy_kernel(const syn_gbj_item *__restrict__ items, int level) {
    const Tdc T = tdc_view(items[blockIdx.x]);
    int lo, mid, hi;
    if (!tdc_node(T, level, blockIdx.z, lo, mid, hi)) return;
    const int k = hi - lo, n = T.n, c = blockIdx.y * 64 + (threadIdx.x & 63), rg = threadIdx.x >> 6;
    const int nr = T.nrot[lo];
    if ((int)blockIdx.y * 64 >= k) return;
    double *rt = T.rt + (int64_t)lo * T.ldr + lo;
    if (nr) {
        // the halves' zero blocks become rows that the rotations fill
        if (c < k)
            for (int i = rg; i < k; i += 4)
                if ((i < mid - lo) != (c < mid - lo)) rt[i * T.ldr + c] = 0.0;
        __syncthreads();
        if (rg == 0 && c < k) {
            for (int q = 0; q < nr; ++q) {
                double *p = rt + T.rp[2 * (lo + q)] * T.ldr + c, *r = rt + T.rp[2 * (lo + q) + 1] * T.ldr + c;
                const double co = T.rcs[2 * (lo + q)], s = T.rcs[2 * (lo + q) + 1], xv = *p, yv = *r;
                *p = fma(co, xv, s * yv);
                *r = fma(co, yv, -s * xv);
            }
        }
        __syncthreads();
    }
    if (c >= k) return;
    double *y = T.y + (int64_t)lo * n + lo;
    for (int i = rg; i < k; i += 4) {
        const int s = T.src[lo + i];
        const bool in = nr || (s < mid - lo) == (c < mid - lo);
        y[(int64_t)i * n + c] = in ? rt[s * T.ldr + c] : 0.0;
    }
}

// ---------------------------------------------------------------------------
// Secular equation 1 + sum_i a_i / (d_i - lambda) = 0, a_i = rho z_i^2, four
// lanes per root, poles in LDS.  A root is kept as its distance tau to the
// nearer pole (its origin), so d_i - lambda = (d_i - d_origin) - tau has no
// cancellation.  Iteration: the rational interpolation through the two poles
// around the root (Li 1993, the middle way), safeguarded by a bracket that
// every evaluation shrinks; it stops at the rounding level of the sum or of
// the bracket.
// ---------------------------------------------------------------------------
constexpr int kSecThreads = 256;
constexpr int kSecRoots = kSecThreads / 4;   // roots of a work-group

// Four lanes (lk) share a root and take every fourth term each; j0 is the
// first root of the wave's 16, so the terms before it are left of every root
// of the wave and those from j0 + 16 on right of it, and only the 16 between
// need a selection.
__device__ __forceinline__ void secular_sums(const double *dl, const double *a, int K, int j0, int j, int lk,
                                             double dorg, double tau, double &psi, double &dpsi, double &phi,
                                             double &dphi) {
    psi = dpsi = phi = dphi = 0.0;
    int i = lk;
#pragma unroll 2
    for (; i < j0; i += 4) {
        const double r = rcp_nr((dl[i] - dorg) - tau), t = a[i] * r;
        psi += t;
        dpsi = fma(t, r, dpsi);
    }
    const int mid = j0 + 16 < K ? j0 + 16 : K;
    for (; i < mid; i += 4) {
        const double r = rcp_nr((dl[i] - dorg) - tau), t = a[i] * r, tt = t * r;
        const bool left = i <= j;
        psi += left ? t : 0.0;
        dpsi += left ? tt : 0.0;
        phi += left ? 0.0 : t;
        dphi += left ? 0.0 : tt;
    }
#pragma unroll 2
    for (; i < K; i += 4) {
        const double r = rcp_nr((dl[i] - dorg) - tau), t = a[i] * r;
        phi += t;
        dphi = fma(t, r, dphi);
    }
    psi = lk_sum(psi);
    dpsi = lk_sum(dpsi);
    phi = lk_sum(phi);
    dphi = lk_sum(dphi);
}

__device__ __forceinline__ bool secular_root(const double *dl, const double *a, int K, int j0, int j, int lk,
                                             double asum, int &org, double &tau) {
    org = j;
    if (K == 1) {
        tau = a[0];
        return true;
    }
    const bool last = j == K - 1;
    const int jl = last ? K - 2 : j, jr = jl + 1;   // the poles of the interpolation
    double lo, hi, psi, dpsi, phi, dphi;
    if (last) {
        lo = 0.0;
        hi = asum;
        tau = 0.5 * hi;
    } else {
        const double gap = dl[j + 1] - dl[j], mid = 0.5 * gap;
        secular_sums(dl, a, K, j0, jl, lk, dl[j], mid, psi, dpsi, phi, dphi);
        const double f = 1.0 + psi + phi, aj = a[j], ar = a[j + 1];
        // the two poles' model with the other terms at their midpoint value
        const double c = f + (aj - ar) / mid;
        if (f >= 0.0) {
            lo = 0.0;
            hi = mid;
            const double b = fma(c, gap, aj + ar), q = aj * gap, ds = sqrt(fmax(fma(b, b, -4.0 * c * q), 0.0));
            tau = b > 0.0 ? 2.0 * q / (b + ds) : (b - ds) / (2.0 * c);
        } else {
            org = j + 1;
            lo = -mid;
            hi = 0.0;
            const double b = fma(-c, gap, aj + ar), q = ar * gap, ds = sqrt(fmax(fma(b, b, 4.0 * c * q), 0.0));
            tau = b > 0.0 ? -2.0 * q / (b + ds) : (b - ds) / (2.0 * c);
        }
        if (!(tau > lo && tau < hi)) tau = 0.5 * (lo + hi);
    }
    const double dorg = dl[org], eps = 1.1102230246251565e-16;
    for (int it = 0; it < 200; ++it) {
        secular_sums(dl, a, K, j0, jl, lk, dorg, tau, psi, dpsi, phi, dphi);
        const double f = 1.0 + psi + phi;
        if (fabs(f) <= eps * (8.0 * (fabs(psi) + fabs(phi)) + 2.0 + fabs(tau) * (dpsi + dphi))) return true;
        if (f < 0.0)
            lo = tau;
        else
            hi = tau;
        if (hi - lo <= 2.0 * eps * fmax(fabs(lo), fabs(hi))) return true;
        const double d1 = (dl[jl] - dorg) - tau, d2 = (dl[jr] - dorg) - tau;
        const double c = f - d1 * dpsi - d2 * dphi, am = (d1 + d2) * f - d1 * d2 * (dpsi + dphi), b = d1 * d2 * f;
        const double ds = sqrt(fmax(fma(am, am, -4.0 * b * c), 0.0));
        double eta;
        if (last)
            eta = am >= 0.0 ? (am + ds) / (2.0 * c) : 2.0 * b / (am - ds);
        else
            eta = am <= 0.0 ? (am - ds) / (2.0 * c) : 2.0 * b / (am + ds);
        if (!(f * eta < 0.0)) eta = -f / (dpsi + dphi);
        double nx = tau + eta;
        if (!(nx > lo && nx < hi) || (it > 12 && (it & 1)))
            nx = lo == 0.0 ? 0.0625 * hi : hi == 0.0 ? 0.0625 * lo : 0.5 * (lo + hi);
        if (nx == tau) return true;
        tau = nx;
    }
    return false;
}

__global__ __launch_bounds__(kSecThreads) void td_secular_kernel(const syn_gbj_item *__restrict__ items, int level) {
    extern __shared__ double sm[];
    const Tdc T = tdc_view(items[blockIdx.x]);
    int lo, mid, hi;
    if (!tdc_node(T, level, blockIdx.z, lo, mid, hi)) return;
    const int K = T.meta[lo], tid = threadIdx.x, lane = tid & 63;
    if ((int)blockIdx.y * kSecRoots >= K) return;
    double *dl = sm, *a = sm + K;
    const double rho = T.rho[lo];
    for (int i = tid; i < K; i += kSecThreads) {
        dl[i] = T.dl[lo + i];
        const double z = T.zl[lo + i];
        a[i] = rho * z * z;
    }
    __syncthreads();
    const int j0 = blockIdx.y * kSecRoots + 16 * (tid >> 6), li = lane & 15, lk = lane >> 4;
    if (j0 >= K) return;
    double asum = 0.0;
    for (int i = lane; i < K; i += 64) asum += a[i];
    asum = all_sum(asum);
    const int j = j0 + li < K ? j0 + li : K - 1;   // lanes past the last root repeat it
    int org;
    double tau;
    const bool ok = secular_root(dl, a, K, j0, j, lk, asum * (1.0 + 1e-15), org, tau);
    if (!ok) *T.fail = 1;
    if (lk == 0 && j0 + li < K) {
        T.org[lo + j] = org;
        T.tr[lo + j] = tau;
        T.dd[lo + j] = dl[org] + tau;
    }
}

// z recomputed from the roots (the z whose secular equation has exactly
// these roots), one thread per entry: z_i^2 = prod_j (lambda_j - d_i) over
// prod_{j != i} (d_j - d_i), up to a constant factor.
constexpr int kZhatThreads = 64;
__global__ __launch_bounds__(kZhatThreads) void td_zhat_kernel(const syn_gbj_item *__restrict__ items, int level) {
    extern __shared__ double sm[];
    const Tdc T = tdc_view(items[blockIdx.x]);
    int lo, mid, hi;
    if (!tdc_node(T, level, blockIdx.z, lo, mid, hi)) return;
    const int K = T.meta[lo], tid = threadIdx.x, i = blockIdx.y * kZhatThreads + tid;
    if ((int)blockIdx.y * kZhatThreads >= K) return;
    double *dl = sm, *od = sm + K, *tr = od + K;
    for (int q = tid; q < K; q += kZhatThreads) {
        dl[q] = T.dl[lo + q];
        od[q] = T.dl[lo + T.org[lo + q]];
        tr[q] = T.tr[lo + q];
    }
    __syncthreads();
    if (i >= K) return;
    const double di = dl[i];
    double prod = (od[i] - di) + tr[i];
    for (int j = 0; j < K; ++j)
        if (j != i) prod *= ((od[j] - di) + tr[j]) * rcp_nr(dl[j] - di);
    T.zh[lo + i] = copysign(sqrt(fabs(prod)), T.zl[lo + i]);
}

// Rows of U^T (eigenvectors of D + rho z z^T, unit norm) into x, a wave per
// root; the deflated rows go back from y to rt as they are.
__global__ __launch_bounds__(256) void td_vec_kernel(const syn_gbj_item *__restrict__ items, int level) {
    const Tdc T = tdc_view(items[blockIdx.x]);
    int lo, mid, hi;
    if (!tdc_node(T, level, blockIdx.z, lo, mid, hi)) return;
    const int K = T.meta[lo], k = hi - lo, n = T.n, lane = threadIdx.x & 63;
    const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (j >= k) return;
    if (j >= K) {
        const double *y = T.y + (int64_t)(lo + j) * n + lo;
        double *r = T.rt + (int64_t)(lo + j) * T.ldr + lo;
        for (int c = lane; c < k; c += 64) r[c] = y[c];
        return;
    }
    const double od = T.dl[lo + T.org[lo + j]], tr = T.tr[lo + j];
    double s = 0.0;
    for (int i = lane; i < K; i += 64) {
        const double u = T.zh[lo + i] * rcp_nr((T.dl[lo + i] - od) - tr);
        s = fma(u, u, s);
    }
    s = rsq_nr(wave_sum(s));
    double *x = T.x + (int64_t)(lo + j) * n + lo;
    for (int i = lane; i < K; i += 64) x[i] = T.zh[lo + i] * rcp_nr((T.dl[lo + i] - od) - tr) * s;
}

// ---------------------------------------------------------------------------
// Products on the 64 x 64 MFMA tile: the merge's rt = U^T y (what 0), and
// with the back-transformed rt: y = G rt^T (1), G = rt y (2).  blockIdx.y
// is the tile, blockIdx.z the node.
// ---------------------------------------------------------------------------
template <bool QUAD>
__global__ __launch_bounds__(256, 2) void td_gemm_kernel(const syn_gbj_item *__restrict__ items, int what,
                                                         int level) {
    const Tdc T = tdc_view(items[blockIdx.x]);
    const int n = T.n;
    syn_gemm_item P;
    P.alpha = 1.0;
    P.beta = 0.0;
    P.transA = P.transB = 0;
    P.tri = 0;
    P.block_start = 0;
    if (what == 0) {
        int lo, mid, hi;
        if (!tdc_node(T, level, blockIdx.z, lo, mid, hi)) return;
        const int K = T.meta[lo];
        P.A = T.x + (int64_t)lo * n + lo;
        P.B = T.y + (int64_t)lo * n + lo;
        P.C = T.rt + (int64_t)lo * T.ldr + lo;
        P.lda = P.ldb = n;
        P.ldc = T.ldr;
        P.m = P.k = K;
        P.n = hi - lo;
    } else {
        if (*T.fail) return;
        P.m = P.n = P.k = n;
        if (what == 1) {
            P.A = T.g;
            P.lda = T.ldg;
            P.B = T.rt;
            P.ldb = T.ldr;
            P.transB = 1;
            P.C = T.y;
            P.ldc = n;
        } else {
            P.A = T.rt;
            P.lda = T.ldr;
            P.B = T.y;
            P.ldb = n;
            P.C = T.g;
            P.ldc = T.ldg;
        }
    }
    P.tiles_n = (P.n + 63) / 64;
    const unsigned tile = QUAD ? blockIdx.y >> 2 : blockIdx.y;
    if (tile >= P.tiles_n * ((P.m + 63) / 64)) return;
    if constexpr (QUAD) {
        gemm_f64_quad<32, double>(P, tile, blockIdx.y & 3);
        return;
    }
    __shared__ GemmSmem<64, 64, 16, double> smem;
    if (what == 1)
        gemm_f64_tile_t<64, 64, 16, 32, 32, false, true, double>(P, tile, smem, 0, INT64_MAX);
    else
        gemm_f64_tile_t<64, 64, 16, 32, 32, false, false, double>(P, tile, smem, 0, INT64_MAX);
}

// ---------------------------------------------------------------------------
// Back-transformation rt <- rt (I - V T^T V^T) block by block from the last:
// the T factor of each block of 32 reflectors (LAPACK dlarft, forward,
// columnwise; V V^T on the MFMA, a row of T per lane: order 256 49 -> 14 us),
// then work-groups of 16 or 32 rows of rt walk the blocks.
// ---------------------------------------------------------------------------
constexpr int kBlk = 32;
__host__ __device__ __forceinline__ int refl_blocks(int n) { return (n - 2 + kBlk - 1) / kBlk; }

__global__ __launch_bounds__(256) void td_tfac_kernel(const syn_gbj_item *__restrict__ items) {
    __shared__ double Sp[4][3][256], S[3][16][17];
    const Tdc T = tdc_view(items[blockIdx.x]);
    const int n = T.n, j0 = blockIdx.y * kBlk, nb = n - 2 - j0 < kBlk ? n - 2 - j0 : kBlk, tid = threadIdx.x;
    if (nb <= 0 || *T.fail) return;
    const int wv = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    // S = V V^T, upper tiles, on the MFMA: lane lk takes four consecutive
    // columns of each 16, the same in both operands
    v4d s00 = {0.0, 0.0, 0.0, 0.0}, s01 = s00, s11 = s00;
    for (int k0 = j0 + 1 + 16 * wv; k0 < n; k0 += 64) {
        const int k = k0 + 4 * lk;
        double v[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int ref = 16 * i + li;
            const double *vp = T.g + (int64_t)(j0 + ref) * T.ldg + k;
            if (nb == kBlk && k0 >= j0 + kBlk && k0 + 16 <= n) {   // right of the block's triangle
                const v2du v0 = *(const v2du *)vp, v1 = *(const v2du *)(vp + 2);
                v[i][0] = v0.x, v[i][1] = v0.y, v[i][2] = v1.x, v[i][3] = v1.y;
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s) v[i][s] = (ref < nb && k + s > j0 + ref && k + s < n) ? vp[s] : 0.0;
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            s00 = __builtin_amdgcn_mfma_f64_16x16x4f64(v[0][s], v[0][s], s00, 0, 0, 0);
            s01 = __builtin_amdgcn_mfma_f64_16x16x4f64(v[0][s], v[1][s], s01, 0, 0, 0);
            s11 = __builtin_amdgcn_mfma_f64_16x16x4f64(v[1][s], v[1][s], s11, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int e = (lk + 4 * r) * 16 + li;
        Sp[wv][0][e] = s00[r];
        Sp[wv][1][e] = s01[r];
        Sp[wv][2][e] = s11[r];
    }
    __syncthreads();
    for (int e = tid; e < 768; e += 256)
        S[e >> 8][(e & 255) >> 4][e & 15] = (Sp[0][e >> 8][e & 255] + Sp[1][e >> 8][e & 255]) +
                                            (Sp[2][e >> 8][e & 255] + Sp[3][e >> 8][e & 255]);
    __syncthreads();
    // T[a][j] = -tau_j sum_{a <= l < j} T[a][l] S[l][j], T[j][j] = tau_j: a row
    // depends on itself only, one lane each
    if (tid < kBlk) {
        double *tf = T.tf + (int64_t)blockIdx.y * kBlk * kBlk + tid * kBlk;
        double row[kBlk];
#pragma unroll
        for (int j = 0; j < kBlk; ++j) {
            const double tj = j < nb ? T.tau[j0 + j] : 0.0;
            double s = 0.0;
#pragma unroll
            for (int l = 0; l < j; ++l)
                s = fma(row[l], l < 16 ? (j < 16 ? S[0][l][j] : S[1][l][j - 16]) : S[2][l - 16][j - 16], s);
            row[j] = tid == j ? tj : tid < j ? -tj * s : 0.0;
            tf[j] = row[j];
        }
    }
}

// A work-group takes 16 RT rows of rt, its NW waves the columns.  Few
// work-groups are bound by the chain of blocks: 16 rows and eight waves take
// half of the time of 32 rows and four (one matrix of order 64 11 / 24 us, 256
// 56 / 126, 2048 1.94 / 4.05 ms; 30 of 256 85 / 129), many by the reads of V,
// which 32 rows share (60 of 256 167 / 168, 150 436 / 402, 800 2.5 / 2.0 ms).
constexpr int64_t kBackFew = 384;   // work-groups of 32 rows
template <int RT, int NW>
__global__ __launch_bounds__(64 * NW) void td_back_kernel(const syn_gbj_item *__restrict__ items) {
    __shared__ double Yp[NW][16 * RT][kBlk + 1], Z[16 * RT][kBlk + 1], F[kBlk][kBlk + 1];
    const Tdc T = tdc_view(items[blockIdx.x]);
    const int n = T.n, r0 = blockIdx.y * 16 * RT;
    if (r0 >= n || *T.fail) return;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    for (int b = refl_blocks(n) - 1; b >= 0; --b) {
        const int j0 = b * kBlk, nb = n - 2 - j0 < kBlk ? n - 2 - j0 : kBlk, cs = j0 + 1;
        __syncthreads();   // Yp, Z and F of the previous block are free
        const double *tf = T.tf + (int64_t)b * kBlk * kBlk;
        for (int e = tid; e < kBlk * kBlk; e += 64 * NW) F[e / kBlk][e % kBlk] = tf[e];
        // Y = rt V^T-rows over this wave's chunks of 16 columns: lane lk
        // takes four consecutive columns of each chunk, element s of every
        // lane in the s-th MFMA (the same columns in both operands)
        v4d acc[RT][2];
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
        for (int k0 = cs + 16 * wv; k0 < n; k0 += 16 * NW) {
            const int k = k0 + 4 * lk;
            double q[RT][4], v[2][4];
            if (nb == kBlk && k0 >= j0 + kBlk && k0 + 16 <= n) {
                // right of the block's triangle: whole rows of V; rows of rt
                // past the last repeat it (their results are not stored)
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const int row = r0 + 16 * i + li < n ? r0 + 16 * i + li : n - 1;
                    const double *qp = T.rt + (int64_t)row * T.ldr + k;
                    const v2du q0 = *(const v2du *)qp, q1 = *(const v2du *)(qp + 2);
                    q[i][0] = q0.x, q[i][1] = q0.y, q[i][2] = q1.x, q[i][3] = q1.y;
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const double *vp = T.g + (int64_t)(j0 + 16 * i + li) * T.ldg + k;
                    const v2du v0 = *(const v2du *)vp, v1 = *(const v2du *)(vp + 2);
                    v[i][0] = v0.x, v[i][1] = v0.y, v[i][2] = v1.x, v[i][3] = v1.y;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int row = r0 + 16 * i + li, ref = 16 * i + li;
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const bool in = k + s < n;
                        if (i < RT) q[i < RT ? i : 0][s] = (in && row < n) ? T.rt[(int64_t)row * T.ldr + k + s] : 0.0;
                        v[i][s] = (in && ref < nb && k + s > j0 + ref) ? T.g[(int64_t)(j0 + ref) * T.ldg + k + s] : 0.0;
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < RT; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(q[i][s], v[j][s], acc[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) Yp[wv][16 * i + lk + 4 * r][16 * j + li] = acc[i][j][r];
        __syncthreads();
        for (int e = tid; e < 16 * RT * kBlk; e += 64 * NW) {
            const int i = e / kBlk, j = e % kBlk;
            double y = 0.0;
#pragma unroll
            for (int w = 0; w < NW; w += 4) y += (Yp[w][i][j] + Yp[w + 1][i][j]) + (Yp[w + 2][i][j] + Yp[w + 3][i][j]);
            Yp[0][i][j] = y;
        }
        __syncthreads();
        // Z = Y T^T, T upper triangular
        for (int e = tid; e < 16 * RT * kBlk; e += 64 * NW) {
            const int i = e / kBlk, a = e % kBlk;
            double s = 0.0;
            for (int c = a; c < kBlk; ++c) s = fma(Yp[0][i][c], F[a][c], s);
            Z[i][a] = s;
        }
        __syncthreads();
        // rt -= Z V, 16 columns of both row tiles at a time
        for (int c0 = cs + 16 * wv; c0 < n; c0 += 16 * NW) {
            const int col = c0 + li;
            v4d o[RT];
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = r0 + 16 * i + lk + 4 * r;
                    o[i][r] = (row < n && col < n) ? T.rt[(int64_t)row * T.ldr + col] : 0.0;
                }
#pragma unroll
            for (int k0 = 0; k0 < kBlk; k0 += 4) {
                const int ref = k0 + lk;
                const double v =
                    (ref < nb && col < n && col > j0 + ref) ? T.g[(int64_t)(j0 + ref) * T.ldg + col] : 0.0;
#pragma unroll
                for (int i = 0; i < RT; ++i)
                    o[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(-Z[16 * i + li][k0 + lk], v, o[i], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = r0 + 16 * i + lk + 4 * r;
                    if (row < n && col < n) T.rt[(int64_t)row * T.ldr + col] = o[i][r];
                }
        }
    }
}

// G's upper triangle back from the lower one (the reflectors are used up),
// a 32 x 32 tile pair per work-group; where the phase does not apply, rt is
// the identity the Jacobi sweeps start from.
__global__ __launch_bounds__(256) void td_restore_kernel(const syn_gbj_item *__restrict__ items) {
    __shared__ double s[32][33];
    const Tdc T = tdc_view(items[blockIdx.x]);
    const int n = T.n, nt = (n + 31) / 32;
    if (blockIdx.y == 0 && threadIdx.x == 0 && *T.fail == kGaveUp) *items[blockIdx.x].counter = 1;   // in host memory
    int bi = 0, t = blockIdx.y;
    if (t >= nt * (nt + 1) / 2) return;
    while (t > bi) t -= ++bi;   // tile (bi, t), t <= bi
    const int r0 = 32 * bi, c0 = 32 * t, tx = threadIdx.x & 31, ty = threadIdx.x >> 5, fail = *T.fail;
    if (fail != kDiagonal) {
        for (int i = ty; i < 32; i += 8)
            s[i][tx] = (r0 + i < n && c0 + tx < n) ? T.g[(int64_t)(r0 + i) * T.ldg + c0 + tx] : 0.0;
        __syncthreads();
        for (int i = ty; i < 32; i += 8) {
            const int r = c0 + i, c = r0 + tx;
            if (r < n && c < n && c > r) T.g[(int64_t)r * T.ldg + c] = s[tx][i];
        }
    }
    if (fail) {
        for (int i = ty; i < 32; i += 8) {
            if (r0 + i < n && c0 + tx < n) T.rt[(int64_t)(r0 + i) * T.ldr + c0 + tx] = (r0 + i == c0 + tx) ? 1.0 : 0.0;
            if (c0 + i < n && r0 + tx < n) T.rt[(int64_t)(c0 + i) * T.ldr + r0 + tx] = (c0 + i == r0 + tx) ? 1.0 : 0.0;
        }
    }
}

constexpr int kSingleMax = 256;   // largest order that one work-group reduces

// largest order of the class (nlo, nhi], 0 if it has none
static int64_t class_max(const std::vector<syn_gbj_item> &host, int nlo, int nhi) {
    int64_t m = 0;
    for (const syn_gbj_item &it : host)
        if (it.nv > nlo && it.nv <= nhi) m = std::max(m, it.nv);
    return m;
}

template <int NB>
static int reduce_single(const syn_gbj_item *items, const std::vector<syn_gbj_item> &host, int nlo, double tol, hipStream_t st) {
    if (!class_max(host, nlo, 16 * NB)) return SYN_OK;
    hipLaunchKernelGGL(td_reduce_kernel<NB>, dim3((unsigned)host.size()), dim3(64 * NB), 0, st, items, nlo, 16 * NB,
                       tol);
    SYN_LAUNCH_CHECK("tridiagonal reduction");
    return SYN_OK;
}

// work-groups of a matrix, and the kernel's launch: how many one XCD gets, and
// whether a whole matrix fits the device
struct MultiPlan {
    unsigned S = 0;
    int grouped = 0;
    bool fits = true, half = true;
};

// work-groups of the kernel that the device holds at a time
template <int P, int Q>
static int64_t multi_slots() {
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, td_reduce_multi_kernel<P, Q>, kMultiThreads, 0) !=
            hipSuccess)
        return 0;
    return (int64_t)cus * per_cu;
}

template <int P, int Q>
static MultiPlan multi_plan(const std::vector<syn_gbj_item> &host, int nlo) {
    MultiPlan m;
    const int64_t nmax = class_max(host, nlo, 64 * P);
    if (!nmax) return m;
    m.S = (unsigned)multi_groups<Q>(nmax);
    // up to 16 work-groups of a matrix on one XCD, more over all of them
    m.grouped = m.S <= kGroupedMax;
    static const int64_t slots = multi_slots<P, Q>();   // a process's devices are alike
    int64_t xcd[kXcds] = {};
    for (size_t i = 0; i < host.size(); ++i)
        if (host[i].nv > nlo && host[i].nv <= 64 * P) {
            if (m.grouped)
                xcd[i & (kXcds - 1)] += m.S;
            else
                for (int64_t &x : xcd) x += (m.S + kXcds - 1) / kXcds;
        }
    m.fits = (int64_t)(m.grouped ? kXcds * m.S : m.S) <= slots;
    m.half = 2 * kXcds * *std::max_element(xcd, xcd + kXcds) <= slots;
    return m;
}

// Launches whose work-groups wait for each other, over all streams of a device:
// side by side they could each hold units that the other waits for.  Two may run
// at once if both take no more than half of the work-groups that fit an XCD (the
// work-groups of one then always find units beside the other's); a larger one runs
// alone.  A turn waits on the device for the one before it in its place (a larger
// one for both) and ends with an event; the lock covers the enqueueing alone.
class SpinTurn {
  public:
    SpinTurn(hipStream_t st, bool half) : lock_(mu()), st_(st) {
        int dev = 0;
        rc_ = hip_check(hipGetDevice(&dev), "direct phase device");
        if (rc_) return;
        auto &all = events();
        if ((size_t)dev >= all.size()) all.resize((size_t)dev + 1);
        Places &pl = all[dev];
        int at = 0;
        if (half) {
            // the place that this stream had last, or the one taken longer ago
            at = pl.last[0] == st ? 0 : pl.last[1] == st ? 1 : pl.next;
            pl.last[at] = st;
            pl.next = at ^ 1;
        }
        for (int i = 0; i < 2 && !rc_; ++i) {
            if (half && i != at) continue;
            hipEvent_t &ev = pl.ev[i];
            if (ev)
                rc_ = hip_check(hipStreamWaitEvent(st, ev, 0), "direct phase turn");
            else
                rc_ = hip_check(hipEventCreateWithFlags(&ev, hipEventDisableTiming), "direct phase event");
            end_[i] = rc_ ? nullptr : ev;
        }
    }
    int rc() const { return rc_; }
    int end() {
        int rc = SYN_OK;
        for (hipEvent_t ev : end_)
            if (ev && !rc) rc = hip_check(hipEventRecord(ev, st_), "direct phase turn");
        return rc;
    }

  private:
    struct Places {
        hipEvent_t ev[2] = {nullptr, nullptr};
        hipStream_t last[2] = {(hipStream_t)-1, (hipStream_t)-1};   // a hint, never used as a stream
        int next = 0;
    };
    static std::mutex &mu() {
        static std::mutex m;
        return m;
    }
    static std::vector<Places> &events() {
        static std::vector<Places> v;
        return v;
    }
    std::lock_guard<std::mutex> lock_;
    hipStream_t st_;
    hipEvent_t end_[2] = {nullptr, nullptr};
    int rc_ = 0;
};

template <int P, int Q>
static int reduce_multi(const syn_gbj_item *items, const std::vector<syn_gbj_item> &host, int nlo, const MultiPlan &m,
                        int polls, double tol, hipStream_t st) {
    if (!m.S) return SYN_OK;
    const int nhi = 64 * P;
    const int64_t nmax = class_max(host, nlo, nhi);
    const unsigned ni = (unsigned)host.size();
    hipLaunchKernelGGL(td_clear_kernel, dim3(ni, (unsigned)((6 * nmax + 255) / 256)), dim3(256), 0, st, items, nlo, nhi,
                       m.fits ? kDiagonal : 1);
    if (m.fits) {
        hipLaunchKernelGGL(td_test_kernel, dim3(ni, 64), dim3(256), 0, st, items, nlo, nhi, tol);
        const unsigned grid = (m.grouped ? (ni + 7) / 8 * 8 : ni) * m.S;
        hipLaunchKernelGGL((td_reduce_multi_kernel<P, Q>), dim3(grid), dim3(kMultiThreads), 0, st, items, (int)ni, nlo,
                           nhi, (int)m.S, m.grouped, polls ? polls : kArrive, polls ? polls : kSpin);
    }
    SYN_LAUNCH_CHECK("tridiagonal reduction over work-groups");
    return SYN_OK;
}

static int reduce_multis(const syn_gbj_item *items, const std::vector<syn_gbj_item> &host, int polls, double tol,
                         hipStream_t st) {
    const MultiPlan m8 = multi_plan<8, 4>(host, kSingleMax), m16 = multi_plan<16, 2>(host, 512),
                    m32 = multi_plan<32, 2>(host, 1024);
    SpinTurn turn(st, m8.half && m16.half && m32.half);
    int rc = turn.rc();
    if (!rc) rc = reduce_multi<8, 4>(items, host, kSingleMax, m8, polls, tol, st);
    if (!rc) rc = reduce_multi<16, 2>(items, host, 512, m16, polls, tol, st);
    if (!rc) rc = reduce_multi<32, 2>(items, host, 1024, m32, polls, tol, st);
    const int ended = turn.end();
    return rc ? rc : ended;
}

// The products of a phase; up to 128 tiles as quadrants, the same bits (the
// line of gemm.hip; one matrix of order 64 7.2 / 4.8 us a launch, 256 13.5 /
// 7.6, 512 20.5 / 11.0).
static void td_gemm(const syn_gbj_item *items, unsigned ni, unsigned tiles, unsigned nodes, int what, int level,
                    hipStream_t st) {
    if ((int64_t)ni * tiles * nodes <= 128)
        hipLaunchKernelGGL(td_gemm_kernel<true>, dim3(ni, 4 * tiles, nodes), dim3(256), 0, st, items, what, level);
    else
        hipLaunchKernelGGL(td_gemm_kernel<false>, dim3(ni, tiles, nodes), dim3(256), 0, st, items, what, level);
}

bool tdc_takes(int64_t nv) { return nv >= kTdcMin && nv <= kTdcMax; }
bool tdc_waits(int64_t nv) { return nv > kSingleMax && nv <= kTdcMax; }

int tdc_launch(const syn_gbj_item *items, const std::vector<syn_gbj_item> &host, int polls, double tol, hipStream_t st) {
    const unsigned ni = (unsigned)host.size();
    int64_t nmax = 0;
    int levels = 0, lmax = 1;
    for (const syn_gbj_item &it : host) {
        nmax = std::max(nmax, it.nv);
        const int L = tdc_leaves(it.nv);
        lmax = std::max(lmax, L);
    }
    while ((1 << levels) < lmax) ++levels;
    {
        ProfScope ps(kTagTdReduce, 0.0, st);
        if (int rc = reduce_single<4>(items, host, 0, tol, st)) return rc;
        if (int rc = reduce_single<8>(items, host, 64, tol, st)) return rc;
        if (int rc = reduce_single<12>(items, host, 128, tol, st)) return rc;
        if (int rc = reduce_single<16>(items, host, 192, tol, st)) return rc;
        if (tdc_waits(nmax))
            if (int rc = reduce_multis(items, host, polls, tol, st)) return rc;
        const unsigned nblk = (unsigned)refl_blocks((int)nmax);
        hipLaunchKernelGGL(td_tfac_kernel, dim3(ni, nblk), dim3(256), 0, st, items);
    }
    {
        ProfScope ps(kTagTdMerge, 0.0, st);
        hipLaunchKernelGGL(td_leaf_kernel, dim3(ni, (unsigned)lmax), dim3(64), 0, st, items);
    }
    for (int l = 1; l <= levels; ++l) {
        // the largest node of the level and how many the largest problem has
        int64_t k = 0;
        for (const syn_gbj_item &it : host) {
            const int64_t L = tdc_leaves(it.nv);
            if ((L >> l) > 0) k = std::max(k, ((it.nv << l) + L - 1) / L);
        }
        const unsigned nodes = (unsigned)(lmax >> l), c64 = (unsigned)((k + 63) / 64);
        ProfScope ps(kTagTdMerge, 0.0, st);
        const size_t plds = (size_t)prep_lds(k) * sizeof(double), slds = (size_t)k * 2 * sizeof(double);
        hipLaunchKernelGGL(td_prep_kernel, dim3(ni, nodes), dim3(kPrepThreads), plds, st, items, l);
        hipLaunchKernelGGL(td_copy_kernel, dim3(ni, c64, nodes), dim3(256), 0, st, items, l);
        hipLaunchKernelGGL(td_secular_kernel, dim3(ni, c64, nodes), dim3(kSecThreads), slds, st, items, l);
        hipLaunchKernelGGL(td_zhat_kernel, dim3(ni, c64, nodes), dim3(kZhatThreads), slds + slds / 2, st, items, l);
        hipLaunchKernelGGL(td_vec_kernel, dim3(ni, (unsigned)((k + 3) / 4), nodes), dim3(256), 0, st, items, l);
        td_gemm(items, ni, c64 * c64, nodes, 0, l, st);
        SYN_LAUNCH_CHECK("divide and conquer");
    }
    const unsigned t32 = (unsigned)((nmax + 31) / 32), t64 = (unsigned)((nmax + 63) / 64);
    double n3 = 0.0;
    for (const syn_gbj_item &it : host) n3 += (double)it.nv * it.nv * it.nv;
    {
        // every reflector meets the columns right of it twice: 2 n^3
        ProfScope ps(kTagTdBack, 2.0 * n3, st);
        if ((int64_t)ni * t32 <= kBackFew)
            hipLaunchKernelGGL((td_back_kernel<1, 8>), dim3(ni, (unsigned)((nmax + 15) / 16)), dim3(512), 0, st, items);
        else
            hipLaunchKernelGGL((td_back_kernel<2, 4>), dim3(ni, t32), dim3(256), 0, st, items);
    }
    hipLaunchKernelGGL(td_restore_kernel, dim3(ni, t32 * (t32 + 1) / 2), dim3(256), 0, st, items);
    {
        ProfScope ps(kTagTdGemm, 4.0 * n3, st);
        td_gemm(items, ni, t64 * t64, 1, 1, 0, st);
        td_gemm(items, ni, t64 * t64, 1, 2, 0, st);
    }
    SYN_LAUNCH_CHECK("direct phase");
    return SYN_OK;
}

}  // namespace syn
