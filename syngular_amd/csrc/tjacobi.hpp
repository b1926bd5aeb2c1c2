// Workspace layout of the blocked Gram eigen-solver, shared by its direct
// phase (tdc.hip) and its Jacobi sweeps (tjacobi.hip).
#pragma once
#include "common.hpp"

namespace syn {

constexpr int kTCol = 64;            // columns of an rt slab

struct TjDims {
    int64_t nblk, np, half, ncs;
};

// rt slab width: the fused 16-row steps give each wave two groups of 16
// columns (fewer, fuller work-groups, so a launch of a few large problems
// fits one round of resident work-groups); the 32-row updates one
template <int TB>
__host__ __device__ constexpr int tj_slab_cols() {
    return TB == 16 ? 2 * kTCol : kTCol;
}

template <int TB>
__host__ __device__ __forceinline__ TjDims tj_dims(int64_t nv) {
    TjDims d;
    d.nblk = (nv + TB - 1) / TB;
    d.np = d.nblk + (d.nblk & 1);
    d.half = d.np / 2;
    d.ncs = (nv + tj_slab_cols<TB>() - 1) / tj_slab_cols<TB>();
    return d;
}

// Absolute rotation floor eps * max_i G_ii (set by the init kernel): Gram
// entries below it are at the rounding level of forming G, so rotating them
// changes nothing that the Gram route can resolve, and in a rank-deficient G
// (a null space at noise level) a purely relative test would never settle.
template <int TB>
__host__ __device__ __forceinline__ int64_t tj_floor_off(int64_t half) {
    return 2 * half * (2 * TB) * (2 * TB) + half;
}

// the second Gram buffer (ld nv), after the sort scratch
template <int TB>
__host__ __device__ __forceinline__ int64_t tj_g2_off(int64_t half, int64_t nv) {
    return tj_floor_off<TB>(half) + 1 + nv * nv + nv + 4;
}

// per-problem workspace: W tiles and flags (two sets), floor, the sort
// scratch (rt copy, s) and the second Gram buffer
template <int TB>
static int64_t tj_work(int64_t nv) {
    const int64_t half = tj_dims<TB>(nv).half;
    return tj_g2_off<TB>(half, nv) + nv * nv;
}

}  // namespace syn
