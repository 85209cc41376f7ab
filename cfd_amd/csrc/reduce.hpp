// Deterministic grid reductions without atomics: a full-grid kernel reduces
// each block's values in a fixed tree and stores one partial per block; a
// one-block finalize kernel combines the partials, each thread folding a fixed
// strided subset in index order, then a fixed tree.  The result does not
// depend on scheduling, so repeated runs are bitwise identical.
#pragma once

#include <hip/hip_runtime.h>

namespace cfd {

// One step of the tree: v of the lane kOff above (as far as lane 0's result
// needs it: lanes kOff and up get some lane's value).  Half and quarter waves
// change places in registers, the rest is DPP inside rows of 16: no step goes
// through LDS, as a shuffle does, and a kernel that is one chain of latencies
// waits for two such trees.  A PCG iteration (two kernels) with shuffles / so,
// one system and two, us: 32,768 rows 8.35, 8.45 / 7.8, 8.0; 131,584 rows
// 11.65, 14.4 / 10.95, 13.55; 524,288 rows 20.2, 31.6 / 19.05, 29.7.
template <int kOff>
__device__ __forceinline__ int lane_above(int v) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    if constexpr (kOff == 32) {
        const u32x2 r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
        return (int)r.y;
    } else if constexpr (kOff == 16) {
        const u32x2 r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
        return (int)r.y;
    } else {
        return __builtin_amdgcn_update_dpp(v, v, 0x100 + kOff, 0xf, 0xf, false);  // row_shl
    }
}
template <int kOff>
__device__ __forceinline__ double lane_above(double v) {
    return __hiloint2double(lane_above<kOff>(__double2hiint(v)), lane_above<kOff>(__double2loint(v)));
}

// Lanes i and i + 32, then i + 16, 8, 4, 2, 1 (the whole wave must be active)
template <class Op>
__device__ inline double wave_reduce(double v, Op op) {
    v = op(v, lane_above<32>(v));
    v = op(v, lane_above<16>(v));
    v = op(v, lane_above<8>(v));
    v = op(v, lane_above<4>(v));
    v = op(v, lane_above<2>(v));
    v = op(v, lane_above<1>(v));
    return v;  // valid in lane 0
}

struct OpMin {
    __device__ double operator()(double a, double b) const { return b < a ? b : a; }
};
struct OpSum {
    __device__ double operator()(double a, double b) const { return a + b; }
};
struct OpMax {
    __device__ double operator()(double a, double b) const { return b > a ? b : a; }
};

// Block-wide reduction; the value is valid in thread 0.  Every thread of the
// block must call it.  Block size: a multiple of 64, at most 1024.
template <class Op>
__device__ inline double block_reduce(double v, Op op) {
    __shared__ double sh[16];
    v = wave_reduce(v, op);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();  // sh may still be read by a previous call
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        v = sh[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) v = op(v, sh[w]);
    }
    return v;
}

// Full-grid pass: one partial per block (at index `at`: the block's logical
// index when the grid is remapped, else blockIdx.x).
template <class Op>
__device__ inline void block_partial(double v, Op op, double* partials, int at) {
    v = block_reduce(v, op);
    if (threadIdx.x == 0) partials[at] = v;
}
template <class Op>
__device__ inline void block_partial(double v, Op op, double* partials) {
    block_partial(v, op, partials, (int)blockIdx.x);
}

// One-block finalize: combine partials[0..n); valid in thread 0.
template <class Op>
__device__ inline double combine_partials(const double* partials, int n, double init, Op op) {
    double acc = init;
    // each thread folds partials threadIdx.x, + blockDim.x, ... in that order;
    // sixteen (then eight, four) at a time are loaded before they are folded,
    // so that large grids keep many loads in flight
    const int stride = (int)blockDim.x;
    int b = (int)threadIdx.x;
    for (; b + 15 * stride < n; b += 16 * stride) {
        double v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = partials[b + q * stride];
#pragma unroll
        for (int q = 0; q < 16; ++q) acc = op(acc, v[q]);
    }
    if (b + 7 * stride < n) {  // then eight
        double v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = partials[b + q * stride];
#pragma unroll
        for (int q = 0; q < 8; ++q) acc = op(acc, v[q]);
        b += 8 * stride;
    }
    if (b + 3 * stride < n) {  // then four
        double v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = partials[b + q * stride];
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = op(acc, v[q]);
        b += 4 * stride;
    }
    for (; b < n; b += stride) acc = op(acc, partials[b]);
    return block_reduce(acc, op);
}

// (A "last block combines" variant -- a device-scope fence and an atomic
// arrival count per block -- measured 2.6x slower per PCG iteration than the
// separate one-block finalize kernel on gfx950: each block's release fence
// writes back its L2.  The next kernel's blocks combine the partials instead, each
// for itself, or a one-block kernel where they are many.)

namespace {
// *out = min(init, partials[0..n)), then min(*out, cap) (one block of 256)
__global__ void __launch_bounds__(256)
k_min_finalize(const double* __restrict__ partials, int n, double init, double cap,
               double* __restrict__ out) {
    double m = combine_partials(partials, n, init, OpMin());
    if (threadIdx.x == 0) *out = m > cap ? cap : m;
}
}  // namespace

}  // namespace cfd
