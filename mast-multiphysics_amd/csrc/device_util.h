// Block-level reductions shared by the kernel files (blockDim 256, 4 waves).
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace mastg {

// XCD-aware work-group order.  The dispatcher deals work-groups to the 8 XCDs
// (each with its own L2) round-robin: block b runs on XCD b % 8.  Renumbering
// block b to this index gives XCD x the contiguous run [x q + min(x, r),
// (x + 1) q + min(x + 1, r)) of an nb-block grid (nb = 8 q + r), so stencil
// neighbours gathered by one work-group were mostly fetched into the same L2
// by the work-groups before it.  A bijection of [0, nb) for every nb >= 1.
__host__ __device__ constexpr int64_t xcd_block(int64_t b, int64_t nb) {
    return (b & 7) * (nb >> 3) + ((b & 7) < (nb & 7) ? (b & 7) : (nb & 7)) + (b >> 3);
}

// LDS written by a wave's lanes before this is seen by all of its lanes after
// it, and what they read before is read: an exchange within the wave, for code
// that the work-group's other waves do not pass through (no barrier; no
// instruction beyond the waits for the wave's own LDS accesses)
__device__ __forceinline__ void wave_exchange() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// block-level FP64 sum into partials[blockIdx.x] (blockDim 256)
__device__ __forceinline__ void block_sum_store(double v, double* partials, int slot) {
    __shared__ double red[4];
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) partials[slot] = (red[0] + red[1]) + (red[2] + red[3]);
}

// deterministic final reduction of `n` partials (one block of 256)
__device__ __forceinline__ double reduce_partials(const double* __restrict__ p, int n) {
    __shared__ double red[4];
    // four independent accumulators keep four loads in flight per thread
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int i = threadIdx.x;
    for (; i + 768 < n; i += 1024) {
        s0 += p[i];
        s1 += p[i + 256];
        s2 += p[i + 512];
        s3 += p[i + 768];
    }
    for (; i < n; i += 256) s0 += p[i];
    double s = (s0 + s1) + (s2 + s3);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    const double t = (red[0] + red[1]) + (red[2] + red[3]);
    __syncthreads();
    return t;
}

// two arrays of partials at once (their loads and exchanges overlap)
__device__ __forceinline__ double2 reduce_partials2(const double* __restrict__ p, const double* __restrict__ q, int n) {
    __shared__ double red[8];
    double a0 = 0.0, a1 = 0.0, b0 = 0.0, b1 = 0.0;
    int i = threadIdx.x;
    for (; i + 256 < n; i += 512) {
        a0 += p[i];
        a1 += p[i + 256];
        b0 += q[i];
        b1 += q[i + 256];
    }
    if (i < n) {
        a0 += p[i];
        b0 += q[i];
    }
    double a = a0 + a1, b = b0 + b1;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        a += __shfl_xor(a, m, 64);
        b += __shfl_xor(b, m, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = a;
        red[4 + (threadIdx.x >> 6)] = b;
    }
    __syncthreads();
    const double2 t = {(red[0] + red[1]) + (red[2] + red[3]), (red[4] + red[5]) + (red[6] + red[7])};
    __syncthreads();
    return t;
}

// block-level max of non-negative values into partials[slot]
__device__ __forceinline__ void block_max_store(double v, double* partials, int slot) {
    __shared__ double red[4];
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = fmax(v, __shfl_xor(v, m, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) partials[slot] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// one work-group of 256: ||r||^2 of the updated residual, the iteration count
// and convergence (after an outcome: handed on)
__device__ __forceinline__ void pcg_check_block(const CGCheck& C) {
    CGScalars* S = C.S;
    const int was = S->done_r;
    if (was) {
        if (threadIdx.x == 0) S->done_z = was;
        return;
    }
    const double rr = reduce_partials(C.part, C.n);
    if (threadIdx.x == 0) {
        const int it = S->iter + 1;
        S->rr = rr;
        S->iter = it;
        S->done_z = !isfinite(rr) ? 4 : rr <= S->tol2 * S->bb ? 1 : it >= S->max_it ? 2 : 0;
    }
}

// whether a V-cycle kernel that may carry the convergence test has nothing to do
// (the test's own flag is written beside it)
__device__ __forceinline__ bool vcycle_done(const CGCheck& C, const int* done) {
    return C.S ? C.S->done_r != 0 : done && *done;
}

// the coefficients of a lattice smoothing pass, and its update of one value
// (y = A x there); returns the value's share of r . out
struct LatCoef {
    float c1, c2;
};
__device__ __forceinline__ LatCoef lat_coef(const LatSmooth& S) {
    return S.step > 0 ? LatCoef{float(S.cheb[2 * S.step]), float(S.cheb[2 * S.step + 1])} : LatCoef{0.f, float(S.cheb[0])};
}
__device__ __forceinline__ double lat_point(const LatSmooth& S, const LatCoef& c, int64_t i, float y, float x, float b,
                                            float dinv, float xp) {
    const float res = b - y;
    if (S.res) {
        S.res[i] = res;
        return 0.0;
    }
    const float z = x + (c.c1 * (x - xp) + c.c2 * dinv * res);
    S.out[i] = z;
    return S.part ? S.r[i] * double(z) : 0.0;
}

}  // namespace mastg
