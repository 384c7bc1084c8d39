// The coarse end of the multigrid V-cycle in one launch: from the first level
// that one work-group holds down to the dense coarsest solve and back up.
//
// Levels of a few thousand unknowns are launch-bound on the whole chip: a
// smoothing step, a transfer or the coarsest solve costs 4-7 us whatever its
// size, most of it launch and the latency of a chain of loads.  Here one
// work-group of 1024 threads keeps every vector of these levels in LDS and goes
// from step to step with barriers.  A thread owns DOFs t, t + 1024, ...; the
// operator is stored by entry (27 or 9 offsets x NAV columns, FP32, zero
// outside the lattice), so a product reads coalesced 16-byte loads without
// pointers.  The arithmetic is that of the separate kernels
// (FP32 entries, FP64 vectors and sums, the same Chebyshev steps).
// One V-cycle's share of these levels: heat 13^3 and 7^3 over 4^3 12.7 us
// against 13 launches (~45 us), plate 17^2 and 9^2 over 5^2 31 us
// (~60 us), hex8 9x5x5 over 5x3x3 21 us (~33 us); bound by the LDS
// reads of the products and the L2 reads of the entries on one CU, which is why
// larger levels stay on the whole chip.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "device_util.h"
#include "kernels.h"

namespace mastg {

namespace {

constexpr int kTailThreads = 1024;

template <int DIM>
__host__ __device__ constexpr int tail_offsets() { return DIM == 3 ? 27 : 9; }

typedef uint32_t tail_u4 __attribute__((ext_vector_type(4)));

// The entries of a DOF go by chunks of a few offsets, each padded to fours:
// value j of chunk c of DOF t at (((c P + j) / 4) n + t) 4 + j % 4, P the padded
// chunk.  A chunk is what a thread has in flight: all of them (28, 84, 48 registers).
constexpr int tail_chunk_offsets(int nav) { return nav == 5 ? 9 : 27; }
constexpr int tail_chunk_padded(int nav) { return (tail_chunk_offsets(nav) * nav + 3) / 4 * 4; }
template <int NAV, int DIM>
__host__ __device__ constexpr int tail_padded() {
    return tail_offsets<DIM>() / tail_chunk_offsets(NAV) * tail_chunk_padded(NAV);
}

// DOFs per thread of the first level at most: on one CU a product's entries
// come from L2 at about 0.15 TB/s, so a larger level is faster on the whole chip
constexpr int tail_passes(int nav) { return nav == 1 ? 3 : nav == 5 ? 2 : 1; }

extern __shared__ double lds[];

struct TailLds {       // a level's vectors: their first entry's place in lds
    int x, d0, d1;     // gathered: padded on both sides for offsets outside the lattice
    int res, r;
};

__host__ __device__ inline int tail_pad(const MGTailLevel& L, int nav) {
    return (1 + (L.nx + 1) * (1 + (L.nz > 0 ? L.ny + 1 : 0))) * nav;
}
__host__ __device__ inline int tail_doubles(const MGTailLevel& L, int nav) {
    const int nd = L.n_nodes * nav;
    return 5 * nd + 6 * tail_pad(L, nav);
}
__device__ __forceinline__ TailLds tail_lds(int base, const MGTailLevel& L, int nav) {
    const int nd = L.n_nodes * nav, pad = tail_pad(L, nav), s = nd + 2 * pad;
    return {base + pad, base + s + pad, base + 2 * s + pad, base + 3 * s, base + 3 * s + nd};
}

// One smoothing phase of a level: pre (x = 0, res = r, the first direction in
// d0; ends with the residual in res) or post (from x; ends with x final).
template <int NAV, int DIM, int PASSES>
__device__ __forceinline__ void tail_smooth(const MGTailLevel& L, const TailLds& V, int k, bool post) {
    constexpr int OC = tail_chunk_offsets(NAV), CP = tail_chunk_padded(NAV), NC = tail_offsets<DIM>() / OC;
    const int nd = L.n_nodes * NAV, nxp = L.nx + 1, nyp = L.ny + 1;
    const auto ent = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(L.ent), 0, NC * CP * 4 * nd, 0x00020000);
    double dinv[PASSES];
    int base[PASSES];
    bool on[PASSES];
#pragma unroll
    for (int p = 0; p < PASSES; p++) {
        const int t = threadIdx.x + kTailThreads * p;
        on[p] = t < nd;
        base[p] = on[p] ? t : 0;
        dinv[p] = L.dinv[uint32_t(base[p])];
    }
    auto product = [&](int in, int p) {
        double y0 = 0.0, y1 = 0.0;
        const int b = in + base[p] - base[p] % NAV;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            float e[CP];
#pragma unroll
            for (int i = 0; i < CP; i += 4) {   // buffer loads: a lane offset and a scalar one
                const tail_u4 q = __builtin_amdgcn_raw_buffer_load_b128(ent, base[p] * 16, (c * CP + i) * 4 * nd, 0);
#pragma unroll
                for (int j = 0; j < 4; j++) e[i + j] = __uint_as_float(q[j]);
            }
#pragma unroll
            for (int oc = 0; oc < OC; oc++) {
                const int o = c * OC + oc;
                const int q = b + ((o % 3 - 1) + nxp * ((o / 3) % 3 - 1 + (DIM == 3 ? nyp * (o / 9 - 1) : 0))) * NAV;
#pragma unroll
                for (int w = 0; w < NAV; w++) {
                    double& y = (oc * NAV + w) & 1 ? y1 : y0;
                    y = fma(double(e[oc * NAV + w]), lds[q + w], y);
                }
            }
        }
        return y0 + y1;
    };
    const double ith = L.cheb[0];
    if (post) {   // res = r - A x, d0 = D^-1 res / theta
#pragma unroll
        for (int p = 0; p < PASSES; p++) {
            const int t = threadIdx.x + kTailThreads * p;
            const double y = product(V.x, p);
            if (on[p]) {
                const double rs = lds[V.r + t] - y;
                lds[V.res + t] = rs;
                lds[V.d0 + t] = dinv[p] * rs * ith;
            }
        }
        __syncthreads();
    }
    const int last = post ? k - 1 : k;   // products with a direction
    for (int i = 1; i <= last; i++) {
        const int in = i & 1 ? V.d0 : V.d1, out = i & 1 ? V.d1 : V.d0;
        const double c1 = L.cheb[2 * (i < kMGMaxCheb ? i : 0)], c2 = L.cheb[2 * (i < kMGMaxCheb ? i : 0) + 1];
#pragma unroll
        for (int p = 0; p < PASSES; p++) {
            const int t = threadIdx.x + kTailThreads * p;
            const double y = product(in, p);
            if (on[p]) {
                const double dv = lds[in + t];
                lds[V.x + t] += dv;
                const double rs = lds[V.res + t] - y;
                lds[V.res + t] = rs;
                if (post || i < k) lds[out + t] = c1 * dv + c2 * dinv[p] * rs;
            }
        }
        __syncthreads();
    }
    if (post) {   // the last direction
        const int in = k & 1 ? V.d0 : V.d1;
#pragma unroll
        for (int p = 0; p < PASSES; p++) {
            const int t = threadIdx.x + kTailThreads * p;
            if (on[p]) lds[V.x + t] += lds[in + t];
        }
        __syncthreads();
    }
}

// a level's start from its right side: x = 0, res = r, d0 = D^-1 r / theta
__device__ __forceinline__ void tail_start(const MGTailLevel& L, const TailLds& V, int t, double r) {
    lds[V.r + t] = r;
    lds[V.x + t] = 0.0;
    lds[V.res + t] = r;
    if (L.ent) lds[V.d0 + t] = L.dinv[t] * r * L.cheb[0];
}

// r_C = P^T res_F (constrained fine residuals are 0: their rows are the identity's)
template <int NAV, int DIM>
__device__ __forceinline__ void tail_restrict(const MGTailLevel& F, const TailLds& VF, const MGTailLevel& Cl,
                                              const TailLds& VC) {
    for (int t = threadIdx.x; t < Cl.n_nodes * NAV; t += kTailThreads) {
        const int n = t / NAV, v = t - n * NAV, cx = Cl.nx + 1, cy = Cl.ny + 1;
        const int I = n % cx, J = (n / cx) % cy, K = n / (cx * cy);
        const bool con = Cl.con[t];
        double s = 0.0;
#pragma unroll
        for (int o = 0; o < tail_offsets<DIM>(); o++) {
            const int oi = o % 3 - 1, oj = (o / 3) % 3 - 1, ok = DIM == 3 ? o / 9 - 1 : 0;
            const int fi = 2 * I + oi, fj = 2 * J + oj, fk = 2 * K + ok;
            const bool in = fi >= 0 && fi <= F.nx && fj >= 0 && fj <= F.ny && fk >= 0 && fk <= F.nz;
            const double w = in ? (ok ? 0.5 : 1.0) * (oj ? 0.5 : 1.0) * (oi ? 0.5 : 1.0) : 0.0;
            const int fp = in ? fi + (F.nx + 1) * (fj + (F.ny + 1) * fk) : 0;
            s += w * lds[VF.res + fp * NAV + v];
        }
        tail_start(Cl, VC, t, con ? 0.0 : s);
    }
    __syncthreads();
}

// x_F += P x_C at unconstrained fine DOFs
template <int NAV, int DIM>
__device__ __forceinline__ void tail_prolong(const MGTailLevel& F, const TailLds& VF, const MGTailLevel& Cl,
                                             const TailLds& VC) {
    for (int t = threadIdx.x; t < F.n_nodes * NAV; t += kTailThreads) {
        const int n = t / NAV, v = t - n * NAV, fx = F.nx + 1, fy = F.ny + 1;
        const int fi = n % fx, fj = (n / fx) % fy, fk = n / (fx * fy);
        const bool con = F.con[t];
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < (1 << DIM); q++) {
            const int a = q & 1, b = (q >> 1) & 1, c = DIM == 3 ? q >> 2 : 0;
            const bool use = !((a && !(fi & 1)) || (b && !(fj & 1)) || (c && !(fk & 1)));
            const double w = use ? ((fi & 1) ? 0.5 : 1.0) * ((fj & 1) ? 0.5 : 1.0) * ((fk & 1) ? 0.5 : 1.0) : 0.0;
            const int CI = min((fi >> 1) + a, Cl.nx), CJ = min((fj >> 1) + b, Cl.ny), CK = min((fk >> 1) + c, Cl.nz);
            s += w * lds[VC.x + (CI + (Cl.nx + 1) * (CJ + (Cl.ny + 1) * CK)) * NAV + v];
        }
        if (!con) lds[VF.x + t] += s;
    }
    __syncthreads();
}

template <int NAV, int DIM>
__global__ __launch_bounds__(kTailThreads) void k_mg_tail(MGTailArgs A, const int* __restrict__ done) {
    if (done && *done) return;
    for (int i = threadIdx.x; i < A.lds_doubles; i += kTailThreads) lds[i] = 0.0;   // the pads
    __syncthreads();
    const MGTailLevel& T = A.lv[0];
    const TailLds VT = tail_lds(0, T, NAV);
    for (int t = threadIdx.x; t < T.n_nodes * NAV; t += kTailThreads) tail_start(T, VT, t, A.r[t]);
    __syncthreads();
    int at = 0;
    for (int l = 0; l + 1 < A.n; l++) {
        const TailLds V = tail_lds(at, A.lv[l], NAV);
        if (l == 0) tail_smooth<NAV, DIM, tail_passes(NAV)>(A.lv[0], V, A.steps, false);
        else tail_smooth<NAV, DIM, 1>(A.lv[l], V, A.steps, false);
        at += tail_doubles(A.lv[l], NAV);
        tail_restrict<NAV, DIM>(A.lv[l], V, A.lv[l + 1], tail_lds(at, A.lv[l + 1], NAV));
    }
    {   // the coarsest level: x = Ainv r, 8 lanes per row
        const TailLds V = tail_lds(at, A.lv[A.n - 1], NAV);
        const int n = A.lv[A.n - 1].n_nodes * NAV, sub = threadIdx.x & 7;
        for (int i = threadIdx.x >> 3; i < n; i += kTailThreads / 8) {
            double s = 0.0;
#pragma unroll 8
            for (int j = sub; j < n; j += 8) s = fma(A.Ainv[i * n + j], lds[V.r + j], s);
#pragma unroll
            for (int m = 4; m >= 1; m >>= 1) s += __shfl_xor(s, m, 8);
            if (sub == 0) lds[V.x + i] = s;
        }
        __syncthreads();
    }
    for (int l = A.n - 2; l >= 0; l--) {
        const int ac = at;
        at -= tail_doubles(A.lv[l], NAV);
        const TailLds V = tail_lds(at, A.lv[l], NAV);
        tail_prolong<NAV, DIM>(A.lv[l], V, A.lv[l + 1], tail_lds(ac, A.lv[l + 1], NAV));
        if (l == 0) tail_smooth<NAV, DIM, tail_passes(NAV)>(A.lv[0], V, A.steps, true);
        else tail_smooth<NAV, DIM, 1>(A.lv[l], V, A.steps, true);
    }
    for (int t = threadIdx.x; t < T.n_nodes * NAV; t += kTailThreads) A.x[t] = lds[VT.x + t];
}

// entries of a level from its FP64 node blocks (lattice order)
template <int NAV, int DIM>
__global__ __launch_bounds__(256) void k_mg_tail_entries(int n_nodes, int nx, int ny, const int64_t* __restrict__ blk_ptr,
                                                         const int32_t* __restrict__ blk_col,
                                                         const double* __restrict__ val, float* __restrict__ ent) {
    const int t = int(blockIdx.x) * 256 + threadIdx.x, nd = n_nodes * NAV;
    if (t >= nd) return;
    const int r = t / NAV, v = t - r * NAV, nxp = nx + 1, nyp = ny + 1;
    constexpr int OC = tail_chunk_offsets(NAV), CP = tail_chunk_padded(NAV);
    auto at = [&](int e) -> float& { return ent[((e >> 2) * nd + t) * 4 + (e & 3)]; };
    for (int e = 0; e < tail_padded<NAV, DIM>(); e++) at(e) = 0.f;
    const int64_t k0 = blk_ptr[r];
    const int deg = int(blk_ptr[r + 1] - k0);
    const double* __restrict__ V = val + k0 * (NAV * NAV);
    const int ri = r % nxp, rj = (r / nxp) % nyp, rk = r / (nxp * nyp);
    for (int k = 0; k < deg; k++) {
        const int c = blk_col[k0 + k];
        const int dx = c % nxp - ri, dy = (c / nxp) % nyp - rj, dz = c / (nxp * nyp) - rk;
        if (dx < -1 || dx > 1 || dy < -1 || dy > 1 || dz < -1 || dz > 1) continue;
        const int o = (dx + 1) + 3 * (dy + 1) + (DIM == 3 ? 9 * (dz + 1) : 0);
#pragma unroll
        for (int w = 0; w < NAV; w++) at(o / OC * CP + o % OC * NAV + w) = float(V[(v * deg + k) * NAV + w]);
    }
}

constexpr int kTailLds = 150 * 1024;     // bytes of LDS at most (160 KB per CU)
constexpr int kTailCoarse = 256;         // DOFs of the coarsest system at most

}  // namespace

int64_t mg_tail_entries(int dim, int nav, int64_t n_nodes) {
    return n_nodes * nav * (dim == 2 ? tail_padded<5, 2>() : nav == 1 ? tail_padded<1, 3>() : tail_padded<3, 3>());
}

int mg_tail_first(const MGTailLevel* lv, int nl, int nav) {
    int first = nl, bytes = 0;
    if (nl < 2 || int64_t(lv[nl - 1].n_nodes) * nav > kTailCoarse) return nl;
    for (int l = nl - 1; l >= 1; l--) {
        if (nl - l > kMGTailLevels) break;
        bytes += tail_doubles(lv[l], nav) * int(sizeof(double));
        // the levels below the first one hold one DOF per thread
        if (l < nl - 1 && int64_t(lv[l].n_nodes) * nav > int64_t(kTailThreads) * tail_passes(nav)) break;
        if (l + 1 < nl - 1 && int64_t(lv[l + 1].n_nodes) * nav > kTailThreads) break;
        if (bytes > kTailLds) break;
        first = l;
    }
    return first < nl - 1 ? first : nl;
}

void launch_mg_tail_entries(const MGLevelArgs& L, float* ent, hipStream_t s) {
    const dim3 g(unsigned((L.n_nodes * L.nav + 255) / 256));
    const int n = int(L.n_nodes);
    if (L.nav == 5)
        hipLaunchKernelGGL((k_mg_tail_entries<5, 2>), g, dim3(256), 0, s, n, L.nx, L.ny, L.blk_ptr, L.blk_col, L.val, ent);
    else if (L.nav == 1)
        hipLaunchKernelGGL((k_mg_tail_entries<1, 3>), g, dim3(256), 0, s, n, L.nx, L.ny, L.blk_ptr, L.blk_col, L.val, ent);
    else
        hipLaunchKernelGGL((k_mg_tail_entries<3, 3>), g, dim3(256), 0, s, n, L.nx, L.ny, L.blk_ptr, L.blk_col, L.val, ent);
}

// LDS beyond the default limit, once per device and kernel
hipError_t mg_tail_prepare() {
    const void* f[3] = {reinterpret_cast<const void*>(&k_mg_tail<5, 2>), reinterpret_cast<const void*>(&k_mg_tail<1, 3>),
                        reinterpret_cast<const void*>(&k_mg_tail<3, 3>)};
    for (const void* k : f) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kTailLds);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

void launch_mg_tail(MGTailArgs A, int nav, const int* done, hipStream_t s) {
    A.lds_doubles = 0;
    for (int l = 0; l < A.n; l++) A.lds_doubles += tail_doubles(A.lv[l], nav);
    const size_t b = size_t(A.lds_doubles) * sizeof(double);
    if (nav == 5) hipLaunchKernelGGL((k_mg_tail<5, 2>), dim3(1), dim3(kTailThreads), b, s, A, done);
    else if (nav == 1) hipLaunchKernelGGL((k_mg_tail<1, 3>), dim3(1), dim3(kTailThreads), b, s, A, done);
    else hipLaunchKernelGGL((k_mg_tail<3, 3>), dim3(1), dim3(kTailThreads), b, s, A, done);
}

}  // namespace mastg
