// Geometric multigrid for hex8 elasticity on lattice meshes: Galerkin coarse
// element matrices, Chebyshev/Jacobi smoothing fused into the level operators,
// trilinear restriction / prolongation, dense coarsest solve, and the
// preconditioned CG kernels around the V-cycle.
//
// Every reduction is a fixed-order sum (no atomics), so a solve is bitwise
// reproducible for a given launch configuration.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "kernels.h"
#include "device_util.h"

namespace mastg {

// libMesh hex8 local node -> cell corner offset
__constant__ int8_t kMGCorner[8][3] = {{0, 0, 0}, {1, 0, 0}, {1, 1, 0}, {0, 1, 0},
                                       {0, 0, 1}, {1, 0, 1}, {1, 1, 1}, {0, 1, 1}};

// tri/bilinear weight of coarse corner A at fine local node a of child cell c
// (c bit d = the child's offset along dimension d inside the coarse cell)
template <int DIM>
__device__ __forceinline__ double mg_q(int c, int a, int A) {
    double w = 1.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const int t = ((c >> d) & 1) + kMGCorner[a][d];   // 0, 1, 2 fine cells
        w *= kMGCorner[A][d] ? 0.5 * t : 1.0 - 0.5 * t;
    }
    return w;
}

// ---- Galerkin coarse element matrices: K_E = sum_c Q_c^T K_c Q_c ---------
// One wave per coarse element, 4 per block; lane (A, B) < NPE^2 owns one
// NAV x NAV block.  Fine blocks are masked (the rows and columns of
// constrained fine DOFs removed, as P has no row for them), the result is made
// exactly symmetric and gets the libMesh constraint convention for
// constrained coarse DOFs (rows / columns zero, unit diagonal).
template <int DIM, int NAV>
__global__ __launch_bounds__(256) void k_mg_galerkin(MGGalerkinArgs G) {
    constexpr int NPE = 1 << DIM, NCH = 1 << DIM, NB = NAV * NAV, SZ = NPE * NPE * NB;
    __shared__ double sK[4][SZ];
    __shared__ double sT[4][SZ];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool lane_on = lane < NPE * NPE;
    const int ln = lane_on ? lane : 0;
    const int hi = ln / NPE, lo = ln % NPE;
    // coarse element of this wave: the listed ones, or all of them
    const int64_t w = int64_t(blockIdx.x) * 4 + wave;
    const bool valid = G.elems ? w < G.n_elems_list : w < G.n_coarse;
    const int64_t E = !valid ? 0 : (G.elems ? int64_t(G.elems[w]) : w);
    // 32-bit index arithmetic (coarse element counts are below 2^31)
    const uint32_t Eu = uint32_t(E), cnx = uint32_t(G.cnx), Eq = Eu / cnx;
    const int64_t I = int64_t(Eu - Eq * cnx), J = int64_t(Eq % uint32_t(G.cny)), K = int64_t(Eq / uint32_t(G.cny));
    double acc[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) acc[i] = 0.0;
    for (int c = 0; c < NCH; c++) {
        const int64_t fi = 2 * I + (c & 1), fj = 2 * J + ((c >> 1) & 1), fk = DIM == 3 ? 2 * K + ((c >> 2) & 1) : 0;
        const int64_t cell = fi + int64_t(G.fnx) * (fj + int64_t(G.fny) * fk);
        const int64_t fe = G.f_elem_of_cell ? int64_t(G.f_elem_of_cell[cell]) : cell;
        if (lane_on) {   // masked fine block (a, b) = (hi, lo)
            const int32_t ra = G.f_econn[fe * NPE + hi], rb = G.f_econn[fe * NPE + lo];
            const double sc = G.Khat ? G.sE_cell[cell] : 1.0;
            const double* kb = G.Khat ? G.Khat + ln * NB : G.Kf + (fe * NPE * NPE + ln) * NB;
#pragma unroll
            for (int v = 0; v < NAV; v++)
#pragma unroll
                for (int w = 0; w < NAV; w++) {
                    double x = sc * kb[v * NAV + w];
                    if (G.f_con[int64_t(ra) * NAV + v] || G.f_con[int64_t(rb) * NAV + w]) x = 0.0;
                    sK[wave][ln * NB + v * NAV + w] = x;
                }
        }
        __syncthreads();
        if (lane_on) {   // T[a][B] = sum_b K[a][b] Q_c[b][B], lane = (a, B)
            double t[NB];
#pragma unroll
            for (int i = 0; i < NB; i++) t[i] = 0.0;
            for (int b = 0; b < NPE; b++) {
                const double q = mg_q<DIM>(c, b, lo);
                if (q != 0.0) {
                    const double* kb = &sK[wave][(hi * NPE + b) * NB];
#pragma unroll
                    for (int i = 0; i < NB; i++) t[i] += kb[i] * q;
                }
            }
#pragma unroll
            for (int i = 0; i < NB; i++) sT[wave][ln * NB + i] = t[i];
        }
        __syncthreads();
        if (lane_on)   // K_E[A][B] += sum_a Q_c[a][A] T[a][B], lane = (A, B)
            for (int a = 0; a < NPE; a++) {
                const double q = mg_q<DIM>(c, a, hi);
                if (q != 0.0) {
                    const double* tb = &sT[wave][(a * NPE + lo) * NB];
#pragma unroll
                    for (int i = 0; i < NB; i++) acc[i] += q * tb[i];
                }
            }
        __syncthreads();
    }
    // exact symmetry: lanes below the diagonal take the transpose of their partner
    if (lane_on)
#pragma unroll
        for (int i = 0; i < NB; i++) sK[wave][ln * NB + i] = acc[i];
    __syncthreads();
    if (!valid || !lane_on) return;
    double out[NB];
    if (hi > lo) {
        const double* tb = &sK[wave][(lo * NPE + hi) * NB];
#pragma unroll
        for (int v = 0; v < NAV; v++)
#pragma unroll
            for (int w = 0; w < NAV; w++) out[v * NAV + w] = tb[w * NAV + v];
    } else if (hi == lo) {
#pragma unroll
        for (int v = 0; v < NAV; v++)
#pragma unroll
            for (int w = 0; w < NAV; w++) out[v * NAV + w] = 0.5 * (acc[v * NAV + w] + acc[w * NAV + v]);
    } else {
#pragma unroll
        for (int i = 0; i < NB; i++) out[i] = acc[i];
    }
    const int32_t cA = G.c_econn[E * NPE + hi], cB = G.c_econn[E * NPE + lo];
    double* o = G.Kc + (E * NPE * NPE + ln) * NB;
#pragma unroll
    for (int v = 0; v < NAV; v++)
#pragma unroll
        for (int w = 0; w < NAV; w++) {
            double x = out[v * NAV + w];
            if (G.c_con[int64_t(cA) * NAV + v] || G.c_con[int64_t(cB) * NAV + w]) x = (hi == lo && v == w) ? 1.0 : 0.0;
            o[v * NAV + w] = x;
        }
}

// Coarse elements of a one-class hex8 lattice with no constrained DOF among
// their 27 fine nodes: K_E = sum_c s_c Gc[c] (Gc exactly symmetric, so K_E is);
// one wave per coarse element, 9 of the 576 entries per lane, coalesced stores.
__global__ __launch_bounds__(256) void k_mg_galerkin_class(MGGalerkinArgs G) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t E = int64_t(blockIdx.x) * 4 + wave;
    if (E >= G.n_coarse || G.dirty[E]) return;
    const int64_t I = E % G.cnx, J = (E / G.cnx) % G.cny, K = E / (int64_t(G.cnx) * G.cny);
    double sc[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int64_t fi = 2 * I + (c & 1), fj = 2 * J + ((c >> 1) & 1), fk = 2 * K + (c >> 2);
        sc[c] = G.sE_cell[fi + int64_t(G.fnx) * (fj + int64_t(G.fny) * fk)];
    }
    double* __restrict__ o = G.Kc + E * 576;
#pragma unroll
    for (int t = 0; t < 9; t++) {
        const int i = lane + 64 * t;
        double acc = 0.0;
#pragma unroll
        for (int c = 0; c < 8; c++) acc = fma(sc[c], G.Gc[c * 576 + i], acc);
        o[i] = acc;
    }
}

// ---- row information and eigenvalue bounds ----------------------------------
__global__ __launch_bounds__(256) void k_mg_max(const double* __restrict__ part, int n, double* __restrict__ out) {
    double m = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) m = fmax(m, part[i]);
    block_max_store(m, out, 0);
}

// Chebyshev coefficients on [lam/ratio, lam] for every level
__global__ void k_mg_cheb(const double* __restrict__ lam, double* __restrict__ cheb, int n_levels, int k,
                          double ratio) {
    const int l = threadIdx.x;
    if (l >= n_levels) return;
    const double b = lam[l] > 0.0 ? lam[l] : 1.0, a = b / ratio;
    const double theta = 0.5 * (b + a), delta = 0.5 * (b - a), sigma = theta / delta;
    double* c = cheb + l * kMGChebStride;
    c[0] = 1.0 / theta;
    c[1] = 0.0;
    double rho = 1.0 / sigma;
    for (int i = 1; i < k; i++) {
        const double rn = 1.0 / (2.0 * sigma - rho);
        c[2 * i] = rn * rho;
        c[2 * i + 1] = 2.0 * rn / delta;
        rho = rn;
    }
}

// ---- smoothing ---------------------------------------------------------------
__device__ __forceinline__ void mg_epilogue(const MGLevelArgs& L, int mode, int64_t i, double y,
                                            const double* __restrict__ din, double* __restrict__ dout,
                                            double c1, double c2, double ith) {
    if (mode == MG_RESID_INIT) {
        const double rs = L.r[i] - y;
        L.res[i] = rs;
        dout[i] = L.dinv[i] * rs * ith;
    } else {
        const double dv = din[i];
        L.x[i] += dv;
        const double rs = L.res[i] - y;
        L.res[i] = rs;
        if (mode == MG_STEP) dout[i] = c1 * dv + c2 * L.dinv[i] * rs;
    }
}

// The start of the problem level's pre-smoothing (x = 0, res = r, the first
// direction), with two neighbours' work in the same launch: a level in lattice
// order takes r from the rank-ordered vector src (null: L.r itself) and writes
// it to L.r, and the last work-group makes CG's convergence test (check).
__global__ __launch_bounds__(256) void k_mg_pre_init(MGLevelArgs L, const double* __restrict__ src,
                                                     const int32_t* __restrict__ rank_of_lat, CGCheck check,
                                                     const int* __restrict__ done) {
    const int64_t nb = gridDim.x - (check.S ? 1 : 0);
    if (int64_t(blockIdx.x) == nb) {
        pcg_check_block(check);
        return;
    }
    if (vcycle_done(check, done)) return;
    const double ith = L.cheb[0];
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < L.n_nodes * L.nav; i += nb * 256) {
        double r;
        if (src) {
            const int64_t p = i / L.nav;
            r = src[int64_t(rank_of_lat[p]) * L.nav + (i - p * L.nav)];
            L.r[i] = r;
        } else {
            r = L.r[i];
        }
        L.x[i] = 0.0;
        L.res[i] = r;
        L.da[i] = L.dinv[i] * r * ith;
    }
}

// the same start with block Jacobi (5 variables per node): da = ith Dinv_b r,
// a thread per DOF (row v of node n's inverse block), so that a wave's loads
// of the blocks and of r cover contiguous memory
__global__ __launch_bounds__(256) void k_mg_pre_init_blk5(MGLevelArgs L, CGCheck check, const int* __restrict__ done) {
    const int64_t nb = gridDim.x - (check.S ? 1 : 0);
    if (int64_t(blockIdx.x) == nb) {
        pcg_check_block(check);
        return;
    }
    if (vcycle_done(check, done)) return;
    const double ith = L.cheb[0];
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < L.n_nodes * 5; i += nb * 256) {
        const int64_t n = i / 5;
        const double* rn = L.r + n * 5;
        const float* B = L.dinvb + i * 5;   // row v = i - 5 n of node n's block
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < 5; w++) t = fma(double(B[w]), rn[w], t);
        L.x[i] = 0.0;
        L.res[i] = rn[i - n * 5];
        L.da[i] = ith * t;
    }
}

// inverse of each node's 5 x 5 diagonal block (Gauss-Jordan without pivoting:
// the blocks of an SPD matrix are SPD; constrained variables keep their unit
// diagonal convention), from the FP64 node-block values (layout (v, k, w))
__global__ __launch_bounds__(256) void k_mg_block_dinv5(MGLevelArgs L, float* __restrict__ dinvb) {
    const int64_t n = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (n >= L.n_nodes) return;
    const int64_t k0 = L.blk_ptr[n];
    const int deg = int(L.blk_ptr[n + 1] - k0);
    int kd = 0;
    for (int k = 0; k < deg; k++)
        if (L.blk_col[k0 + k] == int32_t(n)) kd = k;
    const double* V = L.val + k0 * 25;
    double a[5][5];
#pragma unroll
    for (int v = 0; v < 5; v++)
#pragma unroll
        for (int w = 0; w < 5; w++) a[v][w] = V[(v * deg + kd) * 5 + w];
#pragma unroll
    for (int k = 0; k < 5; k++) {
        const double p = 1.0 / a[k][k];
#pragma unroll
        for (int w = 0; w < 5; w++) a[k][w] = w == k ? p : a[k][w] * p;
#pragma unroll
        for (int v = 0; v < 5; v++) {
            if (v == k) continue;
            const double f = a[v][k];
#pragma unroll
            for (int w = 0; w < 5; w++) a[v][w] = w == k ? -f * p : fma(-f, a[k][w], a[v][w]);
        }
    }
#pragma unroll
    for (int v = 0; v < 5; v++)
#pragma unroll
        for (int w = 0; w < 5; w++) dinvb[n * 25 + v * 5 + w] = float(a[v][w]);
}

// the FP32 start of the hex8 problem level: b = r, x = D^-1 b / theta
__global__ __launch_bounds__(256) void k_mg_pre_init32(MGLevelArgs L, const int* __restrict__ done) {
    if (done && *done) return;
    const float ith = float(L.cheb[0]);
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < L.n_nodes * L.nav; i += int64_t(gridDim.x) * 256) {
        const float r = float(L.r[i]);
        L.b32[i] = r;
        L.x32[i] = L.dinv32[i] * r * ith;
    }
}

__device__ __forceinline__ double mg_val(double v) { return v; }
__device__ __forceinline__ double mg_val(float v) { return double(v); }
__device__ __forceinline__ double mg_val(uint16_t v) { return double(__half2float(__ushort_as_half(v))); }

// FP16 copy of a node-block matrix, each block row (node r, variable v: the
// deg x NAV values V[(v deg + k) NAV + w]) divided by its largest magnitude
template <int NAV>
__global__ __launch_bounds__(256) void k_to_f16_rows(int64_t n_nodes, const int64_t* __restrict__ blk_ptr,
                                                     const double* __restrict__ val, uint16_t* __restrict__ val16,
                                                     float* __restrict__ rs16) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n_nodes * NAV) return;
    const int64_t r = i / NAV, v = i - r * NAV;
    const int64_t k0 = blk_ptr[r];
    const int64_t deg = blk_ptr[r + 1] - k0;
    const int64_t b = k0 * NAV * NAV + v * deg * NAV, n = deg * NAV;
    double m = 0.0;
    for (int64_t t = 0; t < n; t++) m = fmax(m, fabs(val[b + t]));
    const float d = m > 0.0 ? float(m) : 1.0f;
    rs16[i] = d;
    for (int64_t t = 0; t < n; t++) val16[b + t] = __half_as_ushort(__float2half(float(val[b + t] / double(d))));
}

// node-block operator of a level (values T = double, their FP32 copy or the
// row-scaled FP16 copy; products and sums in FP64), 8 lanes per node, fused
// epilogue
template <typename T, int NAV>
__global__ __launch_bounds__(256) void k_mg_bsr(MGLevelArgs L, const T* __restrict__ vals, int mode, int step,
                                                const double* __restrict__ din, double* __restrict__ dout,
                                                const int* __restrict__ done) {
    if (done && *done) return;
    const int sub = threadIdx.x & 7;
    const double* __restrict__ in = mode == MG_RESID_INIT ? L.x : din;
    const double ith = L.cheb[0];
    const double c1 = step > 0 ? L.cheb[2 * step] : 0.0, c2 = step > 0 ? L.cheb[2 * step + 1] : 0.0;
    const int64_t nodes_per_grid = (int64_t(gridDim.x) * 256) / 8;
    for (int64_t r = (int64_t(blockIdx.x) * 256 + threadIdx.x) / 8; r < L.n_nodes; r += nodes_per_grid) {
        const int64_t k0 = L.blk_ptr[r];
        const int deg = int(L.blk_ptr[r + 1] - k0);
        const T* __restrict__ V = vals + k0 * (NAV * NAV);
        double sv[NAV];
#pragma unroll
        for (int v = 0; v < NAV; v++) sv[v] = 0.0;
        for (int k = sub; k < deg; k += 8) {
            const int64_t cb = int64_t(L.blk_col[k0 + k]) * NAV;
            double xw[NAV];
#pragma unroll
            for (int w = 0; w < NAV; w++) xw[w] = in[cb + w];
#pragma unroll
            for (int v = 0; v < NAV; v++) {
                const T* vr = V + (int64_t(v) * deg + k) * NAV;
#pragma unroll
                for (int w = 0; w < NAV; w++) sv[v] += mg_val(vr[w]) * xw[w];
            }
        }
#pragma unroll
        for (int v = 0; v < NAV; v++)
#pragma unroll
            for (int m = 4; m >= 1; m >>= 1) sv[v] += __shfl_xor(sv[v], m, 8);
        if constexpr (sizeof(T) == 2)
#pragma unroll
            for (int v = 0; v < NAV; v++) sv[v] *= double(L.rs16[r * NAV + v]);
        if (NAV == 5 && L.dinvb) {
            // block Jacobi: every lane of the node's group holds the 5 rows y;
            // each forms the 5 new residuals and lane v < 5 its direction entry
            // Dinv_b[v] . res
            const int64_t i0 = r * NAV;
            double rs[NAV];
#pragma unroll
            for (int w = 0; w < NAV; w++) rs[w] = (mode == MG_RESID_INIT ? L.r[i0 + w] : L.res[i0 + w]) - sv[w];
            if (sub < NAV) {
                const int64_t i = i0 + sub;
                double rsv = rs[0];
#pragma unroll
                for (int w = 1; w < NAV; w++) rsv = sub == w ? rs[w] : rsv;
                const float* B = L.dinvb + r * 25 + sub * 5;
                double z = 0.0;
#pragma unroll
                for (int w = 0; w < NAV; w++) z = fma(double(B[w]), rs[w], z);
                if (mode == MG_RESID_INIT) {
                    L.res[i] = rsv;
                    dout[i] = z * ith;
                } else {
                    const double dv = din[i];
                    L.x[i] += dv;
                    L.res[i] = rsv;
                    if (mode == MG_STEP) dout[i] = c1 * dv + c2 * z;
                }
            }
        } else if (sub < NAV) {
            double y = sv[0];
#pragma unroll
            for (int v = 1; v < NAV; v++) y = sub == v ? sv[v] : y;
            mg_epilogue(L, mode, r * NAV + sub, y, din, dout, c1, c2, ith);
        }
    }
}

// ---- a coarse hex8 level as a symmetric 27-point stencil --------------------
// The level's node blocks are exactly symmetric (B(r, m) = B(m, r)^T), so each
// node keeps half of them (FP32, 123 entries, entry e of node r at e N + r):
// the 13 blocks towards the neighbours o = 14..26 (o = (dx+1) + 3 (dy+1) +
// 9 (dz+1)) at e = (o - 14) 9 + 3 v + w, and the 6 entries v <= w of its own
// block at e = 117 + kSymIdx[v][w].  The block towards a neighbour m with
// o < 13 is the transpose of m's block towards r, read at index m (coalesced:
// m = r + a fixed offset).  Offsets outside the lattice hold 0.
__constant__ int8_t kSymIdx[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
constexpr int kStenEntries = 123;

__global__ __launch_bounds__(256) void k_mg_to_stencil(MGLevelArgs L, float* __restrict__ sten) {
    const int64_t r = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (r >= L.n_nodes) return;
    const int64_t N = L.n_nodes;
    const uint32_t nxp = uint32_t(L.nx + 1), nyp = uint32_t(L.ny + 1), ru = uint32_t(r), rq = ru / nxp;
    const int ri = int(ru - rq * nxp), rj = int(rq % nyp), rk = int(rq / nyp);
    for (int e = 0; e < kStenEntries; e++) sten[e * N + r] = 0.f;
    const int64_t k0 = L.blk_ptr[r];
    const int deg = int(L.blk_ptr[r + 1] - k0);
    const float* __restrict__ V = L.val32 + k0 * 9;
    for (int k = 0; k < deg; k++) {
        const uint32_t cu = uint32_t(L.blk_col[k0 + k]), cq = cu / nxp;
        const int dx = int(cu - cq * nxp) - ri, dy = int(cq % nyp) - rj, dz = int(cq / nyp) - rk;
        if (dx < -1 || dx > 1 || dy < -1 || dy > 1 || dz < -1 || dz > 1) continue;   // not a lattice neighbour
        const int o = (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1);
        if (o < 13) continue;   // kept by the neighbour
#pragma unroll
        for (int v = 0; v < 3; v++)
#pragma unroll
            for (int w = 0; w < 3; w++) {
                const float x = V[(v * deg + k) * 3 + w];
                if (o > 13) sten[((o - 14) * 9 + v * 3 + w) * N + r] = x;
                else if (v <= w) sten[(117 + kSymIdx[v][w]) * N + r] = x;
            }
    }
}

// Smoothing step of a stencil level: 64 nodes per work-group, a wave per z-layer
// of offsets, the three layers' sums exchanged through LDS, then a thread per
// DOF for the fused Chebyshev epilogue.  FP32 stencil, FP64 products and sums.
// A wave's neighbours towards (dy, dz) are 66 consecutive nodes: their vector
// goes through LDS (a lane's own loads, 24 bytes apart and three for every row,
// kept the address units busy), the stencil by coalesced buffer loads, a row of
// 27 entries at a time (two or three rows at once take the registers of a wave
// or two per SIMD: 11.2 us at 65x33x33 nodes).  What lies outside the arrays
// reads as 0.  There a thread per node took 16.4 us (one wave per SIMD), a wave
// per layer with its own vector loads 12.8, from LDS 10.4: 500 B of stencil per
// node, each read twice, at 6.5 TB/s.  At 33x17x17, bound by latency, 4.7 us.
constexpr int kStenNodes = 64;
constexpr int kStenRun = 3 * (kStenNodes + 2);   // doubles of a row's vector

typedef uint32_t sten_u2 __attribute__((ext_vector_type(2)));

template <int LZ>
__device__ __forceinline__ void stencil_layer(const MGLevelArgs& L, const float* __restrict__ sten,
                                              const double* __restrict__ in, uint32_t r0, double (&xs)[3][kStenRun],
                                              double (&y)[3]) {
    const uint32_t N = uint32_t(L.n_nodes), nxp = uint32_t(L.nx + 1), nyp = uint32_t(L.ny + 1);
    const uint32_t lane = threadIdx.x & (kStenNodes - 1), r = r0 + lane, rq = r / nxp;
    const int i = int(r - rq * nxp), j = int(rq % nyp), k = int(rq / nyp);
    // row dy of the layer, offset dx: the 9 entries (3 v + w) of the block
    // towards r + off: r's own (o - 14) 9 + 3 v + w, or the neighbour's
    // (12 - o) 9 + 3 w + v for o < 13, or r's 6 symmetric ones for o = 13
    auto entries = [&](int row, float (&e)[27]) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const int o = LZ * 9 + row * 3 + d;
            const int off = (d - 1) + int(nxp) * ((row - 1) + int(nyp) * (LZ - 1));
            const int e0 = o == 13 ? 117 : o < 13 ? (12 - o) * 9 : (o - 14) * 9;
            const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(sten + int64_t(e0) * N), 0,
                                                              (o == 13 ? 6 : 9) * N * 4u, 0x00020000);
            const uint32_t at = (r + uint32_t(o < 13 ? off : 0)) * 4u;
#pragma unroll
            for (int q = 0; q < 9; q++) {
                const int v = q / 3, w = q % 3;
                const int f = o == 13 ? (v <= w ? v * (5 - v) / 2 + w : w * (5 - w) / 2 + v) : o < 13 ? 3 * w + v : q;
                if (o == 13 && v > w) continue;   // the same as (w, v)
                e[d * 9 + q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, at, f * N * 4u, 0));
            }
            if (o == 13) {
                e[d * 9 + 3] = e[d * 9 + 1];
                e[d * 9 + 6] = e[d * 9 + 2];
                e[d * 9 + 7] = e[d * 9 + 5];
            }
        }
    };
    const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(in), 0, N * 24u, 0x00020000);
    constexpr int NT = (kStenRun + kStenNodes - 1) / kStenNodes;
    sten_u2 q[3][NT];
#pragma unroll
    for (int row = 0; row < 3; row++) {
        const uint32_t first = (r0 + uint32_t(int(nxp) * ((row - 1) + int(nyp) * (LZ - 1)) - 1)) * 24u;
#pragma unroll
        for (int t = 0; t < NT; t++)
            q[row][t] = __builtin_amdgcn_raw_buffer_load_b64(xr, first + (t * kStenNodes + lane) * 8u, 0, 0);
    }
    // loads return in the order of issue: the vector's first
    __builtin_amdgcn_sched_barrier(0);
    float e[27];
    entries(0, e);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int row = 0; row < 3; row++)
#pragma unroll
        for (int t = 0; t < NT; t++)
            if (t * kStenNodes + lane < kStenRun)
                xs[row][t * kStenNodes + lane] = __longlong_as_double((long long)(uint64_t(q[row][t][1]) << 32 | q[row][t][0]));
    wave_exchange();   // (xs is this wave's own; the waves come here by different ways)
    double y0 = 0.0, y1 = 0.0, y2 = 0.0;
#pragma unroll
    for (int row = 0; row < 3; row++) {
        if (row > 0) entries(row, e);
        const bool in_yz = j + row >= 1 && j + row <= L.ny + 1 && k + LZ >= 1 && k + LZ <= L.nz + 1;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const int o = LZ * 9 + row * 3 + d;
            double x0 = xs[row][3 * (lane + d)], x1 = xs[row][3 * (lane + d) + 1], x2 = xs[row][3 * (lane + d) + 2];
            if (o < 13) {   // a neighbour outside the lattice (its own entries there are 0)
                const bool inside = in_yz && i + d >= 1 && i + d <= L.nx + 1;
                x0 = inside ? x0 : 0.0;
                x1 = inside ? x1 : 0.0;
                x2 = inside ? x2 : 0.0;
            }
            const float* q = &e[d * 9];
            y0 = fma(double(q[2]), x2, fma(double(q[1]), x1, fma(double(q[0]), x0, y0)));
            y1 = fma(double(q[5]), x2, fma(double(q[4]), x1, fma(double(q[3]), x0, y1)));
            y2 = fma(double(q[8]), x2, fma(double(q[7]), x1, fma(double(q[6]), x0, y2)));
        }
    }
    y[0] = y0;
    y[1] = y1;
    y[2] = y2;
}

__global__ __launch_bounds__(3 * kStenNodes) void k_mg_stencil(MGLevelArgs L, const float* __restrict__ sten, int mode,
                                                               int step, const double* __restrict__ din,
                                                               double* __restrict__ dout,
                                                               const int* __restrict__ done) {
    if (done && *done) return;
    __shared__ double xs[3][3][kStenRun];
    // work-groups in XCD-aware order: the neighbouring rows whose stored
    // blocks this row reads transposed were read by work-groups of the same
    // XCD (its L2), not of another
    const uint32_t r0 = uint32_t(xcd_block(blockIdx.x, gridDim.x)) * kStenNodes;
    const int lane = threadIdx.x & (kStenNodes - 1), layer = __builtin_amdgcn_readfirstlane(threadIdx.x / kStenNodes);
    const double* __restrict__ in = mode == MG_RESID_INIT ? L.x : din;
    double y[3];
    if (layer == 0) stencil_layer<0>(L, sten, in, r0, xs[0], y);
    else if (layer == 1) stencil_layer<1>(L, sten, in, r0, xs[1], y);
    else stencil_layer<2>(L, sten, in, r0, xs[2], y);
    __syncthreads();
    double* sum = &xs[0][0][0];   // [3 layers][DOF of the work-group]
#pragma unroll
    for (int v = 0; v < 3; v++) sum[layer * 3 * kStenNodes + 3 * lane + v] = y[v];
    __syncthreads();
    const int64_t t = int64_t(r0) * 3 + threadIdx.x;
    if (t >= L.n_nodes * 3) return;
    const double ith = L.cheb[0];
    const double c1 = step > 0 ? L.cheb[2 * step] : 0.0, c2 = step > 0 ? L.cheb[2 * step + 1] : 0.0;
    const double s = (sum[threadIdx.x] + sum[3 * kStenNodes + threadIdx.x]) + sum[6 * kStenNodes + threadIdx.x];
    mg_epilogue(L, mode, t, s, din, dout, c1, c2, ith);
}

// ---- the heat problem level as a stencil in lattice order ------------------
// Its Krylov solver keeps the caller's node-rank order; the V-cycle runs the
// problem level in lattice order, so its smoother reads a stencil formed once
// per set-up from the rank-ordered rows instead of values with a column index
// each: entry o = (dx+1) + 3 (dy+1) + 9 (dz+1) of lattice point p at o N + p
// (FP32, all 27 neighbours: the Jacobian is not symmetric; offsets outside
// the lattice hold 0).  (For the plate, 5 variables per node, the node-block
// smoother measured faster than lattice-ordered stencils.)
// A coarse level (lattice order, 1 variable) converted from its rows; the
// problem level (rank order) is gathered through precomputed row positions
// (k_mg_gather_stencil).
__global__ __launch_bounds__(256) void k_mg_to_stencil27(MGLevelArgs L, float* __restrict__ sten) {
    const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (p >= L.n_nodes) return;
    const int64_t N = L.n_nodes;
    const uint32_t nxp = uint32_t(L.nx + 1), nyp = uint32_t(L.ny + 1), pu = uint32_t(p), pq = pu / nxp;
    const int pi = int(pu - pq * nxp), pj = int(pq % nyp), pk = int(pq / nyp);
    for (int e = 0; e < 27; e++) sten[e * N + p] = 0.f;
    const int64_t k0 = L.blk_ptr[p];
    const int deg = int(L.blk_ptr[p + 1] - k0);
    for (int k = 0; k < deg; k++) {
        const uint32_t qu = uint32_t(L.blk_col[k0 + k]), qq = qu / nxp;
        const int dx = int(qu - qq * nxp) - pi, dy = int(qq % nyp) - pj, dz = int(qq / nyp) - pk;
        if (dx < -1 || dx > 1 || dy < -1 || dy > 1 || dz < -1 || dz > 1) continue;   // not a lattice neighbour
        sten[((dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)) * N + p] = L.val32[k0 + k];
    }
}

// the same conversion with the row positions known: kpos[p 27 + o] is the
// position in lattice point p's (rank-ordered) row of its neighbour o, 255 for
// none (the mesh fixes it, so it is formed once on the host)
__global__ __launch_bounds__(256) void k_mg_gather_stencil(MGLevelArgs L, const int32_t* __restrict__ rank_of_lat,
                                                           const uint8_t* __restrict__ kpos,
                                                           float* __restrict__ sten) {
    const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (p >= L.n_nodes) return;
    const int64_t N = L.n_nodes;
    const float* __restrict__ V = L.val32 + L.blk_ptr[rank_of_lat[p]];
#pragma unroll 9
    for (int o = 0; o < 27; o++) {
        const int kk = kpos[p * 27 + o];
        sten[o * N + p] = kk == 255 ? 0.f : V[kk];
    }
}

// The hex8 problem level (rank order, cells of several shapes) as the
// symmetric half stencil of k_mg_stencil in lattice order: lattice point p
// keeps the blocks towards its 13 forward neighbours and the upper triangle of
// its own block, read from the FP32 row values of its rank through kpos.
// Blocks symmetric to rounding become exactly symmetric (the upper ones serve
// both directions).
__global__ __launch_bounds__(256) void k_mg_gather_stencil3(MGLevelArgs L, const int32_t* __restrict__ rank_of_lat,
                                                            const uint8_t* __restrict__ kpos,
                                                            float* __restrict__ sten) {
    const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (p >= L.n_nodes) return;
    const int64_t N = L.n_nodes;
    const int64_t r = rank_of_lat[p], k0 = L.blk_ptr[r];
    const int deg = int(L.blk_ptr[r + 1] - k0);
    const float* __restrict__ V = L.val32 + k0 * 9;
    for (int o = 13; o < 27; o++) {
        const int kk = kpos[p * 27 + o];
#pragma unroll
        for (int v = 0; v < 3; v++)
#pragma unroll
            for (int w = 0; w < 3; w++) {
                const float x = kk == 255 ? 0.f : V[(v * deg + kk) * 3 + w];
                if (o > 13) sten[((o - 14) * 9 + v * 3 + w) * N + p] = x;
                else if (v <= w) sten[(117 + kSymIdx[v][w]) * N + p] = x;
            }
    }
}

// smoothing step of the heat problem level in lattice order (FP32 stencil, FP64
// vectors and sums, fused Chebyshev epilogue)
// the heat problem level's stencil in FP16: each point's 27 entries divided
// by their largest magnitude (srow[p])
__global__ __launch_bounds__(256) void k_sten27_to_f16(int64_t N, const float* __restrict__ sten,
                                                       uint16_t* __restrict__ sten16, float* __restrict__ srow) {
    const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (p >= N) return;
    float m = 0.f;
    for (int o = 0; o < 27; o++) m = fmaxf(m, fabsf(sten[o * N + p]));
    const float d = m > 0.f ? m : 1.f;
    srow[p] = d;
    for (int o = 0; o < 27; o++) sten16[o * N + p] = __half_as_ushort(__float2half(sten[o * N + p] / d));
}

// T = float: the stencil; T = uint16_t: its FP16 copy, rows scaled by L.rs16
template <typename T>
__global__ __launch_bounds__(256) void k_mg_stencil_heat(MGLevelArgs L, const T* __restrict__ sten, int mode,
                                                         int step, const double* __restrict__ din,
                                                         double* __restrict__ dout, const int* __restrict__ done) {
    if (done && *done) return;
    // work-groups in XCD-aware order: neighbouring rows' state through one L2
    const int64_t p = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (p >= L.n_nodes) return;
    const int64_t N = L.n_nodes;
    const double* __restrict__ in = mode == MG_RESID_INIT ? L.x : din;
    const uint32_t nxp = uint32_t(L.nx + 1), nyp = uint32_t(L.ny + 1), pu = uint32_t(p), pq = pu / nxp;
    const int i = int(pu - pq * nxp), j = int(pq % nyp), k = int(pq / nyp);
    double y = 0.0;
#pragma unroll 9
    for (int o = 0; o < 27; o++) {
        // neighbours outside the lattice are clamped into it (their entries are 0)
        const int ni = min(max(i + o % 3 - 1, 0), L.nx), nj = min(max(j + (o / 3) % 3 - 1, 0), L.ny),
                  nk = min(max(k + o / 9 - 1, 0), L.nz);
        const int64_t m = int64_t(uint32_t(ni) + nxp * (uint32_t(nj) + nyp * uint32_t(nk)));
        y = fma(mg_val(sten[o * N + p]), in[m], y);
    }
    if constexpr (sizeof(T) == 2) y *= double(L.rs16[p]);
    const double ith = L.cheb[0];
    const double c1 = step > 0 ? L.cheb[2 * step] : 0.0, c2 = step > 0 ? L.cheb[2 * step + 1] : 0.0;
    mg_epilogue(L, mode, p, y, din, dout, c1, c2, ith);
}

// node-major vectors between rank order and lattice order: to_lat = 1:
// dst[p nav + v] = src[rank_of_lat[p] nav + v], else the inverse scatter
__global__ __launch_bounds__(256) void k_perm_rank_lat(int64_t n_nodes, int nav, const int32_t* __restrict__ rank_of_lat,
                                                       const double* __restrict__ src, double* __restrict__ dst,
                                                       int to_lat, const int* __restrict__ done) {
    if (done && *done) return;
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n_nodes * nav) return;
    const int64_t p = i / nav, v = i - p * nav, r = int64_t(rank_of_lat[p]) * nav + v;
    if (to_lat) dst[i] = src[r];
    else dst[r] = src[i];
}

// out (rank order) = x0 + dlast (lattice order): the V-cycle's output
__global__ __launch_bounds__(256) void k_mg_combine_rank(int64_t n_nodes, int nav,
                                                         const int32_t* __restrict__ rank_of_lat,
                                                         const double* __restrict__ x0,
                                                         const double* __restrict__ dlast, double* __restrict__ out,
                                                         const int* __restrict__ done) {
    if (done && *done) return;
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n_nodes * nav) return;
    const int64_t p = i / nav, v = i - p * nav;
    out[int64_t(rank_of_lat[p]) * nav + v] = x0[i] + dlast[i];
}

// ---- level 0 on a lattice: per-node matrix-free operator -------------------
// For congruent cells that are no axis-aligned boxes (lattice_box.hip has those).
// Thread per lattice point n, vectors component-major in lattice order (x
// fastest), so each neighbour gather of a wave is one contiguous 512-byte run;
// work-groups in XCD-aware order; for each existing cell at n
// (local corner a) y_n += s_e Khat[a][b] x_b.  Khat indices are uniform
// across the wave, so the class matrix is read with scalar-cache loads.  Each
// y_n is a fixed-order sum: results are deterministic.
__host__ __device__ constexpr int lat_cx(int b) { return (b == 1 || b == 2 || b == 5 || b == 6) ? 1 : 0; }
__host__ __device__ constexpr int lat_cy(int b) { return (b == 2 || b == 3 || b == 6 || b == 7) ? 1 : 0; }
__host__ __device__ constexpr int lat_cz(int b) { return b >= 4 ? 1 : 0; }
__host__ __device__ constexpr int lat_corner(int dx, int dy, int dz) {
    return dz * 4 + (dy ? (dx ? 2 : 3) : (dx ? 1 : 0));
}

template <typename T>
__device__ __forceinline__ T fma_t(T a, T b, T c) {
    if constexpr (sizeof(T) == 4) return fmaf(a, b, c);
    else return fma(a, b, c);
}

// Row n = (i, j, k) of the lattice operator in T (double: the CG product;
// float: the multigrid smoothing): y = sum over the existing cells at n of
// s_c Khat[a_c][b] x_b with the class matrix K (Khat or its FP32 copy), and
// cnt = the number of cells at n.  x is component-major with stride n_lat.
template <typename T>
__device__ __forceinline__ void lattice_row(const LatticeOpArgs& O, const T* __restrict__ in,
                                            const T* __restrict__ Kc, int64_t n_lat, int i, int j, int k, bool valid,
                                            T& y0, T& y1, T& y2, int& cnt) {
    const int64_t nxp = O.nx + 1, nyp = O.ny + 1;
    // neighbour-outer, one z-layer of 9 neighbours at a time (bounded live
    // ranges): each neighbour value is read once and feeds every cell shared
    // with n, y += s_c Khat[a_c][b] x_o (scaled per block product, so only y
    // is carried: fewer registers, more waves in flight to hide the gathers).
    // Neighbours outside the lattice are clamped into it; every cell holding
    // one is missing and scaled by 0.  Gathers address each component array
    // from a uniform base with a 32-bit byte offset (fewer than 2^29 lattice
    // points), and the products are explicit FMA chains: 9 FMAs per 3x3
    // block, 3 per (cell, layer) scaling.
    const char* __restrict__ b0 = reinterpret_cast<const char*>(in);
    const char* __restrict__ b1 = reinterpret_cast<const char*>(in + n_lat);
    const char* __restrict__ b2 = reinterpret_cast<const char*>(in + 2 * n_lat);
    const uint32_t sx = uint32_t(nxp), sz = uint32_t(nxp * nyp);
    auto load_layer = [&](int lz, T (&xv)[9][3]) __attribute__((always_inline)) {
        const uint32_t mk = uint32_t(min(max(k + lz - 1, 0), O.nz));
#pragma unroll
        for (int q = 0; q < 9; q++) {
            const uint32_t mi = uint32_t(min(max(i + (q % 3) - 1, 0), O.nx));
            const uint32_t mj = uint32_t(min(max(j + (q / 3) - 1, 0), O.ny));
            const uint32_t off = (mi + sx * mj + sz * mk) * uint32_t(sizeof(T));
            xv[q][0] = *reinterpret_cast<const T*>(b0 + off);
            xv[q][1] = *reinterpret_cast<const T*>(b1 + off);
            xv[q][2] = *reinterpret_cast<const T*>(b2 + off);
        }
    };
    // the first layer's gathers are issued before the scale loads (both in flight together)
    T x0v[9][3];
    load_layer(0, x0v);
    // cells at n (c bit d: the cell extends towards +d from n - 1) and their
    // scales; a missing cell gets the scale 0 (its index is clamped into the
    // lattice so every load stays in bounds)
    T sc[8];
    cnt = 0;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
        const int ci = i - 1 + cx, cj = j - 1 + cy, ck = k - 1 + cz;
        const bool has = valid & (ci >= 0) & (ci < O.nx) & (cj >= 0) & (cj < O.ny) & (ck >= 0) & (ck < O.nz);
        const int cell = min(max(ci, 0), O.nx - 1) + O.nx * (min(max(cj, 0), O.ny - 1) + O.ny * min(max(ck, 0), O.nz - 1));
        // unconditional load (the index is clamped) weighted 0 for a missing
        // cell: used on every path, so it is not sunk into a branch
        sc[c] = T(O.sE_cell[cell]) * T(has ? 1 : 0);
        cnt += has ? 1 : 0;
    }
    auto compute_layer = [&](int lz, const T (&xv)[9][3]) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
            const int bz = lz - cz;                      // uniform across the wave
            if (bz < 0 || bz > 1) continue;
            const int a = lat_corner(1 - cx, 1 - cy, 1 - cz);
            T t0 = T(0), t1 = T(0), t2 = T(0);
#pragma unroll
            for (int q = 0; q < 9; q++) {
                const int bx = (q % 3) - cx, by = (q / 3) - cy;
                if (bx < 0 || bx > 1 || by < 0 || by > 1) continue;   // compile time
                const int b = bz * 4 + lat_corner(bx, by, 0);
                const T* K = Kc + (a * 8 + b) * 9;
                t0 = fma_t(K[0], xv[q][0], t0); t0 = fma_t(K[1], xv[q][1], t0); t0 = fma_t(K[2], xv[q][2], t0);
                t1 = fma_t(K[3], xv[q][0], t1); t1 = fma_t(K[4], xv[q][1], t1); t1 = fma_t(K[5], xv[q][2], t1);
                t2 = fma_t(K[6], xv[q][0], t2); t2 = fma_t(K[7], xv[q][1], t2); t2 = fma_t(K[8], xv[q][2], t2);
            }
            y0 = fma_t(sc[c], t0, y0);
            y1 = fma_t(sc[c], t1, y1);
            y2 = fma_t(sc[c], t2, y2);
        }
    };
    y0 = y1 = y2 = T(0);
    compute_layer(0, x0v);
#pragma unroll 1
    for (int lz = 1; lz < 3; lz++) {
        T xv[9][3];
        load_layer(lz, xv);
        compute_layer(lz, xv);
    }
}

__device__ __forceinline__ void lattice_point(const LatticeOpArgs& O, int64_t p, int& i, int& j, int& k) {
    // 32-bit index arithmetic (the lattice has fewer than 2^29 points)
    const uint32_t pu = uint32_t(p), nxu = uint32_t(O.nx + 1), pj = pu / nxu;
    i = int(pu - pj * nxu);
    j = int(pj % uint32_t(O.ny + 1));
    k = int(pj / uint32_t(O.ny + 1));
}

// y = A x (FP64 CG operator) and partial sums of x.y into C.part0
__global__ __launch_bounds__(256) void k_lattice_apply(CGArgs C, const double* __restrict__ in,
                                                       double* __restrict__ ycg, const int* __restrict__ done) {
    if (done && *done) return;
    const LatticeOpArgs& O = C.lat;
    const int64_t n_lat = int64_t(O.nx + 1) * (O.ny + 1) * (O.nz + 1);
    const int64_t p = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    const bool valid = p < n_lat;
    const int64_t r = valid ? p : 0;
    int i, j, k, cnt;
    lattice_point(O, r, i, j, k);
    double y0, y1, y2;
    lattice_row<double>(O, in, O.Khat, n_lat, i, j, k, valid, y0, y1, y2, cnt);
    double dsum = 0.0;
    if (valid) {
        const int m = O.nodecon[r];
        const double x0 = in[r], x1 = in[r + n_lat], x2 = in[r + 2 * n_lat];
        if (m & 1) y0 = cnt * x0;
        if (m & 2) y1 = cnt * x1;
        if (m & 4) y2 = cnt * x2;
        ycg[r] = y0;
        ycg[r + n_lat] = y1;
        ycg[r + 2 * n_lat] = y2;
        dsum = y0 * x0 + y1 * x1 + y2 * x2;
    }
    block_sum_store(dsum, C.part0, blockIdx.x);
}

// One pass of the hex8 problem level's FP32 smoothing (LatSmooth).  The
// smoother is part of the preconditioner; the CG operator, its residuals and
// the convergence test stay FP64.  The last work-group, if S.check, only decides
// on convergence.
__global__ __launch_bounds__(256) void k_lattice_smooth(LatticeOpArgs O, LatSmooth S, const int* __restrict__ done) {
    unsigned nb = gridDim.x;
    if (S.check.S) {
        nb--;
        if (blockIdx.x == nb) {
            pcg_check_block(S.check);
            return;
        }
    }
    if (vcycle_done(S.check, done)) return;
    const int64_t n_lat = int64_t(O.nx + 1) * (O.ny + 1) * (O.nz + 1);
    const int64_t t = xcd_block(blockIdx.x, nb) * 256 + threadIdx.x, p = t < n_lat ? t : 0;
    int i, j, k, cnt;
    lattice_point(O, p, i, j, k);
    float y[3];
    lattice_row<float>(O, S.x, O.Khat32, n_lat, i, j, k, true, y[0], y[1], y[2], cnt);
    const int m = O.nodecon[p];
    const LatCoef cf = lat_coef(S);
    double rz = 0.0;
    if (t < n_lat)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int64_t q = c * n_lat + p;
            const float x = S.x[q];
            rz += lat_point(S, cf, q, (m >> c) & 1 ? float(cnt) * x : y[c], x, S.b[q], S.res ? 0.f : S.dinv[q],
                            S.xp ? S.xp[q] : 0.f);
        }
    if (S.part) block_sum_store(rz, S.part, blockIdx.x);
}

// Row information of the lattice operator without an assembled matrix: for
// each row the assembled entries A_rj = sum over the cells shared by the two
// nodes of s_c Khat[a_c][b_c], so the inverse diagonal and the Gershgorin
// ratio sum_j |A_rj| / A_rr equal those of the assembled matrix (constrained
// rows and columns as assembled: zero off the diagonal, cells-at-node on it).
__global__ __launch_bounds__(256) void k_lattice_rowinfo(LatticeOpArgs O, double* __restrict__ dinv,
                                                         float* __restrict__ dinv32, double* __restrict__ part) {
    const int64_t nxp = O.nx + 1, nyp = O.ny + 1;
    const int64_t n_lat = nxp * nyp * (O.nz + 1);
    const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
    double g = 0.0;
    if (p < n_lat) {
        int i, j, k;
        lattice_point(O, p, i, j, k);
        double sc[8];
        int cnt = 0;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
            const int ci = i - 1 + cx, cj = j - 1 + cy, ck = k - 1 + cz;
            const bool has = ci >= 0 && ci < O.nx && cj >= 0 && cj < O.ny && ck >= 0 && ck < O.nz;
            const int cell = min(max(ci, 0), O.nx - 1) + O.nx * (min(max(cj, 0), O.ny - 1) + O.ny * min(max(ck, 0), O.nz - 1));
            sc[c] = has ? O.sE_cell[cell] : 0.0;
            cnt += has ? 1 : 0;
        }
        const int mn = O.nodecon[p];
        double rs[3] = {0.0, 0.0, 0.0}, dg[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int d = 0; d < 27; d++) {
            const int dx = d % 3 - 1, dy = (d / 3) % 3 - 1, dz = d / 9 - 1;
            // neighbour o = n + (dx, dy, dz), clamped into the lattice (a
            // neighbour outside lies only in missing cells: its block is 0)
            const int oi = min(max(i + dx, 0), O.nx), oj = min(max(j + dy, 0), O.ny), ok = min(max(k + dz, 0), O.nz);
            const int mo = O.nodecon[oi + nxp * (oj + nyp * int64_t(ok))];
            double B[9];
#pragma unroll
            for (int e = 0; e < 9; e++) B[e] = 0.0;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
                // o lies in cell c when each offset is cell_d - 1 or cell_d
                if (dx < cx - 1 || dx > cx || dy < cy - 1 || dy > cy || dz < cz - 1 || dz > cz) continue;
                const int a = lat_corner(1 - cx, 1 - cy, 1 - cz);
                const int b = lat_corner(dx - cx + 1, dy - cy + 1, dz - cz + 1);
                const double* K = O.Khat + (a * 8 + b) * 9;
#pragma unroll
                for (int e = 0; e < 9; e++) B[e] = fma(sc[c], K[e], B[e]);
            }
#pragma unroll
            for (int v = 0; v < 3; v++)
#pragma unroll
                for (int w = 0; w < 3; w++) {
                    const double val = ((mn >> v) & 1) || ((mo >> w) & 1) ? 0.0 : B[v * 3 + w];
                    rs[v] += fabs(val);
                    if (d == 13 && v == w) dg[v] = val;
                }
        }
#pragma unroll
        for (int v = 0; v < 3; v++) {
            // constrained rows hold only the diagonal (one per cell at the node)
            const bool cv = (mn >> v) & 1;
            const double diag = cv ? double(cnt) : dg[v];
            const double di = diag > 0.0 ? 1.0 / diag : 0.0;
            g = fmax(g, cv ? 1.0 : (diag > 0.0 ? rs[v] / diag : 0.0));
            dinv[v * n_lat + p] = di;
            dinv32[v * n_lat + p] = float(di);
        }
    }
    block_max_store(g, part, blockIdx.x);
}

// node-vector permutation between rank order (node-major, 3 values per node)
// and the component-major lattice order: gather dst[v N + p] = src[3 map[p] + v],
// or scatter src[v N + p] -> dst[3 map[p] + v]
__global__ __launch_bounds__(256) void k_perm_nodes(int64_t n_nodes, const int32_t* __restrict__ map,
                                                    const double* __restrict__ src, double* __restrict__ dst,
                                                    int scatter) {
    const int64_t p = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (p >= n_nodes) return;
    const int64_t m = int64_t(map[p]) * 3;
    if (scatter) {
        dst[m] = src[p]; dst[m + 1] = src[n_nodes + p]; dst[m + 2] = src[2 * n_nodes + p];
    } else {
        dst[p] = src[m]; dst[n_nodes + p] = src[m + 1]; dst[2 * n_nodes + p] = src[m + 2];
    }
}

// dinv (when wanted) and the Gershgorin bound over node blocks, 8 lanes per node
template <int NAV>
__global__ __launch_bounds__(256) void k_mg_rowinfo_nb(int64_t n_nodes, const int64_t* __restrict__ blk_ptr,
                                                       const int32_t* __restrict__ blk_col,
                                                       const double* __restrict__ val, double* __restrict__ dinv,
                                                       double* __restrict__ part) {
    const int sub = threadIdx.x & 7;
    double g = 0.0;
    const int64_t nodes_per_grid = (int64_t(gridDim.x) * 256) / 8;
    for (int64_t r = (int64_t(blockIdx.x) * 256 + threadIdx.x) / 8; r < n_nodes; r += nodes_per_grid) {
        const int64_t k0 = blk_ptr[r];
        const int deg = int(blk_ptr[r + 1] - k0);
        const double* __restrict__ V = val + k0 * (NAV * NAV);
        double sv[NAV], dv[NAV];
#pragma unroll
        for (int v = 0; v < NAV; v++) sv[v] = dv[v] = 0.0;
        for (int kk = sub; kk < deg; kk += 8) {
            const bool dg = blk_col[k0 + kk] == r;
#pragma unroll
            for (int v = 0; v < NAV; v++) {
                const double* vr = V + (int64_t(v) * deg + kk) * NAV;
#pragma unroll
                for (int w = 0; w < NAV; w++) sv[v] += fabs(vr[w]);
                if (dg) dv[v] = vr[v];
            }
        }
#pragma unroll
        for (int v = 0; v < NAV; v++)
#pragma unroll
            for (int m = 4; m >= 1; m >>= 1) {
                sv[v] += __shfl_xor(sv[v], m, 8);
                dv[v] += __shfl_xor(dv[v], m, 8);
            }
        if (sub == 0)
#pragma unroll
            for (int v = 0; v < NAV; v++) {
                g = fmax(g, dv[v] > 0.0 ? sv[v] / dv[v] : 0.0);
                if (dinv) dinv[r * NAV + v] = dv[v] > 0.0 ? 1.0 / dv[v] : 0.0;
            }
    }
    block_max_store(g, part, blockIdx.x);
}

// the rows of one level in a power step, 8 lanes per node
template <int NAV>
__device__ __forceinline__ void mg_power_rows(const MGPowerLevel& L, const double* __restrict__ in, double sc,
                                              bool start, double* __restrict__ out, double* part, int blk, int nblk) {
    const int sub = threadIdx.x & 7;
    double acc = 0.0;
    for (int64_t r = (int64_t(blk) * 256 + threadIdx.x) / 8; r < L.n_nodes; r += int64_t(nblk) * 32) {
        const int64_t k0 = L.blk_ptr[r];
        const int deg = int(L.blk_ptr[r + 1] - k0);
        const double* __restrict__ V = L.val + k0 * (NAV * NAV);
        double sv[NAV];
#pragma unroll
        for (int v = 0; v < NAV; v++) sv[v] = 0.0;
        for (int k = sub; k < deg; k += 8) {
            const int64_t cb = int64_t(L.blk_col[k0 + k]) * NAV;
            double xw[NAV];
#pragma unroll
            for (int w = 0; w < NAV; w++)
                xw[w] = start ? 1.0 + double(((cb + w) * 7919) % 1000) / 1000.0 : sc * in[cb + w];
#pragma unroll
            for (int v = 0; v < NAV; v++) {
                const double* vr = V + (int64_t(v) * deg + k) * NAV;
#pragma unroll
                for (int w = 0; w < NAV; w++) sv[v] += vr[w] * xw[w];
            }
        }
#pragma unroll
        for (int v = 0; v < NAV; v++)
#pragma unroll
            for (int m = 4; m >= 1; m >>= 1) sv[v] += __shfl_xor(sv[v], m, 8);
        if (sub == 0)
#pragma unroll
            for (int v = 0; v < NAV; v++) {
                double o = L.dinv[r * NAV + v] * sv[v];
                if (NAV == 5 && L.dinvb) {   // block Jacobi: Dinv_b A
                    o = 0.0;
#pragma unroll
                    for (int w = 0; w < NAV; w++) o = fma(double(L.dinvb[r * 25 + v * 5 + w]), sv[w], o);
                }
                out[r * NAV + v] = o;
                acc += o * o;
            }
    }
    block_sum_store(acc, part, blk);
}

// Power iteration for lambda_max(D^-1 A) of several levels at once: one step of
// every level per launch (work-groups [first[l], first[l + 1]) take level l),
// out = D^-1 A (in / ||in||), ||in||^2 summed by every work-group from the
// partials the step before left, partial sums of out.out.  The start vector
// (step 0) is 1 + ((i 7919) mod 1000) / 1000.  Level by level, with a kernel for
// each norm, the 20 steps were 42 launches per level of 5-7 us each (64x64
// plate: 0.9 ms for 5 levels, now 0.15 ms).
__global__ __launch_bounds__(256) void k_mg_power(MGPowerArgs P, int step) {
    int l = 0;
    while (int(blockIdx.x) >= P.first[l + 1]) l++;
    const MGPowerLevel& L = P.level[l];
    const int blk = blockIdx.x - P.first[l], nblk = P.first[l + 1] - P.first[l];
    const double* __restrict__ in = step & 1 ? L.w0 : L.w1;
    double* __restrict__ out = step & 1 ? L.w1 : L.w0;
    double* part = P.part + P.first[l] + (step & 1 ? P.first[P.n] : 0);
    double sc = 1.0;
    if (step > 0) {
        const double s = reduce_partials(P.part + P.first[l] + (step & 1 ? 0 : P.first[P.n]), nblk);
        sc = s > 0.0 ? 1.0 / sqrt(s) : 0.0;
    }
    if (P.nav == 5) mg_power_rows<5>(L, in, sc, step == 0, out, part, blk, nblk);
    else mg_power_rows<3>(L, in, sc, step == 0, out, part, blk, nblk);
}

// lam[l] = safety ||out|| of the last step (its input had norm 1)
__global__ __launch_bounds__(256) void k_mg_power_lam(MGPowerArgs P, int last, double safety) {
    const int l = blockIdx.x;
    const double s = reduce_partials(P.part + P.first[l] + (last & 1 ? P.first[P.n] : 0), P.first[l + 1] - P.first[l]);
    if (threadIdx.x == 0) *P.level[l].lam = safety * sqrt(s);
}

// ---- transfers ---------------------------------------------------------------
// r_C = sum over the 3^DIM fine points around 2C of w * res_f (w = prod of 1 or
// 1/2), constrained fine DOFs weighted 0, constrained coarse DOFs zero (P^T),
// fused with the start of the coarse level's pre-smoothing.
// FL: layout of the fine vectors (FL_LAT lattice order, node-major; FL_RANK
// indexed through rank_of_lat, the assembled problem levels: plate, heat and
// hex8 with cells of several shapes; FL_PLANAR lattice order, component-major,
// the matrix-free hex8 problem level); coarse levels are in lattice order,
// node-major.
enum { FL_LAT = 0, FL_RANK = 1, FL_PLANAR = 2 };
template <int FL, int NAV>
__device__ __forceinline__ int64_t mg_fine_index(const MGLevelArgs& F, int64_t p, int v) {
    if (FL == FL_PLANAR) return int64_t(v) * F.n_nodes + p;
    return (FL == FL_RANK ? int64_t(F.rank_of_lat[p]) : p) * NAV + v;
}

// The transfers take a thread per DOF: with a thread per node the chip is nearly
// empty on the coarse levels and a thread's loads wait for each other (3
// variables, 33x17x17 coarse nodes in 65x33x33: restriction 7.7 us against now
// 4.8, prolongation 7.3 against 4.9; 65x33x33 in 129x65x65 14.1 / 12.9 and 15.9 /
// 13.3; the plate's 33^2 in 65^2 7.7 / 5.1 and 6.4 / 3.7).
// point and variable of thread t: planar levels by variable (coalesced per
// component), the others as their vectors lie
template <int NAV, int FL>
__device__ __forceinline__ void mg_dof(uint32_t t, uint32_t n_nodes, uint32_t& p, int& v) {
    if (FL == FL_PLANAR) {
        v = int(t / n_nodes);
        p = t - uint32_t(v) * n_nodes;
    } else {
        p = t / NAV;
        v = int(t - p * NAV);
    }
}

template <int DIM, int NAV, int FL>
__global__ __launch_bounds__(256) void k_mg_restrict(MGLevelArgs F, MGLevelArgs Cl, const int* __restrict__ done) {
    if (done && *done) return;
    const uint32_t t = blockIdx.x * 256 + threadIdx.x, nc = uint32_t(Cl.n_nodes);
    if (t >= nc * NAV) return;
    uint32_t p;
    int v;
    mg_dof<NAV, FL>(t, nc, p, v);
    // 32-bit index arithmetic (lattice point counts are below 2^31)
    const uint32_t cx = uint32_t(Cl.nx + 1), cy = uint32_t(Cl.ny + 1), pq = p / cx;
    const int I = int(p - pq * cx), J = int(pq % cy), K = int(pq / cy);
    const uint32_t fx = uint32_t(F.nx + 1), fy = uint32_t(F.ny + 1);
    constexpr int NO = DIM == 3 ? 27 : 9;
    const int64_t rc = int64_t(p) * NAV + v;
    const bool con = Cl.con[rc];
    const double dinv = Cl.dinv[rc], ith = Cl.cheb[0];
    // all loads are independent (unrolled, predicated) so they are in flight together
    double s = 0.0;
#pragma unroll
    for (int o = 0; o < NO; o++) {
        const int oi = (o % 3) - 1, oj = ((o / 3) % 3) - 1, ok = DIM == 3 ? (o / 9) - 1 : 0;
        const int fi = 2 * I + oi, fj = 2 * J + oj, fk = 2 * K + ok;
        const bool in_lat = fi >= 0 && fi <= F.nx && fj >= 0 && fj <= F.ny && fk >= 0 && fk <= F.nz;
        // out-of-lattice points are clamped (valid address) and weighted 0
        const double w = in_lat ? (ok ? 0.5 : 1.0) * (oj ? 0.5 : 1.0) * (oi ? 0.5 : 1.0) : 0.0;
        const uint32_t fp = uint32_t(in_lat ? fi : 0) + fx * (uint32_t(in_lat ? fj : 0) + fy * uint32_t(in_lat ? fk : 0));
        const int64_t rf = mg_fine_index<FL, NAV>(F, fp, v);
        const double res = FL == FL_PLANAR ? double(F.res32[rf]) : F.res[rf];
        s += (w * (1.0 - double(F.con[rf]))) * res;
    }
    // and the coarse level's pre-smoothing start (x = 0, res = r, first
    // Chebyshev direction D^-1 r / theta)
    const double r = con ? 0.0 : s;
    Cl.r[rc] = r;
    Cl.x[rc] = 0.0;
    Cl.res[rc] = r;
    Cl.da[rc] = dinv * r * ith;
}

// x_f += P (x_C + dlast_C) at unconstrained fine DOFs (tri/bilinear interpolation)
template <int DIM, int NAV, int FL>
__global__ __launch_bounds__(256) void k_mg_prolong(MGLevelArgs F, MGLevelArgs Cl, const double* __restrict__ dlast,
                                                    const int* __restrict__ done) {
    if (done && *done) return;
    const uint32_t t = blockIdx.x * 256 + threadIdx.x, nf = uint32_t(F.n_nodes);
    if (t >= nf * NAV) return;
    uint32_t p;
    int v;
    mg_dof<NAV, FL>(t, nf, p, v);
    // 32-bit index arithmetic (lattice point counts are below 2^31)
    const uint32_t fx = uint32_t(F.nx + 1), fy = uint32_t(F.ny + 1), pq = p / fx;
    const int fi = int(p - pq * fx), fj = int(pq % fy), fk = int(pq / fy);
    const uint32_t cx = uint32_t(Cl.nx + 1), cy = uint32_t(Cl.ny + 1);
    const int64_t rf = mg_fine_index<FL, NAV>(F, p, v);
    const bool con = F.con[rf];
    const double x0 = FL == FL_PLANAR ? double(F.x32[rf]) : F.x[rf];
    constexpr int NQ = 1 << DIM;
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int a = q & 1, b = (q >> 1) & 1, c = DIM == 3 ? (q >> 2) : 0;
        // an even fine index takes its one coarse point (a = 0), an odd one both
        // neighbours; the unused corner of an even index is clamped and weighted 0
        const bool use = !((a && !(fi & 1)) || (b && !(fj & 1)) || (c && !(fk & 1)));
        const double w = use ? ((fi & 1) ? 0.5 : 1.0) * ((fj & 1) ? 0.5 : 1.0) * ((fk & 1) ? 0.5 : 1.0) : 0.0;
        const uint32_t CI = uint32_t(min((fi >> 1) + a, Cl.nx)), CJ = uint32_t(min((fj >> 1) + b, Cl.ny)),
                       CK = uint32_t(min((fk >> 1) + c, Cl.nz));
        const int64_t rc = int64_t(CI + cx * (CJ + cy * CK)) * NAV + v;
        if (use) s += w * (dlast ? Cl.x[rc] + dlast[rc] : Cl.x[rc]);
    }
    if (con) return;
    if (FL == FL_PLANAR) F.x32[rf] = float(x0) + float(s);
    else F.x[rf] = x0 + s;
}

// ---- coarsest level: dense inverse -------------------------------------------
template <int NAV>
__global__ __launch_bounds__(256) void k_mg_dense_gather(MGLevelArgs L, double* __restrict__ A) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const int64_t n = L.n_nodes * NAV;
    if (i >= n) return;
    const int64_t r = i / NAV;
    const int v = int(i - r * NAV);
    const int64_t k0 = L.blk_ptr[r];
    const int64_t deg = L.blk_ptr[r + 1] - k0;
    const double* row = L.val + k0 * (NAV * NAV) + int64_t(v) * deg * NAV;
    for (int64_t k = 0; k < deg; k++) {
        const int64_t c = L.blk_col[k0 + k];
#pragma unroll
        for (int w = 0; w < NAV; w++) A[i * n + c * NAV + w] = row[k * NAV + w];
    }
}

// Blocked Gauss-Jordan inverse (no pivoting: the coarsest operators are SPD,
// or the heat Jacobian's, whose symmetric part is), one launch per 32 x 32
// diagonal block, out of place: with D the kb-th diagonal block of `in`,
//   out[kb][kb] = D^-1,  out[kb][j] = D^-1 in[kb][j],  out[i][kb] = -in[i][kb] D^-1,
//   out[i][j] = in[i][j] - in[i][kb] (D^-1 in[kb][j]).
// Bound by the chain of n pivots, each waiting for the one before it.  A
// work-group per 32 x 32 tile; the one that updates the next diagonal block
// also inverts it (Dinv of the next launch), so the pivots run once and not in
// every work-group (which took 42 us per step at n = 1188, all of them
// competing for the FP64 units).  Against the whole matrix updated pivot by
// pivot from one work-group: n = 1188 732 ms -> 0.97 ms, n = 135 (in
// registers, 1024 threads) 0.25 ms -> 0.10 ms.
constexpr int kInvB = 32;

// D^-1 of the 32 x 32 block whose entries (r0 + 8 q, c) thread t holds in a,
// in place: one barrier per pivot, the pivot row and column double-buffered
// (0.4 us per pivot; every thread dividing for itself instead of the shuffle
// and scaled row measured 5% slower)
__device__ __forceinline__ void mg_invert_block(double a[4], double (&colk)[2][kInvB], double (&rowk)[2][kInvB]) {
    const int t = threadIdx.x, lane = t & 63, c = t & 31, r0 = t >> 5;
    for (int k = 0; k < kInvB; k++) {
        const int b = k & 1, kq = k >> 3;
        if (c == k)
#pragma unroll
            for (int q = 0; q < 4; q++) colk[b][r0 + 8 * q] = a[q];
        if (r0 == (k & 7)) {   // the half wave holding pivot row k
            const double v = kq == 0 ? a[0] : kq == 1 ? a[1] : kq == 2 ? a[2] : a[3];
            const double p = 1.0 / __shfl(v, (lane & 32) | k, 64);
            rowk[b][c] = c == k ? p : v * p;
        }
        __syncthreads();   // (a buffer is rewritten two pivots later, past the next barrier)
        const double p = rowk[b][k], rk = rowk[b][c];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const double ck = colk[b][r0 + 8 * q];
            const double v = c == k ? -ck * p : fma(-ck, rk, a[q]);
            a[q] = r0 + 8 * q == k ? rk : v;
        }
    }
}

// entry (row, col) of the matrix; past n the identity's, so a last partial
// block inverts like a whole one
__device__ __forceinline__ double mg_invert_load(const double* __restrict__ A, int n, int row, int col) {
    return row < n && col < n ? A[int64_t(row) * n + col] : (row == col ? 1.0 : 0.0);
}

// the first diagonal block's inverse
__global__ __launch_bounds__(256) void k_mg_invert_first(int n, const double* __restrict__ in,
                                                         double* __restrict__ Dinv) {
    __shared__ double colk[2][kInvB], rowk[2][kInvB];
    const int c = threadIdx.x & 31, r0 = threadIdx.x >> 5;
    double a[4];
#pragma unroll
    for (int q = 0; q < 4; q++) a[q] = mg_invert_load(in, n, r0 + 8 * q, c);
    mg_invert_block(a, colk, rowk);
#pragma unroll
    for (int q = 0; q < 4; q++) Dinv[(r0 + 8 * q) * kInvB + c] = a[q];
}

__global__ __launch_bounds__(256) void k_mg_invert_step(int n, int kb, const double* __restrict__ in,
                                                        double* __restrict__ out, const double* __restrict__ Dinv,
                                                        double* __restrict__ Dnext) {
    __shared__ double D[kInvB][kInvB + 1], R[kInvB][kInvB + 1], Cl[kInvB][kInvB + 1];
    __shared__ double colk[2][kInvB], rowk[2][kInvB];
    const int c = threadIdx.x & 31, r0 = threadIdx.x >> 5;   // entries (r0 + 8 q, c), q < 4
    // the tile, tiles counted from the next diagonal block on: the work-group
    // with the longest way is dealt out first
    const int nt = gridDim.x;
    int ib = blockIdx.y + kb + 1, jb = blockIdx.x + kb + 1;
    ib -= ib >= nt ? nt : 0;
    jb -= jb >= nt ? nt : 0;
    const int gi = ib * kInvB, gj = jb * kInvB, gk = kb * kInvB;
    double o[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int r = r0 + 8 * q;
        D[r][c] = Dinv[r * kInvB + c];
        o[q] = ib != kb && jb != kb ? mg_invert_load(in, n, gi + r, gj + c) : 0.0;
        if (jb != kb) R[r][c] = mg_invert_load(in, n, gk + r, gj + c);
        if (ib != kb) Cl[r][c] = mg_invert_load(in, n, gi + r, gk + c);
    }
    __syncthreads();
    if (jb == kb) {
        if (ib == kb) {
#pragma unroll
            for (int q = 0; q < 4; q++) o[q] = D[r0 + 8 * q][c];
        } else {
#pragma unroll 8
            for (int k = 0; k < kInvB; k++) {
                const double d = D[k][c];
#pragma unroll
                for (int q = 0; q < 4; q++) o[q] = fma(-Cl[r0 + 8 * q][k], d, o[q]);
            }
        }
    } else {
        double x[4] = {0.0, 0.0, 0.0, 0.0};   // D^-1 in[kb][jb]
#pragma unroll 8
        for (int k = 0; k < kInvB; k++) {
            const double v = R[k][c];
#pragma unroll
            for (int q = 0; q < 4; q++) x[q] = fma(D[r0 + 8 * q][k], v, x[q]);
        }
        if (ib == kb) {
#pragma unroll
            for (int q = 0; q < 4; q++) o[q] = x[q];
        } else {
            __syncthreads();   // R is read
#pragma unroll
            for (int q = 0; q < 4; q++) R[r0 + 8 * q][c] = x[q];
            __syncthreads();
#pragma unroll 8
            for (int k = 0; k < kInvB; k++) {
                const double v = R[k][c];
#pragma unroll
                for (int q = 0; q < 4; q++) o[q] = fma(-Cl[r0 + 8 * q][k], v, o[q]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int r = gi + r0 + 8 * q;
        if (r < n && gj + c < n) out[int64_t(r) * n + gj + c] = o[q];
    }
    if (ib == kb + 1 && jb == kb + 1) {   // (no such tile in the last step)
        mg_invert_block(o, colk, rowk);
#pragma unroll
        for (int q = 0; q < 4; q++) Dnext[(r0 + 8 * q) * kInvB + c] = o[q];
    }
}

// x = Ainv r, one wave per row
__global__ __launch_bounds__(256) void k_mg_coarse_solve(int n, const double* __restrict__ Ainv,
                                                         const double* __restrict__ r, double* __restrict__ x,
                                                         const int* __restrict__ done) {
    if (done && *done) return;
    const int64_t i = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= n) return;
    double s = 0.0;
    for (int j = lane; j < n; j += 64) s += Ainv[i * n + j] * r[j];
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) s += __shfl_xor(s, m, 64);
    if (lane == 0) x[i] = s;
}

// ---- preconditioned CG ---------------------------------------------------------
// alpha = r.z / p.q, p.q from the operator's partials, summed by every
// work-group (a launch less than a kernel for alpha); false: over, or breakdown /
// NaN, the same in every work-group
__device__ __forceinline__ bool pcg_alpha(const CGArgs& C, double& a) {
    CGScalars* S = C.S;
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    const int was = S->done;
    if (was) {
        if (lead) S->done_r = was;
        return false;
    }
    const double pq = reduce_partials(C.part0, C.nparts_op);
    const bool bad = !(pq > 0.0) || !isfinite(pq);
    if (lead) S->done_r = bad ? 3 : 0;
    if (bad) return false;
    a = S->rz2[S->iter & 1] / pq;
    return true;
}

// x += alpha p ; r -= alpha q ; partials r.r
__global__ __launch_bounds__(256) void k_pcg_update(CGArgs C) {
    double a, rr = 0.0;
    if (!pcg_alpha(C, a)) return;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < C.n; i += int64_t(gridDim.x) * 256) {
        C.x[i] += a * C.p[i];
        const double r = C.r[i] - a * C.q[i];
        C.r[i] = r;
        rr += r * r;
    }
    block_sum_store(rr, C.part1, blockIdx.x);
}

// the lattice solver's update: x, r, the partials of r.r, and the start of the
// FP32 pre-smoothing (b = r, x = D^-1 b / theta)
__global__ __launch_bounds__(256) void k_pcg_update_lat(CGArgs C, MGLevelArgs L) {
    double a, rr = 0.0;
    if (!pcg_alpha(C, a)) return;
    const float ith = float(L.cheb[0]);
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < C.n; i += int64_t(gridDim.x) * 256) {
        C.x[i] += a * C.p[i];
        const double r = C.r[i] - a * C.q[i];
        C.r[i] = r;
        rr += r * r;
        const float rf = float(r);
        L.b32[i] = rf;
        L.x32[i] = L.dinv32[i] * rf * ith;
    }
    block_sum_store(rr, C.part1, blockIdx.x);
}

// r.z summed by every work-group, beta = r.z / the last r.z, p = z + beta p
// (first: p = z); a non-positive r.z means the preconditioner is not SPD
template <typename T>
__global__ __launch_bounds__(256) void k_pcg_p(CGArgs C, const T* __restrict__ z, int n, int first) {
    CGScalars* S = C.S;
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    const int was = S->done_z;
    if (was) {
        if (lead) S->done = was;
        return;
    }
    const double rz = reduce_partials(C.part0, n);
    const int it = S->iter;
    const bool bad = !(rz > 0.0) || !isfinite(rz);
    if (lead) S->done = bad ? 3 : 0;
    if (bad) return;
    const double beta = first ? 0.0 : rz / S->rz2[(it + 1) & 1];
    if (lead) S->rz2[it & 1] = rz;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < C.n; i += int64_t(gridDim.x) * 256)
        C.p[i] = first ? double(z[i]) : double(z[i]) + beta * C.p[i];
}

// z = x0 + dlast (the level-0 V-cycle output) ; partials r.z
__global__ __launch_bounds__(256) void k_pcg_rz(CGArgs C, const double* __restrict__ x0,
                                                const double* __restrict__ dlast) {
    if (C.S->done_z) return;
    double rz = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < C.n; i += int64_t(gridDim.x) * 256) {
        const double z = dlast ? x0[i] + dlast[i] : x0[i];
        C.z[i] = z;
        rz += C.r[i] * z;
    }
    block_sum_store(rz, C.part0, blockIdx.x);
}

// the same for a problem level in lattice order: z and r in rank order
__global__ __launch_bounds__(256) void k_pcg_rz_rank(CGArgs C, int nav, const int32_t* __restrict__ rank_of_lat,
                                                     const double* __restrict__ x0,
                                                     const double* __restrict__ dlast) {
    if (C.S->done_z) return;
    double rz = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < C.n; i += int64_t(gridDim.x) * 256) {
        const int64_t p = i / nav, k = int64_t(rank_of_lat[p]) * nav + (i - p * nav);
        const double z = x0[i] + dlast[i];
        C.z[k] = z;
        rz += C.r[k] * z;
    }
    block_sum_store(rz, C.part0, blockIdx.x);
}

__global__ __launch_bounds__(256) void k_mg_combine(int64_t n, const double* __restrict__ x0,
                                                    const double* __restrict__ dlast, double* __restrict__ out,
                                                    const int* __restrict__ done) {
    if (done && *done) return;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256)
        out[i] = dlast ? x0[i] + dlast[i] : x0[i];
}

__global__ __launch_bounds__(256) void k_pcg_start(CGArgs C, const double* __restrict__ b) {
    double bb = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < C.n; i += int64_t(gridDim.x) * 256)
        bb += b[i] * b[i];
    block_sum_store(bb, C.part1, blockIdx.x);
}

__global__ __launch_bounds__(256) void k_pcg_start_scalars(CGArgs C, double tol2, int max_it) {
    const double bb = reduce_partials(C.part1, C.nvec);
    if (threadIdx.x == 0) {
        CGScalars* S = C.S;
        S->bb = bb;
        S->rr = bb;
        S->iter = 0;
        S->tol2 = tol2;
        S->max_it = max_it;
        S->done = S->done_z = (bb == 0.0) ? 1 : (isfinite(bb) ? 0 : 4);
    }
}

// after a restart from the true residual (partials of r.r in part1): converged?
__global__ __launch_bounds__(256) void k_pcg_recheck(CGArgs C) {
    const double rr = reduce_partials(C.part1, C.nvec);
    if (threadIdx.x == 0) {
        CGScalars* S = C.S;
        S->rr = rr;
        S->done = S->done_z = !isfinite(rr) ? 4 : rr <= S->tol2 * S->bb ? 1 : S->iter >= S->max_it ? 2 : 0;
    }
}

// ---- launchers -------------------------------------------------------------------
static inline unsigned mg_blocks(int64_t n, int per) { return unsigned((n + per - 1) / per); }
static inline unsigned mg_grid(int64_t n) {
    const int64_t b = (n + 255) / 256;
    return unsigned(b < 1 ? 1 : (b > 4096 ? 4096 : b));
}

void launch_mg_galerkin(const MGGalerkinArgs& g, hipStream_t s) {
    const int64_t n = g.elems ? g.n_elems_list : g.n_coarse;
    if (n <= 0) return;
    const dim3 grid(mg_blocks(n, 4));
    if (g.dim == 2)
        hipLaunchKernelGGL((k_mg_galerkin<2, 5>), grid, dim3(256), 0, s, g);
    else if (g.nav == 1)
        hipLaunchKernelGGL((k_mg_galerkin<3, 1>), grid, dim3(256), 0, s, g);
    else
        hipLaunchKernelGGL((k_mg_galerkin<3, 3>), grid, dim3(256), 0, s, g);
}
void launch_mg_galerkin_class(const MGGalerkinArgs& g, hipStream_t s) {
    if (g.n_coarse <= 0) return;
    hipLaunchKernelGGL(k_mg_galerkin_class, dim3(mg_blocks(g.n_coarse, 4)), dim3(256), 0, s, g);
}
void launch_mg_cheb(const double* lam, double* cheb, int n_levels, int k, double ratio, hipStream_t s) {
    hipLaunchKernelGGL(k_mg_cheb, dim3(1), dim3(64), 0, s, lam, cheb, n_levels, k, ratio);
}
void launch_mg_dense_gather(const MGLevelArgs& L, double* A, hipStream_t s) {
    if (L.nav == 5)
        hipLaunchKernelGGL(k_mg_dense_gather<5>, dim3(mg_blocks(L.n_nodes * 5, 256)), dim3(256), 0, s, L, A);
    else if (L.nav == 1)
        hipLaunchKernelGGL(k_mg_dense_gather<1>, dim3(mg_blocks(L.n_nodes, 256)), dim3(256), 0, s, L, A);
    else
        hipLaunchKernelGGL(k_mg_dense_gather<3>, dim3(mg_blocks(L.n_nodes * 3, 256)), dim3(256), 0, s, L, A);
}
int64_t mg_invert_work(int n) { return int64_t(n) * n + 2 * kInvB * kInvB; }
double* mg_invert_input(int n, double* A, double* W) { return ((n + kInvB - 1) / kInvB) & 1 ? W : A; }
void launch_mg_invert(int n, double* A, double* W, hipStream_t s) {
    const int nt = (n + kInvB - 1) / kInvB;
    double *in = mg_invert_input(n, A, W), *out = in == A ? W : A;   // the last step writes A
    double *d0 = W + int64_t(n) * n, *d1 = d0 + kInvB * kInvB;
    hipLaunchKernelGGL(k_mg_invert_first, dim3(1), dim3(256), 0, s, n, in, d0);
    for (int k = 0; k < nt; k++) {
        hipLaunchKernelGGL(k_mg_invert_step, dim3(nt, nt), dim3(256), 0, s, n, k, in, out, d0, d1);
        std::swap(in, out);
        std::swap(d0, d1);
    }
}
static inline int nb_grid(int64_t n_nodes) {
    const int64_t blocks = (n_nodes * 8 + 255) / 256;
    return int(blocks < 1 ? 1 : (blocks > 8192 ? 8192 : blocks));
}
void launch_mg_rowinfo_nb(int nav, int64_t n_nodes, const int64_t* blk_ptr, const int32_t* blk_col,
                          const double* val, double* dinv, double* part, double* lam, hipStream_t s) {
    const int nb = nb_grid(n_nodes);
    if (nav == 5)
        hipLaunchKernelGGL(k_mg_rowinfo_nb<5>, dim3(nb), dim3(256), 0, s, n_nodes, blk_ptr, blk_col, val, dinv, part);
    else if (nav == 1)
        hipLaunchKernelGGL(k_mg_rowinfo_nb<1>, dim3(nb), dim3(256), 0, s, n_nodes, blk_ptr, blk_col, val, dinv, part);
    else
        hipLaunchKernelGGL(k_mg_rowinfo_nb<3>, dim3(nb), dim3(256), 0, s, n_nodes, blk_ptr, blk_col, val, dinv, part);
    hipLaunchKernelGGL(k_mg_max, dim3(1), dim3(256), 0, s, part, nb, lam);
}
// work-groups of a level: enough for its rows, at most kPowerBlocks (each sums
// all the level's partials)
constexpr int kPowerBlocks = 1024;
int64_t mg_power_partials(int n_levels) { return 2 * int64_t(n_levels) * kPowerBlocks; }
bool launch_mg_power(MGPowerArgs P, int n_it, double safety, hipStream_t s) {
    if (P.n <= 0) return true;
    if (P.nav != 3 && P.nav != 5) return false;
    P.first[0] = 0;
    for (int l = 0; l < P.n; l++) P.first[l + 1] = P.first[l] + std::min(nb_grid(P.level[l].n_nodes), kPowerBlocks);
    for (int it = 0; it < n_it; it++) hipLaunchKernelGGL(k_mg_power, dim3(P.first[P.n]), dim3(256), 0, s, P, it);
    hipLaunchKernelGGL(k_mg_power_lam, dim3(P.n), dim3(256), 0, s, P, n_it - 1, safety);
    return true;
}
static int64_t lattice_blocks(const LatticeOpArgs& l) {
    return (int64_t(l.nx + 1) * (l.ny + 1) * (l.nz + 1) + 255) / 256;
}
int64_t lattice_partials(const LatticeOpArgs& l) { return l.is_box ? box_partials(l) : lattice_blocks(l); }
int64_t lattice_partials_most(const LatticeOpArgs& l) { return std::max(lattice_blocks(l), box_partials_most(l)); }
void launch_lattice_apply(const CGArgs& c, const double* x, double* y, hipStream_t s) {
    const int* done = c.S ? &c.S->done : nullptr;
    if (c.lat.is_box) return launch_box_apply(c.lat, x, y, c.part0, done, s);
    hipLaunchKernelGGL(k_lattice_apply, dim3(unsigned(lattice_blocks(c.lat))), dim3(256), 0, s, c, x, y, done);
}
void launch_lattice_smooth(const LatticeOpArgs& l, const LatSmooth& S, const int* done, hipStream_t s) {
    if (l.is_box) return launch_box_smooth(l, S, done, s);
    hipLaunchKernelGGL(k_lattice_smooth, dim3(unsigned(lattice_blocks(l)) + (S.check.S ? 1 : 0)), dim3(256), 0, s, l, S,
                       done);
}
void launch_lattice_rowinfo(const LatticeOpArgs& l, double* dinv, float* dinv32, double* part, double* lam,
                            hipStream_t s) {
    const int nb = int(lattice_blocks(l));
    hipLaunchKernelGGL(k_lattice_rowinfo, dim3(nb), dim3(256), 0, s, l, dinv, dinv32, part);
    hipLaunchKernelGGL(k_mg_max, dim3(1), dim3(256), 0, s, part, nb, lam);
}
void launch_perm_nodes(int64_t n_nodes, const int32_t* map, const double* src, double* dst, int scatter,
                       hipStream_t s) {
    hipLaunchKernelGGL(k_perm_nodes, dim3(mg_blocks(n_nodes, 256)), dim3(256), 0, s, n_nodes, map, src, dst, scatter);
}
void launch_mg_pre_init(const MGLevelArgs& L, const double* src, const int32_t* rank_of_lat, const CGCheck& check,
                        const int* done, hipStream_t s) {
    const dim3 g(mg_grid(L.n_nodes * L.nav) + (check.S ? 1 : 0));
    if (L.planar) hipLaunchKernelGGL(k_mg_pre_init32, dim3(mg_grid(L.n_nodes * L.nav)), dim3(256), 0, s, L, done);
    else if (L.dinvb) hipLaunchKernelGGL(k_mg_pre_init_blk5, g, dim3(256), 0, s, L, check, done);
    else hipLaunchKernelGGL(k_mg_pre_init, g, dim3(256), 0, s, L, src, rank_of_lat, check, done);
}
void launch_mg_block_dinv5(const MGLevelArgs& L, float* dinvb, hipStream_t s) {
    hipLaunchKernelGGL(k_mg_block_dinv5, dim3(mg_blocks(L.n_nodes, 256)), dim3(256), 0, s, L, dinvb);
}
void launch_mg_to_stencil(const MGLevelArgs& L, float* sten, hipStream_t s) {
    hipLaunchKernelGGL(k_mg_to_stencil, dim3(mg_blocks(L.n_nodes, 256)), dim3(256), 0, s, L, sten);
}
void launch_mg_gather_stencil3(const MGLevelArgs& L, const int32_t* rank_of_lat, const uint8_t* kpos, float* sten,
                               hipStream_t s) {
    hipLaunchKernelGGL(k_mg_gather_stencil3, dim3(mg_blocks(L.n_nodes, 256)), dim3(256), 0, s, L, rank_of_lat, kpos,
                       sten);
}
void launch_mg_stencil(const MGLevelArgs& L, const float* sten, int mode, int step, const double* din, double* dout,
                       const int* done, hipStream_t s) {
    hipLaunchKernelGGL(k_mg_stencil, dim3(mg_blocks(L.n_nodes, kStenNodes)), dim3(3 * kStenNodes), 0, s, L, sten, mode, step, din,
                       dout, done);
}
void launch_mg_to_stencil27(const MGLevelArgs& L, float* sten, hipStream_t s) {
    hipLaunchKernelGGL(k_mg_to_stencil27, dim3(mg_blocks(L.n_nodes, 256)), dim3(256), 0, s, L, sten);
}
void launch_mg_gather_stencil(const MGLevelArgs& L, const int32_t* rank_of_lat, const uint8_t* kpos, float* sten,
                              hipStream_t s) {
    hipLaunchKernelGGL(k_mg_gather_stencil, dim3(mg_blocks(L.n_nodes, 256)), dim3(256), 0, s, L, rank_of_lat, kpos,
                       sten);
}
void launch_mg_stencil_rank(const MGLevelArgs& L, const float* sten, int mode, int step, const double* din,
                            double* dout, const int* done, hipStream_t s) {
    if (L.val16)
        hipLaunchKernelGGL(k_mg_stencil_heat<uint16_t>, dim3(mg_blocks(L.n_nodes, 256)), dim3(256), 0, s, L, L.val16,
                           mode, step, din, dout, done);
    else
        hipLaunchKernelGGL(k_mg_stencil_heat<float>, dim3(mg_blocks(L.n_nodes, 256)), dim3(256), 0, s, L, sten, mode,
                           step, din, dout, done);
}
void launch_sten27_to_f16(int64_t n, const float* sten, uint16_t* sten16, float* srow, hipStream_t s) {
    hipLaunchKernelGGL(k_sten27_to_f16, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, n, sten, sten16, srow);
}
void launch_perm_rank_lat(int64_t n_nodes, int nav, const int32_t* rank_of_lat, const double* src, double* dst,
                          int to_lat, const int* done, hipStream_t s) {
    hipLaunchKernelGGL(k_perm_rank_lat, dim3(mg_blocks(n_nodes * nav, 256)), dim3(256), 0, s, n_nodes, nav,
                       rank_of_lat, src, dst, to_lat, done);
}
void launch_mg_combine_rank(int64_t n_nodes, int nav, const int32_t* rank_of_lat, const double* x0,
                            const double* dlast, double* out, const int* done, hipStream_t s) {
    hipLaunchKernelGGL(k_mg_combine_rank, dim3(mg_blocks(n_nodes * nav, 256)), dim3(256), 0, s, n_nodes, nav,
                       rank_of_lat, x0, dlast, out, done);
}
void launch_to_f16_rows(int64_t n_nodes, int nav, const int64_t* blk_ptr, const double* val, uint16_t* val16,
                        float* rs16, hipStream_t s) {
    if (nav != 5) return;
    hipLaunchKernelGGL(k_to_f16_rows<5>, dim3(unsigned((n_nodes * 5 + 255) / 256)), dim3(256), 0, s, n_nodes, blk_ptr,
                       val, val16, rs16);
}
void launch_mg_bsr(const MGLevelArgs& L, int mode, int step, const double* din, double* dout, const int* done,
                   hipStream_t s) {
    const unsigned g = unsigned(nb_grid(L.n_nodes));
    if (L.nav == 5) {
        if (L.val16)
            hipLaunchKernelGGL((k_mg_bsr<uint16_t, 5>), dim3(g), dim3(256), 0, s, L, L.val16, mode, step, din, dout,
                               done);
        else if (L.val32)
            hipLaunchKernelGGL((k_mg_bsr<float, 5>), dim3(g), dim3(256), 0, s, L, L.val32, mode, step, din, dout, done);
        else
            hipLaunchKernelGGL((k_mg_bsr<double, 5>), dim3(g), dim3(256), 0, s, L, L.val, mode, step, din, dout, done);
    } else if (L.nav == 1) {
        if (L.val32)
            hipLaunchKernelGGL((k_mg_bsr<float, 1>), dim3(g), dim3(256), 0, s, L, L.val32, mode, step, din, dout, done);
        else
            hipLaunchKernelGGL((k_mg_bsr<double, 1>), dim3(g), dim3(256), 0, s, L, L.val, mode, step, din, dout, done);
    } else {
        if (L.val32)
            hipLaunchKernelGGL((k_mg_bsr<float, 3>), dim3(g), dim3(256), 0, s, L, L.val32, mode, step, din, dout, done);
        else
            hipLaunchKernelGGL((k_mg_bsr<double, 3>), dim3(g), dim3(256), 0, s, L, L.val, mode, step, din, dout, done);
    }
}
void launch_mg_restrict(const MGLevelArgs& F, const MGLevelArgs& C, const int* done, hipStream_t s) {
    const dim3 g(mg_blocks(C.n_nodes * C.nav, 256));
    const int fl = F.planar ? FL_PLANAR : F.rank_of_lat ? FL_RANK : FL_LAT;
    if (F.dim == 2) {
        if (fl == FL_RANK) hipLaunchKernelGGL((k_mg_restrict<2, 5, FL_RANK>), g, dim3(256), 0, s, F, C, done);
        else hipLaunchKernelGGL((k_mg_restrict<2, 5, FL_LAT>), g, dim3(256), 0, s, F, C, done);
    } else if (F.nav == 1) {
        if (fl == FL_RANK) hipLaunchKernelGGL((k_mg_restrict<3, 1, FL_RANK>), g, dim3(256), 0, s, F, C, done);
        else hipLaunchKernelGGL((k_mg_restrict<3, 1, FL_LAT>), g, dim3(256), 0, s, F, C, done);
    } else {
        if (fl == FL_PLANAR) hipLaunchKernelGGL((k_mg_restrict<3, 3, FL_PLANAR>), g, dim3(256), 0, s, F, C, done);
        else if (fl == FL_RANK) hipLaunchKernelGGL((k_mg_restrict<3, 3, FL_RANK>), g, dim3(256), 0, s, F, C, done);
        else hipLaunchKernelGGL((k_mg_restrict<3, 3, FL_LAT>), g, dim3(256), 0, s, F, C, done);
    }
}
void launch_mg_prolong(const MGLevelArgs& F, const MGLevelArgs& C, const double* dlast, const int* done,
                       hipStream_t s) {
    const dim3 g(mg_blocks(F.n_nodes * F.nav, 256));
    const int fl = F.planar ? FL_PLANAR : F.rank_of_lat ? FL_RANK : FL_LAT;
    if (F.dim == 2) {
        if (fl == FL_RANK) hipLaunchKernelGGL((k_mg_prolong<2, 5, FL_RANK>), g, dim3(256), 0, s, F, C, dlast, done);
        else hipLaunchKernelGGL((k_mg_prolong<2, 5, FL_LAT>), g, dim3(256), 0, s, F, C, dlast, done);
    } else if (F.nav == 1) {
        if (fl == FL_RANK) hipLaunchKernelGGL((k_mg_prolong<3, 1, FL_RANK>), g, dim3(256), 0, s, F, C, dlast, done);
        else hipLaunchKernelGGL((k_mg_prolong<3, 1, FL_LAT>), g, dim3(256), 0, s, F, C, dlast, done);
    } else {
        if (fl == FL_PLANAR)
            hipLaunchKernelGGL((k_mg_prolong<3, 3, FL_PLANAR>), g, dim3(256), 0, s, F, C, dlast, done);
        else if (fl == FL_RANK)
            hipLaunchKernelGGL((k_mg_prolong<3, 3, FL_RANK>), g, dim3(256), 0, s, F, C, dlast, done);
        else hipLaunchKernelGGL((k_mg_prolong<3, 3, FL_LAT>), g, dim3(256), 0, s, F, C, dlast, done);
    }
}
void launch_mg_coarse_solve(int n, const double* Ainv, const double* r, double* x, const int* done,
                            hipStream_t s) {
    hipLaunchKernelGGL(k_mg_coarse_solve, dim3(mg_blocks(n, 4)), dim3(256), 0, s, n, Ainv, r, x, done);
}
void launch_pcg_update(const CGArgs& c, hipStream_t s) {
    hipLaunchKernelGGL(k_pcg_update, dim3(c.nvec), dim3(256), 0, s, c);
}
void launch_pcg_update_lat(const CGArgs& c, const MGLevelArgs& L, hipStream_t s) {
    hipLaunchKernelGGL(k_pcg_update_lat, dim3(c.nvec), dim3(256), 0, s, c, L);
}
void launch_pcg_p(const CGArgs& c, const float* z, int n, int first, hipStream_t s) {
    hipLaunchKernelGGL(k_pcg_p<float>, dim3(c.nvec), dim3(256), 0, s, c, z, n, first);
}
void launch_pcg_p(const CGArgs& c, const double* z, int n, int first, hipStream_t s) {
    hipLaunchKernelGGL(k_pcg_p<double>, dim3(c.nvec), dim3(256), 0, s, c, z, n, first);
}
void launch_pcg_rz(const CGArgs& c, const double* x0, const double* dlast, hipStream_t s) {
    hipLaunchKernelGGL(k_pcg_rz, dim3(c.nvec), dim3(256), 0, s, c, x0, dlast);
}
void launch_pcg_rz_rank(const CGArgs& c, int nav, const int32_t* rank_of_lat, const double* x0, const double* dlast,
                        hipStream_t s) {
    hipLaunchKernelGGL(k_pcg_rz_rank, dim3(c.nvec), dim3(256), 0, s, c, nav, rank_of_lat, x0, dlast);
}
void launch_mg_combine(int64_t n, const double* x0, const double* dlast, double* out, const int* done,
                       hipStream_t s) {
    hipLaunchKernelGGL(k_mg_combine, dim3(mg_grid(n)), dim3(256), 0, s, n, x0, dlast, out, done);
}
void launch_pcg_start(const CGArgs& c, const double* b, double tol2, int max_it, hipStream_t s) {
    hipLaunchKernelGGL(k_pcg_start, dim3(c.nvec), dim3(256), 0, s, c, b);
    hipLaunchKernelGGL(k_pcg_start_scalars, dim3(1), dim3(256), 0, s, c, tol2, max_it);
}
void launch_pcg_recheck(const CGArgs& c, hipStream_t s) {
    hipLaunchKernelGGL(k_pcg_start, dim3(c.nvec), dim3(256), 0, s, c, c.r);
    hipLaunchKernelGGL(k_pcg_recheck, dim3(1), dim3(256), 0, s, c);
}

}  // namespace mastg
