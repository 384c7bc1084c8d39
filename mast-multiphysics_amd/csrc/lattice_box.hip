// The hex8 problem level of the multigrid solver on a lattice of equal
// axis-aligned boxes: the FP64 CG product and the FP32 Chebyshev smoothing
// steps, matrix-free.
//
// In the sum / difference modes of a cell's 8 nodes (per axis: sum or
// difference of the two ends) the box's class matrix is nearly diagonal: the
// derivative along an axis takes a mode with that axis' difference to the one
// without it, and different modes are orthogonal, so of the 24 x 24 entries 45
// remain (BoxOp, 33 distinct): a cell costs 45 multiply-adds and its share of
// the transforms instead of 576.
//
// A wave covers 62 consecutive points of an x-y plane (lane l is point
// 62 w + l - 1 of the plane, x fastest, rows run on) and marches NL layers in
// z.  A lane forms the cells (i, j-1) and (i, j) of its point in each layer:
// x + 1 from the next lane, y +- 1 from memory (rows just read, L1 / L2), the
// layer below carried in registers; of a cell's forces it keeps the two
// corners on its row and hands the right one to the next lane.  No LDS, no
// barrier; all layers' loads are in flight at once.  Points outside the lattice
// are clamped into it, cells outside have the scale 0.  Every sum has a fixed
// order.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "device_util.h"
#include "kernels.h"

namespace mastg {

namespace {

// the value of the next / previous lane of the wave (0 past its ends)
__device__ __forceinline__ float lane_next(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_prev(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_next(double v) {
    const uint64_t u = uint64_t(__double_as_longlong(v));
    const uint32_t lo = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(u)), 0x130, 0xf, 0xf, true));
    const uint32_t hi = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(u >> 32)), 0x130, 0xf, 0xf, true));
    return __longlong_as_double((long long)((uint64_t(hi) << 32) | lo));
}
__device__ __forceinline__ double lane_prev(double v) {
    const uint64_t u = uint64_t(__double_as_longlong(v));
    const uint32_t lo = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(u)), 0x138, 0xf, 0xf, true));
    const uint32_t hi = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(u >> 32)), 0x138, 0xf, 0xf, true));
    return __longlong_as_double((long long)((uint64_t(hi) << 32) | lo));
}

constexpr int kOut = 62;   // points per wave
enum { MX = 1, MY = 2, MZ = 4 };

// the points of a wave: lane l's plane index, its lattice row and column, and
// the layers k0 .. k0 + NL - 1
struct BoxPoint {
    uint32_t pc;      // plane index, clamped into the plane
    int i, j, k0;
    bool out;         // the lane owns a point
    bool inside;      // its plane index needed no clamping
};

__device__ __forceinline__ BoxPoint box_point(const LatticeOpArgs& O, uint32_t w, int lane, int nl) {
    const uint32_t nxp = uint32_t(O.nx + 1), plane = nxp * uint32_t(O.ny + 1), npw = (plane + kOut - 1) / kOut;
    const uint32_t chunk = w / npw;
    const int p = int((w - chunk * npw) * kOut) + lane - 1;
    BoxPoint b;
    b.inside = p >= 0 && p < int(plane);
    b.pc = uint32_t(min(max(p, 0), int(plane) - 1));
    b.j = int(b.pc / nxp);
    b.i = int(b.pc - uint32_t(b.j) * nxp);
    b.k0 = int(chunk) * nl;
    b.out = lane >= 1 && lane <= kOut && b.inside && b.k0 <= O.nz;
    return b;
}

// what a lane reads: the values of its three rows in NL + 2 layers, the scales
// of its two cells in NL + 1
template <typename T, int NL>
struct BoxIn {
    T u[NL + 2][3][3], s[NL + 1][2];
};

template <typename T, int NL>
__device__ __forceinline__ void box_load(const LatticeOpArgs& O, const T* __restrict__ sE, const T* __restrict__ in,
                                         int64_t n_lat, const BoxPoint& b, BoxIn<T, NL>& B) {
    const uint32_t nxp = uint32_t(O.nx + 1), plane = nxp * uint32_t(O.ny + 1);
    const uint32_t rows[3] = {b.pc - (b.j > 0 ? nxp : 0u), b.pc, b.pc + (b.j < O.ny ? nxp : 0u)};
#pragma unroll
    for (int q = 0; q < NL + 2; q++) {
        const uint32_t base = uint32_t(min(max(b.k0 - 1 + q, 0), O.nz)) * plane;
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) B.u[q][r][c] = (in + c * n_lat)[base + rows[r]];
    }
    const bool hx = b.inside && b.i < O.nx;
    const int ci = min(b.i, O.nx - 1);
#pragma unroll
    for (int q = 0; q < NL + 1; q++) {
        const int kc = b.k0 - 1 + q, kz = min(max(kc, 0), O.nz - 1);
        const bool hz = hx && kc >= 0 && kc < O.nz;
        const T a0 = sE[ci + O.nx * (max(b.j - 1, 0) + O.ny * kz)];
        const T a1 = sE[ci + O.nx * (min(b.j, O.ny - 1) + O.ny * kz)];
        B.s[q][0] = hz && b.j > 0 ? a0 : T(0);
        B.s[q][1] = hz && b.j < O.ny ? a1 : T(0);
    }
}

// y[q][c] = (A u) at the lane's point in layers k0 + q, before the constraint
// convention (u there: B.u[q + 1][1][c])
template <typename T, int NL>
__device__ __forceinline__ void box_rows(const BoxOp<T>& K, const BoxIn<T, NL>& B, T (&y)[NL][3]) {
    // planar modes of a layer: per cell row (A: j-1, B: j) and component 0, X, Y, XY
    T lo[2][3][4], h0[3], hX[3];
#pragma unroll
    for (int q = 0; q < NL + 2; q++) {
        T up[2][3][4];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            T sx[3], dx[3];
#pragma unroll
            for (int r = 0; r < 3; r++) {
                const T n = lane_next(B.u[q][r][c]);
                sx[r] = n + B.u[q][r][c];
                dx[r] = n - B.u[q][r][c];
            }
#pragma unroll
            for (int r = 0; r < 2; r++) {
                up[r][c][0] = sx[r] + sx[r + 1];
                up[r][c][MX] = dx[r] + dx[r + 1];
                up[r][c][MY] = sx[r + 1] - sx[r];
                up[r][c][MX | MY] = dx[r + 1] - dx[r];
            }
        }
        if (q > 0) {   // the cells between layers q - 1 and q
            T l0[3] = {T(0), T(0), T(0)}, lX[3] = {T(0), T(0), T(0)}, p0[3], pX[3];
#pragma unroll
            for (int c = 0; c < 3; c++) p0[c] = pX[c] = T(0);
#pragma unroll
            for (int r = 0; r < 2; r++) {
                T m[3][8], g[3][8];
                const T sc = B.s[q - 1][r];
#pragma unroll
                for (int c = 0; c < 3; c++) {
#pragma unroll
                    for (int a = 0; a < 4; a++) {
                        if (a) m[c][a] = sc * (up[r][c][a] + lo[r][c][a]);
                        m[c][a | MZ] = sc * (up[r][c][a] - lo[r][c][a]);
                    }
                }
#pragma unroll
                for (int c = 0; c < 3; c++)
#pragma unroll
                    for (int a = 1; a < 8; a++) g[c][a] = K.d[c][a] * m[c][a];
                // pairs (x, y), (x, z), (y, z); kb: the third axis
#pragma unroll
                for (int pr = 0; pr < 3; pr++) {
                    const int ca = pr == 2 ? 1 : 0, cb = pr == 0 ? 1 : 2, kb = 1 << (3 - ca - cb);
                    const int ma = 1 << ca, mb = 1 << cb;
                    g[ca][ma] += K.l0[pr] * m[cb][mb];
                    g[cb][mb] += K.l0[pr] * m[ca][ma];
                    g[ca][ma | kb] += K.l1[pr] * m[cb][mb | kb];
                    g[cb][mb | kb] += K.l1[pr] * m[ca][ma | kb];
                    g[ca][mb] += K.m0[pr] * m[cb][ma];
                    g[cb][ma] += K.m0[pr] * m[ca][mb];
                    g[ca][mb | kb] += K.m1[pr] * m[cb][ma | kb];
                    g[cb][ma | kb] += K.m1[pr] * m[ca][mb | kb];
                }
                // forces on the lane's row: cell A's upper, cell B's lower y corners
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const T f = r == 0 ? g[c][MY] : -g[c][MY];
                    const T e = r == 0 ? g[c][MZ] + g[c][MY | MZ] : g[c][MZ] - g[c][MY | MZ];
                    const T t = r == 0 ? g[c][MX] + g[c][MX | MY] : g[c][MX] - g[c][MX | MY];
                    const T v = r == 0 ? g[c][MX | MZ] + g[c][7] : g[c][MX | MZ] - g[c][7];
                    l0[c] += f - e;
                    p0[c] += f + e;
                    lX[c] += t - v;
                    pX[c] += t + v;
                }
            }
            if (q >= 2) {   // layer q - 1 = k0 + q - 2 is complete
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    const T a0 = h0[c] + l0[c], aX = hX[c] + lX[c];
                    y[q - 2][c] = (a0 - aX) + lane_prev(a0 + aX);
                }
            }
#pragma unroll
            for (int c = 0; c < 3; c++) {
                h0[c] = p0[c];
                hX[c] = pX[c];
            }
        }
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int a = 0; a < 4; a++) lo[r][c][a] = up[r][c][a];
    }
}

// cells that exist at a lattice point
__device__ __forceinline__ int cells_at(const LatticeOpArgs& O, int i, int j, int k) {
    return ((i > 0) + (i < O.nx)) * ((j > 0) + (j < O.ny)) * ((k > 0) + (k < O.nz));
}

// y = A x (FP64, the CG product) and partial sums of x.y
template <int NL>
__global__ __launch_bounds__(256) void k_box_apply(LatticeOpArgs O, const double* __restrict__ in,
                                                   double* __restrict__ out, double* __restrict__ part,
                                                   const int* __restrict__ done) {
    if (done && *done) return;
    const int64_t plane = int64_t(O.nx + 1) * (O.ny + 1), n_lat = plane * (O.nz + 1);
    const uint32_t w = uint32_t(xcd_block(blockIdx.x, gridDim.x)) * 4 + (threadIdx.x >> 6);
    const BoxPoint b = box_point(O, w, threadIdx.x & 63, NL);
    double y[NL][3], dsum = 0.0;
    BoxIn<double, NL> B;
    box_load<double, NL>(O, O.sE_cell, in, n_lat, b, B);
    box_rows<double, NL>(O.box, B, y);
    if (b.out)
#pragma unroll
        for (int q = 0; q < NL; q++) {
            if (b.k0 + q > O.nz) break;
            const int64_t p = (b.k0 + q) * plane + b.pc;
            const int m = O.nodecon[p], cnt = cells_at(O, b.i, b.j, b.k0 + q);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const double x = B.u[q + 1][1][c], v = (m >> c) & 1 ? cnt * x : y[q][c];
                out[c * n_lat + p] = v;
                dsum = fma(v, x, dsum);
            }
        }
    block_sum_store(dsum, part, blockIdx.x);
}

// one pass of the FP32 smoothing (see LatSmooth); the last work-group, if
// S.check, only decides on convergence
template <int NL>
__global__ __launch_bounds__(256) void k_box_smooth(LatticeOpArgs O, LatSmooth S, const int* __restrict__ done) {
    unsigned nb = gridDim.x;
    if (S.check.S) {
        nb--;
        if (blockIdx.x == nb) {
            pcg_check_block(S.check);
            return;
        }
    }
    if (vcycle_done(S.check, done)) return;
    const int64_t plane = int64_t(O.nx + 1) * (O.ny + 1), n_lat = plane * (O.nz + 1);
    const uint32_t w = uint32_t(xcd_block(blockIdx.x, nb)) * 4 + (threadIdx.x >> 6);
    const BoxPoint b = box_point(O, w, threadIdx.x & 63, NL);
    BoxIn<float, NL> B;
    box_load<float, NL>(O, O.sE_cell32, S.x, n_lat, b, B);
    // the epilogue's own values arrive while the rows are computed
    float rb[NL][3], dv[NL][3], xp[NL][3];
    int con[NL];
#pragma unroll
    for (int q = 0; q < NL; q++) {
        const int64_t p = min(b.k0 + q, O.nz) * plane + b.pc;
        con[q] = O.nodecon[p];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            rb[q][c] = S.b[c * n_lat + p];
            dv[q][c] = S.res ? 0.f : S.dinv[c * n_lat + p];
            xp[q][c] = S.xp ? S.xp[c * n_lat + p] : 0.f;
        }
    }
    const LatCoef cf = lat_coef(S);
    float y[NL][3];
    box_rows<float, NL>(O.box32, B, y);
    double rz = 0.0;
    if (b.out)
#pragma unroll
        for (int q = 0; q < NL; q++) {
            if (b.k0 + q > O.nz) break;
            const int64_t p = (b.k0 + q) * plane + b.pc;
            const float cnt = float(cells_at(O, b.i, b.j, b.k0 + q));
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float x = B.u[q + 1][1][c], yv = (con[q] >> c) & 1 ? cnt * x : y[q][c];
                rz += lat_point(S, cf, c * n_lat + p, yv, x, rb[q][c], dv[q][c], xp[q][c]);
            }
        }
    if (S.part) block_sum_store(rz, S.part, blockIdx.x);
}

// Layers per wave: 2 where that leaves the chip at least this many waves
// (marching shares the layers' loads and one of three cell layers), else 1.
// Smoothing pass at 128x64x64: 12.7 us with 2 layers, 13.6 with 1, 14.1 with 4;
// 96x48x48 7.6 with 4, 7.9 with 2 and 1; 64x32x32 5.5 with 1, 7.4 with 4, the waves
// in flight hiding the latency.  The general form (576 multiply-adds per point,
// seven vectors per pass) took 23.8 us at 128x64x64 and 8.2 us at 8x4x4 (now 4.4);
// the FP64 product 31 us (now 16) and 9.5 (4.3).  At 128x64x64 the five vectors
// (33 MB) alone take 6.5 us and the arithmetic as long, of which the one round
// of waves overlaps little.
constexpr int64_t kBoxWaves = 2048;
int64_t box_waves(const LatticeOpArgs& l, int nl) {
    const int64_t plane = int64_t(l.nx + 1) * (l.ny + 1);
    return ((plane + kOut - 1) / kOut) * ((l.nz + nl) / nl);
}
int box_layers(const LatticeOpArgs& l) { return box_waves(l, 2) >= kBoxWaves ? 2 : 1; }
unsigned box_blocks(const LatticeOpArgs& l, int nl) { return unsigned((box_waves(l, nl) + 3) / 4); }

}  // namespace

bool box_operator(const double* Khat, BoxOp<double>& op) {
    // Kt = H Khat H^T / 64, H the 8 x 8 sum / difference transform of the nodes
    static const int corner[8][3] = {{0, 0, 0}, {1, 0, 0}, {1, 1, 0}, {0, 1, 0}, {0, 0, 1}, {1, 0, 1}, {1, 1, 1}, {0, 1, 1}};
    auto sign = [&](int m, int n) {
        double s = 1.0;
        for (int d = 0; d < 3; d++)
            if ((m >> d) & 1) s *= corner[n][d] ? 1.0 : -1.0;
        return s;
    };
    double Kt[8][3][8][3] = {}, big = 0.0;
    for (int m = 0; m < 8; m++)
        for (int n = 0; n < 8; n++)
            for (int v = 0; v < 3; v++)
                for (int w = 0; w < 3; w++) {
                    double s = 0.0;
                    for (int a = 0; a < 8; a++)
                        for (int b = 0; b < 8; b++) s += sign(m, a) * sign(n, b) * Khat[(a * 8 + b) * 9 + v * 3 + w];
                    Kt[m][v][n][w] = s / 64.0;
                    big = std::max(big, std::fabs(s) / 64.0);
                }
    op = BoxOp<double>{};
    bool keep[8][3][8][3] = {};
    auto take = [&](int m, int v, int n, int w) {
        keep[m][v][n][w] = keep[n][w][m][v] = true;
        return 0.5 * (Kt[m][v][n][w] + Kt[n][w][m][v]);
    };
    for (int v = 0; v < 3; v++)
        for (int m = 1; m < 8; m++) op.d[v][m] = take(m, v, m, v);
    for (int pr = 0; pr < 3; pr++) {
        const int a = pr == 2 ? 1 : 0, b = pr == 0 ? 1 : 2, k = 1 << (3 - a - b), ma = 1 << a, mb = 1 << b;
        op.l0[pr] = take(ma, a, mb, b);
        op.l1[pr] = take(ma | k, a, mb | k, b);
        op.m0[pr] = take(mb, a, ma, b);
        op.m1[pr] = take(mb | k, a, ma | k, b);
    }
    // the other entries vanish for an axis-aligned box, to the rounding of Khat
    for (int m = 0; m < 8; m++)
        for (int n = 0; n < 8; n++)
            for (int v = 0; v < 3; v++)
                for (int w = 0; w < 3; w++) {
                    const double x = Kt[m][v][n][w];
                    if (!std::isfinite(x) || (!keep[m][v][n][w] && std::fabs(x) > 1e-13 * big)) return false;
                }
    return big > 0.0;
}

// Against the element-wise product of matrix-free CG: a plane of a few points
// fills little of its wave, and each wave costs the same.  An iteration takes
// about 10.5 us + 1.4 ns a wave + 0.045 ns a point here and 20.4 us + 0.1 ns a
// point there; measured (here / there, us): 1x1x8000 cells 21 / 23, 1x1x12000
// 27 / 25, 1x1x40000 70 / 35, 2x2x12000 31 / 35, 2x2x30000 62 / 46, 3x3x16000
// 44 / 49, 5x5x8000 37 / 59, 45x23x23 12.7 / 23.4.
bool box_apply_pays(const LatticeOpArgs& l) {
    const int64_t points = int64_t(l.nx + 1) * (l.ny + 1) * (l.nz + 1);
    return box_waves(l, 1) <= 7600 + points / 23;
}

int64_t box_partials_most(const LatticeOpArgs& l) { return box_blocks(l, 1); }
int64_t box_partials(const LatticeOpArgs& l) { return box_blocks(l, box_layers(l)); }

void launch_box_apply(const LatticeOpArgs& l, const double* x, double* y, double* part, const int* done, hipStream_t s) {
    const int nl = box_layers(l);
    const dim3 g(box_blocks(l, nl));
    if (nl == 2) hipLaunchKernelGGL(k_box_apply<2>, g, dim3(256), 0, s, l, x, y, part, done);
    else hipLaunchKernelGGL(k_box_apply<1>, g, dim3(256), 0, s, l, x, y, part, done);
}

void launch_box_smooth(const LatticeOpArgs& l, const LatSmooth& S, const int* done, hipStream_t s) {
    const int nl = box_layers(l);
    const dim3 g(box_blocks(l, nl) + (S.check.S ? 1 : 0));
    if (nl == 2) hipLaunchKernelGGL(k_box_smooth<2>, g, dim3(256), 0, s, l, S, done);
    else hipLaunchKernelGGL(k_box_smooth<1>, g, dim3(256), 0, s, l, S, done);
}

}  // namespace mastg
