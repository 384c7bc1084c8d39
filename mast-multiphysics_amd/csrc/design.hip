// Element-wise design space of a mesh: the density filter, the material
// volume and its gradient, and the optimality-criteria update -- the steps of
// a SIMP topology-optimisation loop after the design evaluation.
//
// Filter: MAST::FilterBase (src/level_set/filter_base.cpp:35-142, 244-420)
// over the points that carry the design variables.  MAST filters a nodal
// level-set field; the configurations here carry one density per element, so
// the points are the element centroids:
//     rho~_e = sum_{f : |c_e - c_f| <= r} (r - d_ef) rho_f / sum_f (r - d_ef).
// The neighbour lists are built once on the host (a bucket grid of cell size
// r instead of MAST's all-pairs / k-d tree search; same sets) and kept on the
// device as a CSR of unnormalised weights a_ef = r - d_ef with the row sums
// S_e (on structured meshes as the few distinct rows, see k_filter_pattern);
// the relation is symmetric, so the transpose (the chain rule of a
// sensitivity, dJ/drho_f = sum_e a_ef / S_e dJ/drho~_e) is the same gather
// over row f with the input scaled by 1/S_e.  Both are deterministic gathers
// (no atomics).
//
// Volume: V = sum_e V_e rho_e, dV/drho_e = V_e (examples/structural/example_6/
// example_6.cpp:714-791 with element densities; V_e the element volume, or
// area for a plate whose design variable is its thickness).
//
// Optimality-criteria step (the standard SIMP update; MAST's examples drive
// external optimisers through src/optimization/*, whose algorithms are not in
// the reference): rho_new = clamp(rho B_e^(1/2) lambda^(-1/2), max(rho_min,
// rho - m), min(1, rho + m)), B_e = -dC/drho_e / dV/drho_e, with lambda such
// that V(rho_new) = vf V_total.  The multiplier is found on the device by
// multi-section: each pass evaluates the volume at 64 candidates spread
// logarithmically over the current bracket in one sweep of the elements and
// keeps the sub-interval that holds the root (7 passes narrow 60 decades to a
// relative width ~3e-11), with no host round trip between passes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <unordered_map>
#include <vector>

#include "device_util.h"
#include "hip_lock.h"
#include "mastg/mastg.h"

using namespace mastg;

namespace {

constexpr int kOcCand = 64;                // candidates per multi-section pass: one per lane
constexpr int kOcPasses = 7;
constexpr int kOcWaves = 8;                // waves per work-group of the candidate sweep
constexpr int kOcBlocks = 256;             // its work-groups (and k_vdot's) at most: one per CU
constexpr double kOcLo = 1e-30, kOcHi = 1e30;   // the first bracket
// distinct filter rows (column offsets and weights) kept in place of the CSR
constexpr int kMaxPatterns = 4096;
constexpr int kPatBatch = 16;
constexpr int64_t kMaxPatternEntries = int64_t(1) << 19;

// neighbours of a filter row: weights, and columns less the row's
struct alignas(64) FilterBatch {
    double a[kPatBatch];
    int32_t off[kPatBatch];
};

struct Buf {
    void* p = nullptr;
    size_t bytes = 0;
    ~Buf() {
        if (p) {
            HipLock l(hip_mutex());
            (void)hipFree(p);
        }
    }
    template <class T> T* as() const { return static_cast<T*>(p); }
};

}  // namespace

struct mastg_design {
    int64_t n = 0;          // elements (design variables)
    double radius = 0;
    double v_total = 0;
    std::string err;
    hipStream_t stream = nullptr;
    Buf row_ptr, col, a, inv_s, vol, part, bracket, tmp_in, tmp_out, tmp_dc, tmp_dv, scal;
    Buf pat_rows, wave_pat, pat;            // filter rows by pattern (in place of row_ptr, col, a)
    int n_waves = 0;                        // 0: the CSR
    double* h_pin = nullptr;
    int64_t nnz = 0;
};

namespace {

int dfail(mastg_design* d, int code, const std::string& m) {
    if (d) d->err = m;
    return code;
}

#define DHIPC(d, expr)                                                                   \
    do {                                                                                 \
        hipError_t _e = (expr);                                                          \
        if (_e != hipSuccess)                                                            \
            return dfail((d), MASTG_ERR_DEVICE, std::string(#expr " failed: ") + hipGetErrorString(_e)); \
    } while (0)

int dalloc(mastg_design* d, Buf& b, size_t bytes) {
    if (b.p && b.bytes >= bytes) return MASTG_OK;
    HipLock l(hip_mutex());
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    if (hipMalloc(&b.p, std::max<size_t>(bytes, 8)) != hipSuccess) {
        b.p = nullptr;
        return dfail(d, MASTG_ERR_OOM, "hipMalloc of " + std::to_string(bytes) + " bytes failed");
    }
    b.bytes = bytes;
    return MASTG_OK;
}

template <class T>
int upload(mastg_design* d, Buf& b, const std::vector<T>& v) {
    int rc = dalloc(d, b, v.size() * sizeof(T));
    if (rc) return rc;
    HipLock l(hip_mutex());
    DHIPC(d, hipMemcpy(b.p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return MASTG_OK;
}

// Finds the rows that are copies of one another: the same column offsets, and
// weights that agree to tol.
struct RowPatterns {
    double tol;
    std::vector<int32_t> ptr{0};                 // pattern k: batches ptr[k] .. ptr[k + 1] of pat
    std::vector<FilterBatch> pat;
    std::unordered_map<uint64_t, std::vector<std::pair<double, int32_t>>> known;   // by their offsets' hash: weights' sum, number
    int32_t last = -1;                           // the row before's

    bool same(int32_t k, int64_t e, const int32_t* col, const double* a, size_t m) const {
        const size_t b = size_t(ptr[size_t(k)]), nb = (m + kPatBatch - 1) / kPatBatch;
        if (size_t(ptr[size_t(k) + 1]) - b != nb) return false;
        for (size_t i = 0; i < m; i += kPatBatch) {
            const FilterBatch& P = pat[b + i / kPatBatch];
            const size_t q = std::min(m - i, size_t(kPatBatch));
            bool ok = true;
            for (size_t j = 0; j < q; j++)
                ok &= (P.off[j] == int32_t(col[i + j] - e)) & (std::fabs(P.a[j] - a[i + j]) <= tol);
            // (the rest of the last batch: this row is no shorter than the pattern)
            for (size_t j = q; j < size_t(kPatBatch); j++) ok &= P.a[j] == 0.0;
            if (!ok) return false;
        }
        return true;
    }
    // the number of row e's pattern (m columns and weights, their sum), a new one
    // when there is none; -1 once there are too many
    int32_t find(int64_t e, const int32_t* col, const double* a, size_t m, double sum) {
        if (last >= 0 && same(last, e, col, a, m)) return last;
        uint64_t h = m;                          // of the column offsets (no chain of products)
        for (size_t i = 0; i < m; i++) h += uint64_t(int64_t(col[i] - e)) * (2 * i + 1);
        std::vector<std::pair<double, int32_t>>& alike = known[h];
        const double near = double(m) * (tol + 4.5e-16 * sum);   // sums of weights within tol, rounded m times
        for (const auto& k : alike)
            if (std::fabs(k.first - sum) <= near && same(k.second, e, col, a, m)) return last = k.second;
        const size_t nb = (m + kPatBatch - 1) / kPatBatch;
        if (int64_t(ptr.size()) > kMaxPatterns || int64_t(pat.size() + nb) * kPatBatch > kMaxPatternEntries) return -1;
        last = int32_t(ptr.size()) - 1;
        alike.push_back({sum, last});
        pat.resize(pat.size() + nb, FilterBatch{});
        for (size_t i = 0; i < m; i++) {
            FilterBatch& P = pat[size_t(ptr[size_t(last)]) + i / kPatBatch];
            P.a[i % kPatBatch] = a[i];
            P.off[i % kPatBatch] = int32_t(col[i] - e);
        }
        ptr.push_back(int32_t(pat.size()));
        return last;
    }
};

// Whether the filter by patterns takes less time than by its CSR of nnz entries,
// in units of 10 ps (both directions together).  The CSR streams its entries:
// 0.58 each.  By patterns a wave's gather of one neighbour costs 8, or about one
// for each line of memory its 64 rows lie in beyond 10 (rows that a mesh graded
// along x scatters; ordinary ones lie in 5 to 20), whether its lanes hold rows or
// padding, and a row's batches wait for each other: 2.5 us a batch of the longest
// pattern.  Both forms measured (by patterns / CSR, us, there and back together):
// 16^3 cells with 67 neighbours a row 27 / 13, each row its own pattern 47 / 14;
// 32^3 35 / 23, 40^3 29 / 36, 48^3 44 / 61, 96x48x48 53 / 108, the same graded
// along x 230 / 109, along z 50 / 109; with 19 neighbours 32^3 15 / 12, 40^3
// 14 / 14, 48^3 16 / 20, 96x48x48 21 / 40; 5x200x200 with 65 neighbours 46 / 89.
int64_t pattern_budget(int64_t nnz, int64_t longest_row) {   // what the waves' gathers may cost
    return int64_t(0.58 * double(nnz)) - 250000 * ((longest_row + kPatBatch - 1) / kPatBatch);
}
int64_t pattern_wave_cost(int64_t batches, const int32_t* rows) {   // 64 rows, ascending, -1 past the last
    int64_t lines = 0, last = -1;
    for (int l = 0; l < 64; l++)
        if (rows[l] >= 0 && rows[l] / 16 != last) {
            lines++;
            last = rows[l] / 16;
        }
    return batches * kPatBatch * std::max<int64_t>(8, lines - 10);
}

// element volume (hex8, 2x2x2 Gauss: exact for the trilinear map's Jacobian)
// or area (quad4, 2x2 Gauss, in the plane of its nodes' first two coordinates
// after projecting on the element's own plane: |dx/dxi x dx/deta|)
double hex8_volume(const double X[8][3]) {
    const double g = 0.57735026918962576451;
    double V = 0;
    for (int q = 0; q < 8; q++) {
        const double xi = (q & 1) ? g : -g, eta = (q & 2) ? g : -g, zeta = (q & 4) ? g : -g;
        double J[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        for (int n = 0; n < 8; n++) {
            const double sx = (n == 1 || n == 2 || n == 5 || n == 6) ? 1.0 : -1.0;
            const double sy = (n == 2 || n == 3 || n == 6 || n == 7) ? 1.0 : -1.0;
            const double sz = (n >= 4) ? 1.0 : -1.0;
            const double fx = 0.5 * (1 + sx * xi), fy = 0.5 * (1 + sy * eta), fz = 0.5 * (1 + sz * zeta);
            const double d[3] = {0.5 * sx * fy * fz, fx * 0.5 * sy * fz, fx * fy * 0.5 * sz};
            for (int i = 0; i < 3; i++)
                for (int r = 0; r < 3; r++) J[i * 3 + r] += X[n][i] * d[r];
        }
        V += J[0] * (J[4] * J[8] - J[7] * J[5]) + J[3] * (J[7] * J[2] - J[1] * J[8]) + J[6] * (J[1] * J[5] - J[4] * J[2]);
    }
    return V;
}

double quad4_area(const double X[4][3]) {
    const double g = 0.57735026918962576451;
    double A = 0;
    for (int q = 0; q < 4; q++) {
        const double xi = (q & 1) ? g : -g, eta = (q & 2) ? g : -g;
        double t0[3] = {0, 0, 0}, t1[3] = {0, 0, 0};
        for (int n = 0; n < 4; n++) {
            const double sx = (n == 1 || n == 2) ? 1.0 : -1.0, sy = (n >= 2) ? 1.0 : -1.0;
            const double dxi = 0.25 * sx * (1 + sy * eta), deta = 0.25 * sy * (1 + sx * xi);
            for (int i = 0; i < 3; i++) {
                t0[i] += X[n][i] * dxi;
                t1[i] += X[n][i] * deta;
            }
        }
        const double c0 = t0[1] * t1[2] - t0[2] * t1[1], c1 = t0[2] * t1[0] - t0[0] * t1[2],
                     c2 = t0[0] * t1[1] - t0[1] * t1[0];
        A += std::sqrt(c0 * c0 + c1 * c1 + c2 * c2);
    }
    return A;
}

// ------------------------------------------------------------------ kernels --
// out_e = s_e sum_k a_k in[col_k] over row e; transpose: the input scaled by
// 1/S of its own row (inv_s), s_e = 1.  LANES lanes per row, fixed order.
template <int LANES>
__global__ __launch_bounds__(256) void k_filter(int64_t n, const int64_t* __restrict__ rp,
                                                const int32_t* __restrict__ col, const double* __restrict__ a,
                                                const double* __restrict__ inv_s, const double* __restrict__ in,
                                                double* __restrict__ out, int transpose) {
    const int64_t row = (int64_t(blockIdx.x) * 256 + threadIdx.x) / LANES;
    const int lane = threadIdx.x % LANES;
    double s = 0.0;
    if (row < n) {
        for (int64_t k = rp[row] + lane; k < rp[row + 1]; k += LANES) {
            const int32_t f = col[k];
            s += a[k] * (transpose ? in[f] * inv_s[f] : in[f]);
        }
    }
#pragma unroll
    for (int m = LANES / 2; m >= 1; m >>= 1) s += __shfl_xor(s, m, LANES);
    if (row < n && lane == 0) out[row] = transpose ? s : s * inv_s[row];
}

// The filter of a mesh whose rows are copies of a few patterns (a structured
// mesh: the interior row and its cut-off forms near the boundary): row e's
// columns are e + off_k and its weights a_k of its pattern, so a row costs its
// number and the neighbours' values (through L1 / L2) instead of 12 bytes of
// CSR per neighbour.  A thread per row, rows grouped so that the 64 of a wave
// share their pattern (rows[] pads a group's last wave with -1): offsets and
// weights are scalar loads, and the neighbours' values of the interior rows
// nearly contiguous runs.  96x48x48 elements, 81 neighbours: 18 us (transpose,
// which gathers 1/S too, 32 us) against 55 us for the CSR; in row order, where
// two waves of three mix patterns and read the entries per lane, 22 and 34 us.
// Bound by the gathers (a 512-byte run per neighbour and wave): the
// entries come in batches (three wide scalar loads, then kPatBatch gathers in
// flight), a pattern padded to whole batches with weights 0 on its own row, whose
// products are left out (0 times an infinity there would be no number).
__global__ __launch_bounds__(256) void k_filter_pattern(int n_waves, const int32_t* __restrict__ rows,
                                                        const int2* __restrict__ wave_pat,
                                                        const FilterBatch* __restrict__ pat,
                                                        const double* __restrict__ inv_s,
                                                        const double* __restrict__ in, double* __restrict__ out,
                                                        int transpose) {
    const int w = __builtin_amdgcn_readfirstlane(int(xcd_block(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6)));
    if (w >= n_waves) return;
    const uint32_t row = uint32_t(rows[int64_t(w) * 64 + (threadIdx.x & 63)]);
    if (int32_t(row) < 0) return;
    const int2 k01 = wave_pat[w];   // the pattern's batches
    double s = 0.0;
    if (transpose) {
        for (int k = k01.x; k < k01.y; k++) {
            const FilterBatch P = pat[k];
            double t[kPatBatch], u[kPatBatch];
#pragma unroll
            for (int j = 0; j < kPatBatch; j++) {
                t[j] = (in + P.off[j])[row];
                u[j] = (inv_s + P.off[j])[row];
            }
#pragma unroll
            for (int j = 0; j < kPatBatch; j++) s = fma(P.a[j], P.a[j] != 0.0 ? t[j] * u[j] : 0.0, s);
        }
        out[row] = s;
    } else {
        for (int k = k01.x; k < k01.y; k++) {
            const FilterBatch P = pat[k];
            double t[kPatBatch];
#pragma unroll
            for (int j = 0; j < kPatBatch; j++) t[j] = (in + P.off[j])[row];
#pragma unroll
            for (int j = 0; j < kPatBatch; j++) s = fma(P.a[j], P.a[j] != 0.0 ? t[j] : 0.0, s);
        }
        out[row] = s * inv_s[row];
    }
}

__global__ __launch_bounds__(256) void k_vdot(int64_t n, const double* __restrict__ a, const double* __restrict__ b,
                                              double* __restrict__ part) {
    double s = 0.0;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) s += a[i] * b[i];
    block_sum_store(s, part, blockIdx.x);
}

__global__ __launch_bounds__(256) void k_vreduce(const double* __restrict__ part, int np, double* __restrict__ out) {
    const double s = reduce_partials(part, np);
    if (threadIdx.x == 0) *out = s;
}

// the update of one density: clamp(t lam^(-1/2)), t = rho B^(1/2)
__device__ __forceinline__ double oc_clamp(double t, double lo, double hi, double lam_m12) {
    return fmin(hi, fmax(lo, t * lam_m12));
}

// candidate c of the bracket [lo, hi] (log-spaced interior points)
__device__ __forceinline__ double oc_cand(double lo, double hi, int c) {
    const double t = double(c + 1) / double(kOcCand + 1);
    return exp(log(lo) + t * (log(hi) - log(lo)));
}

// Volume at every candidate multiplier: partial sums part[block][candidate].
// A lane owns a candidate and its wave walks a share of the elements through
// LDS (every lane reads the same element: broadcasts), so no sum crosses lanes
// and an element's rho B^(1/2) and move limits are formed once per pass, not
// once per candidate.  br = null: the first bracket.  Bound by latency (the
// bracket from the launch before, the elements); 96x48x48 elements: 10 us
// per pass against 24 us in the form that swept the elements eight times for
// 8 candidates each, and 14 us with 192 candidates (and one pass fewer).
__global__ __launch_bounds__(64 * kOcWaves) void k_oc_sweep(int64_t n, const double* __restrict__ rho,
                                                  const double* __restrict__ dc, const double* __restrict__ dv,
                                                  const double* __restrict__ br, double move, double rho_min,
                                                  double* __restrict__ part) {
    __shared__ double4 el[kOcWaves][64];      // t, lo, hi, v of each wave's next elements
    __shared__ double red[kOcWaves][kOcCand];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // contiguous equal shares: every wave of the grid ends at once
    const int64_t nw = int64_t(gridDim.x) * kOcWaves, per = (n + nw - 1) / nw;
    const int64_t e0 = (int64_t(blockIdx.x) * kOcWaves + wave) * per, e1 = min(n, e0 + per);
    auto load = [&](int64_t i, double& r, double& c, double& v) {
        const int64_t j = i < e1 ? i : 0;     // past the share: any element, weighted 0 below
        r = rho[j];
        c = dc[j];
        v = dv[j];
    };
    double r, c, v;
    load(e0 + lane, r, c, v);                 // in flight while the candidate is formed
    const double lam = 1.0 / sqrt(oc_cand(br ? br[0] : kOcLo, br ? br[1] : kOcHi, lane));
    double s = 0.0;
    double4* __restrict__ w = el[wave];
    for (int64_t e = e0; e < e1; e += 64) {
        w[lane] = {r * sqrt(fmax(0.0, -c) / v), fmax(rho_min, r - move), fmin(1.0, r + move), v};
        if (e + 64 < e1) load(e + 64 + lane, r, c, v);
        wave_exchange();
        const int m = int(min(int64_t(64), e1 - e));
#pragma unroll 8
        for (int j = 0; j < m; j++) {
            const double4 q = w[j];
            s = fma(q.w, oc_clamp(q.x, q.y, q.z, lam), s);
        }
        wave_exchange();                      // the batch is read; the next overwrites it
    }
    red[wave][lane] = s;
    __syncthreads();
    if (wave == 0) {
        double t = 0.0;
#pragma unroll
        for (int j = 0; j < kOcWaves; j++) t += red[j][lane];
        part[int64_t(blockIdx.x) * kOcCand + lane] = t;
    }
}

// Candidate volumes (fixed-order sums over the sweep's work-groups) and the
// next bracket: the root of V(lambda) = target lies between the last candidate
// above the target and the first one at or below it (V is non-increasing in
// lambda).  One work-group: thread (c, j) sums every kOcSlices-th partial of
// candidate c, reads coalesced over c (one wave summing each candidate's
// partials in turn took 57 us).
constexpr int kOcSlices = 16;
__global__ __launch_bounds__(kOcCand * kOcSlices) void k_oc_select(const double* __restrict__ part, int nb,
                                                                   double target, int first_pass,
                                                                   double* __restrict__ br) {
    __shared__ double vol[kOcSlices][kOcCand];
    const int c = threadIdx.x % kOcCand, j = threadIdx.x / kOcCand;
    const double lo = first_pass ? kOcLo : br[0], hi = first_pass ? kOcHi : br[1];
    double s = 0.0;
    // batches of loads in flight (an absent partial reads the first, weighted 0)
    for (int b = j; b < nb; b += 16 * kOcSlices) {
        double t[16];
#pragma unroll
        for (int i = 0; i < 16; i++) t[i] = part[int64_t(b + i * kOcSlices < nb ? b + i * kOcSlices : j) * kOcCand + c];
#pragma unroll
        for (int i = 0; i < 16; i++) s += b + i * kOcSlices < nb ? t[i] : 0.0;
    }
    vol[j][c] = s;
    __syncthreads();
    if (j == 0) {   // one wave, a candidate per lane
#pragma unroll
        for (int k = 1; k < kOcSlices; k++) s += vol[k][c];
        const uint64_t below = __ballot(s <= target);
        const int first = below ? __builtin_ctzll(below) : kOcCand;
        if (c < 2) {   // lane 0 the lower end, lane 1 the upper
            const int k = first - 1 + c;
            br[c] = k < 0 ? lo : k == kOcCand ? hi : oc_cand(lo, hi, k);
        }
    }
}

__global__ __launch_bounds__(256) void k_oc_final(int64_t n, const double* __restrict__ rho,
                                                  const double* __restrict__ dc, const double* __restrict__ dv,
                                                  const double* __restrict__ br, double move, double rho_min,
                                                  double* __restrict__ out) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const double r = rho[i], t = r * sqrt(fmax(0.0, -dc[i]) / dv[i]);
    out[i] = oc_clamp(t, fmax(rho_min, r - move), fmin(1.0, r + move), 1.0 / sqrt(br[1]));
}

int64_t blocks_of(int64_t n, int per) { return std::max<int64_t>(1, (n + per - 1) / per); }

// out = the filter (or its transpose) of in
void filter_launch(mastg_design* d, const double* in, double* out, int transpose) {
    const int64_t n = d->n;
    if (d->n_waves > 0)
        hipLaunchKernelGGL(k_filter_pattern, dim3(blocks_of(d->n_waves, 4)), dim3(256), 0, d->stream, d->n_waves,
                           d->pat_rows.as<int32_t>(), d->wave_pat.as<int2>(), d->pat.as<FilterBatch>(), d->inv_s.as<double>(), in, out, transpose);
    else
        hipLaunchKernelGGL(k_filter<8>, dim3(blocks_of(n * 8, 256)), dim3(256), 0, d->stream, n,
                           d->row_ptr.as<int64_t>(), d->col.as<int32_t>(), d->a.as<double>(), d->inv_s.as<double>(),
                           in, out, transpose);
}

// host or device input -> device pointer (staged in `tmp` for host data)
int stage(mastg_design* d, const double* src, int where, Buf& tmp, const double** out) {
    if (where == MASTG_DEVICE) {
        *out = src;
        return MASTG_OK;
    }
    int rc = dalloc(d, tmp, size_t(d->n) * sizeof(double));
    if (rc) return rc;
    DHIPC(d, hipMemcpyAsync(tmp.p, src, size_t(d->n) * sizeof(double), hipMemcpyHostToDevice, d->stream));
    *out = tmp.as<double>();
    return MASTG_OK;
}

}  // namespace

extern "C" {

int mastg_design_create(const mastg_problem_desc* desc, double radius, mastg_design** out) {
    if (!desc || !out || !desc->xyz || !desc->conn || desc->n_elems <= 0) return MASTG_ERR_INVALID;
    if (!(radius > 0)) return MASTG_ERR_INVALID;
    const int npe = desc->physics == MASTG_QUAD4_MINDLIN ? 4 : 8;
    auto* d = new mastg_design;
    d->n = desc->n_elems;
    d->radius = radius;
    const int64_t n = d->n;
    // centroids and volumes
    std::vector<double> c(size_t(n) * 3), vol(n);
    double lo[3] = {1e300, 1e300, 1e300};
    for (int64_t e = 0; e < n; e++) {
        double X[8][3];
        for (int a = 0; a < npe; a++) {
            const int32_t nd = desc->conn[e * npe + a];
            if (nd < 0 || nd >= desc->n_nodes) {
                delete d;
                return MASTG_ERR_INVALID;
            }
            for (int i = 0; i < 3; i++) X[a][i] = desc->xyz[int64_t(nd) * 3 + i];
        }
        for (int i = 0; i < 3; i++) {
            double s = 0;
            for (int a = 0; a < npe; a++) s += X[a][i];
            c[e * 3 + i] = s / npe;
            lo[i] = std::min(lo[i], c[e * 3 + i]);
        }
        vol[e] = npe == 8 ? hex8_volume(X) : quad4_area(reinterpret_cast<const double(*)[3]>(X));
        d->v_total += vol[e];
    }
    // neighbours within the radius: bucket grid of cell size r
    auto key = [&](int64_t e, int k) { return int64_t(std::floor((c[e * 3 + k] - lo[k]) / radius)); };
    int64_t nb[3] = {1, 1, 1};
    for (int64_t e = 0; e < n; e++)
        for (int k = 0; k < 3; k++) nb[k] = std::max(nb[k], key(e, k) + 1);
    std::unordered_map<int64_t, std::vector<int32_t>> bucket;
    bucket.reserve(size_t(n));
    auto bid = [&](int64_t i, int64_t j, int64_t k) { return (k * nb[1] + j) * nb[0] + i; };
    for (int64_t e = 0; e < n; e++) bucket[bid(key(e, 0), key(e, 1), key(e, 2))].push_back(int32_t(e));
    std::vector<int64_t> rp(n + 1, 0);
    std::vector<int32_t> col;
    std::vector<double> a, inv_s(n);
    std::vector<std::pair<int32_t, double>> row;
    // rows are copies of one another when their weights agree to the rounding
    // that the centroids' coordinates carry into their distances, but to 2^-40 of
    // the radius wherever the mesh lies: far from the origin that rounding is as
    // large as a mesh's own differences, and its rows stay their own
    double cmax = 0.0;
    for (const double x : c) cmax = std::max(cmax, std::fabs(x));
    const double tol = std::min(16.0 * 2.220446049250313e-16 * cmax, std::ldexp(radius, -40));
    int64_t longest = 0;
    for (int64_t e = 0; e < n; e++) {
        row.clear();
        const int64_t ki = key(e, 0), kj = key(e, 1), kk = key(e, 2);
        for (int64_t z = kk - 1; z <= kk + 1; z++)
            for (int64_t y = kj - 1; y <= kj + 1; y++)
                for (int64_t x = ki - 1; x <= ki + 1; x++) {
                    if (x < 0 || y < 0 || z < 0 || x >= nb[0] || y >= nb[1] || z >= nb[2]) continue;
                    auto it = bucket.find(bid(x, y, z));
                    if (it == bucket.end()) continue;
                    for (int32_t f : it->second) {
                        const double dx = c[e * 3] - c[f * 3], dy = c[e * 3 + 1] - c[f * 3 + 1],
                                     dz = c[e * 3 + 2] - c[f * 3 + 2];
                        const double dist = std::sqrt(dx * dx + dy * dy + dz * dz);
                        if (dist <= radius) row.emplace_back(f, radius - dist);
                    }
                }
        std::sort(row.begin(), row.end());
        double s = 0;
        for (auto& p : row) {
            col.push_back(p.first);
            a.push_back(p.second);
            s += p.second;
        }
        inv_s[e] = 1.0 / s;
        rp[e + 1] = int64_t(col.size());
        longest = std::max(longest, int64_t(row.size()));
    }
    d->nnz = rp[n];
    // the rows' patterns, looked for while they can be the faster form (a
    // pattern fills a wave at least, at the least cost of its gathers)
    int64_t budget = pattern_budget(d->nnz, longest), least = 0;
    bool patterns = budget > 0;
    RowPatterns rows{tol};
    std::vector<int32_t> pat_id(patterns ? size_t(n) : 0);
    const std::vector<int32_t>& pat_ptr = rows.ptr;
    for (int64_t e = 0; e < n && patterns; e++) {
        const size_t seen = rows.pat.size();
        pat_id[size_t(e)] = rows.find(e, &col[size_t(rp[e])], &a[size_t(rp[e])], size_t(rp[e + 1] - rp[e]),
                                     1.0 / inv_s[size_t(e)]);
        least += int64_t(rows.pat.size() - seen) * kPatBatch * 8;
        patterns = pat_id[size_t(e)] >= 0 && least < budget;
    }
    // grouped by pattern, a wave of 64 at a time; kept where that is the faster form
    std::vector<int32_t> pat_rows;
    std::vector<int2> wave_pat;
    if (patterns) {
        std::vector<int64_t> first(pat_ptr.size(), 0);
        for (const int32_t k : pat_id) first[size_t(k) + 1]++;
        for (size_t k = 1; k < first.size(); k++) {
            for (int64_t w = 0; w < (first[k] + 63) / 64; w++) wave_pat.push_back(make_int2(pat_ptr[k - 1], pat_ptr[k]));
            first[k] = int64_t(wave_pat.size()) * 64;
        }
        pat_rows.assign(wave_pat.size() * 64, -1);
        for (int64_t e = 0; e < n; e++) pat_rows[size_t(first[size_t(pat_id[size_t(e)])]++)] = int32_t(e);
        for (size_t w = 0; w < wave_pat.size(); w++)
            budget -= pattern_wave_cost(wave_pat[w].y - wave_pat[w].x, &pat_rows[w * 64]);
        patterns = budget > 0;
    }
    d->n_waves = patterns ? int(wave_pat.size()) : 0;
    {
        HipLock l(hip_mutex());
        if (hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess ||
            hipHostMalloc((void**)&d->h_pin, 8 * sizeof(double)) != hipSuccess) {
            mastg_design_destroy(d);
            return MASTG_ERR_DEVICE;
        }
    }
    int rc;
    if (patterns)
        (rc = upload(d, d->pat_rows, pat_rows)) || (rc = upload(d, d->wave_pat, wave_pat)) ||
            (rc = upload(d, d->pat, rows.pat));
    else
        (rc = upload(d, d->row_ptr, rp)) || (rc = upload(d, d->col, col)) || (rc = upload(d, d->a, a));
    if (rc || (rc = upload(d, d->inv_s, inv_s)) || (rc = upload(d, d->vol, vol)) ||
        (rc = dalloc(d, d->part, size_t(kOcCand) * kOcBlocks * sizeof(double))) ||
        (rc = dalloc(d, d->bracket, 2 * sizeof(double))) ||
        (rc = dalloc(d, d->scal, sizeof(double))) ||
        (rc = dalloc(d, d->tmp_out, size_t(n) * sizeof(double)))) {
        mastg_design_destroy(d);
        return rc;
    }
    *out = d;
    return MASTG_OK;
}

int mastg_design_destroy(mastg_design* d) {
    if (!d) return MASTG_OK;
    {
        HipLock l(hip_mutex());
        if (d->stream) (void)hipStreamSynchronize(d->stream);
        if (d->h_pin) (void)hipHostFree(d->h_pin);
    }
    hipStream_t s = d->stream;
    delete d;
    if (s) {
        HipLock l(hip_mutex());
        (void)hipStreamDestroy(s);
    }
    return MASTG_OK;
}

const char* mastg_design_last_error(const mastg_design* d) { return d ? d->err.c_str() : ""; }

int mastg_design_info(const mastg_design* d, int64_t* n_elems, int64_t* nnz, double* v_total) {
    if (!d) return MASTG_ERR_INVALID;
    if (n_elems) *n_elems = d->n;
    if (nnz) *nnz = d->nnz;
    if (v_total) *v_total = d->v_total;
    return MASTG_OK;
}

int mastg_design_filter(mastg_design* d, const double* in, double* out, int transpose, int where) {
    if (!d || !in || !out || (where != MASTG_HOST && where != MASTG_DEVICE)) return MASTG_ERR_INVALID;
    const double* din;
    int rc = stage(d, in, where, d->tmp_in, &din);
    if (rc) return rc;
    double* dout = where == MASTG_DEVICE ? out : d->tmp_out.as<double>();
    filter_launch(d, din, dout, transpose ? 1 : 0);
    DHIPC(d, hipGetLastError());
    if (where == MASTG_HOST)
        DHIPC(d, hipMemcpyAsync(out, dout, size_t(d->n) * sizeof(double), hipMemcpyDeviceToHost, d->stream));
    DHIPC(d, hipStreamSynchronize(d->stream));
    return MASTG_OK;
}

int mastg_design_volume(mastg_design* d, const double* rho, int where, double* volume, double* dvol) {
    if (!d || !rho || (where != MASTG_HOST && where != MASTG_DEVICE)) return MASTG_ERR_INVALID;
    const double* dr;
    int rc = stage(d, rho, where, d->tmp_in, &dr);
    if (rc) return rc;
    if (volume) {
        const int nb = int(std::min<int64_t>(kOcBlocks, blocks_of(d->n, 256)));
        hipLaunchKernelGGL(k_vdot, dim3(nb), dim3(256), 0, d->stream, d->n, d->vol.as<double>(), dr,
                           d->part.as<double>());
        hipLaunchKernelGGL(k_vreduce, dim3(1), dim3(256), 0, d->stream, d->part.as<double>(), nb,
                           d->scal.as<double>());
        DHIPC(d, hipGetLastError());
        DHIPC(d, hipMemcpyAsync(d->h_pin, d->scal.p, sizeof(double), hipMemcpyDeviceToHost, d->stream));
    }
    if (dvol)
        DHIPC(d, hipMemcpyAsync(dvol, d->vol.p, size_t(d->n) * sizeof(double),
                                where == MASTG_HOST ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice, d->stream));
    DHIPC(d, hipStreamSynchronize(d->stream));
    if (volume) *volume = d->h_pin[0];
    return MASTG_OK;
}

int mastg_design_oc_update(mastg_design* d, const double* rho, const double* dc, const double* dv,
                           double volfrac, double move, double rho_min, double* rho_new, int where,
                           double* lambda) {
    if (!d || !rho || !dc || !dv || !rho_new || (where != MASTG_HOST && where != MASTG_DEVICE))
        return MASTG_ERR_INVALID;
    if (!(volfrac > 0 && volfrac <= 1) || !(move > 0) || !(rho_min >= 0 && rho_min < 1))
        return dfail(d, MASTG_ERR_INVALID, "volume fraction in (0, 1], move > 0, 0 <= rho_min < 1");
    const double* dr;
    const double* ddc;
    const double* ddv;
    int rc;
    if ((rc = stage(d, rho, where, d->tmp_in, &dr)) || (rc = stage(d, dc, where, d->tmp_dc, &ddc)) ||
        (rc = stage(d, dv, where, d->tmp_dv, &ddv)))
        return rc;
    const double target = volfrac * d->v_total;
    const int nb = int(std::min<int64_t>(kOcBlocks, blocks_of(d->n, 64 * kOcWaves)));
    for (int p = 0; p < kOcPasses; p++) {
        hipLaunchKernelGGL(k_oc_sweep, dim3(nb), dim3(64 * kOcWaves), 0, d->stream, d->n, dr, ddc, ddv,
                           p ? d->bracket.as<double>() : nullptr, move, rho_min, d->part.as<double>());
        hipLaunchKernelGGL(k_oc_select, dim3(1), dim3(kOcCand * kOcSlices), 0, d->stream, d->part.as<double>(), nb,
                           target, p ? 0 : 1, d->bracket.as<double>());
    }
    double* dout = where == MASTG_DEVICE ? rho_new : d->tmp_out.as<double>();
    hipLaunchKernelGGL(k_oc_final, dim3(blocks_of(d->n, 256)), dim3(256), 0, d->stream, d->n, dr, ddc, ddv,
                       d->bracket.as<double>(), move, rho_min, dout);
    DHIPC(d, hipGetLastError());
    if (where == MASTG_HOST)
        DHIPC(d, hipMemcpyAsync(rho_new, dout, size_t(d->n) * sizeof(double), hipMemcpyDeviceToHost, d->stream));
    DHIPC(d, hipMemcpyAsync(d->h_pin, d->bracket.p, 2 * sizeof(double), hipMemcpyDeviceToHost, d->stream));
    DHIPC(d, hipStreamSynchronize(d->stream));
    if (lambda) *lambda = d->h_pin[1];
    return MASTG_OK;
}

}  // extern "C"
