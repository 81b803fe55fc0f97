// Device code shared by the kernels of the backprojection path: wavefront
// reductions, batch descriptors, the pixel tiling and the split-precision
// phase fit.
#pragma once

#include <hip/hip_runtime.h>
#include <limits.h>

#include "bp_internal.h"

namespace bp {
namespace {

__device__ inline int wave_min_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ inline int wave_max_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ inline long long wave_sum_ll(long long v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Workgroups are dispatched round-robin over the 8 XCDs; remap group `it` of
// `ng` (it = blockIdx.x, or blockIdx.x plus multiples of a grid that is a
// multiple of 8, so that it % 8 is the XCD) so that each XCD (own L2) walks a
// contiguous run of tiles, which share pulse data.  Returns the global
// wavefront-tile index of this wavefront (4 per group).
__device__ inline int64_t group_tile(int64_t it, int64_t ng, int* lane)
{
    const int64_t per = ng / 8, rem = ng % 8;
    const int64_t xcd = it % 8, idx = it / 8;
    const int64_t lb = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
    *lane = threadIdx.x & 63;
    return lb * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// Descriptor words read through vector loads are not known to be uniform;
// readfirstlane moves them into scalar registers (every lane of the
// wavefront reads the same descriptor).
__device__ inline int64_t uniform64(int64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uint64_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// A read-only buffer read at wave-uniform indices as a constant-address-space
// pointer: its loads go through the scalar data cache into scalar registers
// (one load per wavefront, no vector memory instruction).  Only for data no
// kernel writes while the reading kernel runs.
template<class T>
__device__ inline const __attribute__((address_space(4))) T* uniform_ptr(const T* p)
{
    return (const __attribute__((address_space(4))) T*)(p);
}

// Output grid owning global wavefront tile s (s uniform across the wavefront).
__device__ inline int find_grid(const OutDesc* g, int n, int64_t s)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (uniform64(g[mid].seq_base) <= s)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Copy of descriptor i held in scalar registers.
__device__ inline OutDesc load_desc(const OutDesc* g, int i)
{
    static_assert(sizeof(OutDesc) % 4 == 0, "descriptor must be whole dwords");
    OutDesc d;
    const uint32_t* src = reinterpret_cast<const uint32_t*>(g + i);
    uint32_t* dst = reinterpret_cast<uint32_t*>(&d);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(OutDesc) / 4); ++k) dst[k] = __builtin_amdgcn_readfirstlane(src[k]);
    return d;
}

// Pixel j (0 <= j < lane_rows) of `lane` in wavefront tile `tile`.
__device__ inline bool tile_pixel(const TileMap& m, int64_t tile, int lane, int j, int64_t* row,
                                  int64_t* col)
{
    if (tile >= m.n_tiles) return false;
    const int64_t ty = tile / m.tiles_x, tx = tile % m.tiles_x;
    *row = (ty * m.tile_rows + lane / m.tile_cols) * m.lane_rows + j;
    *col = tx * m.tile_cols + lane % m.tile_cols;
    return *row < m.length && *col < m.width;
}

constexpr int kFitNodes = kFitDegree + 1;

// Chebyshev nodes cos(pi (m + 1/2) / M), M = 5
__device__ inline double fit_node(int m)
{
    return m == 0 ? 0.95105651629515353
                  : m == 1 ? 0.58778525229247314
                           : m == 2 ? 0.0 : m == 3 ? -0.58778525229247314 : -0.95105651629515353;
}

__device__ inline double readlane_f64(double x, int lane)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

__device__ inline V3 readlane_v3(V3 x, int lane)
{
    return {readlane_f64(x.x, lane), readlane_f64(x.y, lane), readlane_f64(x.z, lane)};
}

// The pulse phase of one pixel in cycles as a polynomial in j = k - kw0 over
// the window [kw0, kw1): P(j) = c_ref + sum av[i] j^i, and the range bin
// u(k) = u_ref + (P(k) - c_ref) / (fc dtau).
struct PhaseFit {
    double c_ref;          // reference phase (cycles, reduced)
    double u_ref;          // range bin at the reference phase
    double av[kFitNodes];
    double bnd;            // bins the range may move over the window, at most
};

// Degree-4 Chebyshev interpolant of the phase over [kw0, kw1) evaluated in
// FP64 and re-expanded about kw0.  tau_c: the delay at the reference pulse
// kc; gm[m]: the phase in cycles at Chebyshev node m relative to the
// reference pulse's.
__device__ inline PhaseFit fit_phase(const GeomArgs& a, int kw0, int kw1, double tau_c,
                                     const double (&gm)[kFitNodes])
{
    PhaseFit o;
    const double kc = 0.5 * ((double)kw0 + (double)(kw1 - 1));
    const double h = fmax(0.5 * (double)(kw1 - 1 - kw0), 0.5);
    constexpr int M = kFitNodes;
    // Chebyshev nodes cos(pi (m + 1/2) / M) and T_j at the nodes
    constexpr double kNode[M] = {0.95105651629515353, 0.58778525229247314, 0.0,
                                 -0.58778525229247314, -0.95105651629515353};
    // Chebyshev coefficients c_j = 2/M sum_m g_m T_j(s_m), c_0 halved,
    // with T_j(s_m) = cos(j pi (m + 1/2) / M).
    double cc[M];
#pragma unroll
    for (int j = 0; j < M; ++j) {
        double acc = 0.;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            // T_j(s_m) by the recurrence (exact to rounding at these nodes)
            double t0 = 1., t1 = kNode[m], tj = j == 0 ? 1. : kNode[m];
#pragma unroll
            for (int i = 2; i <= j; ++i) {
                tj = 2. * kNode[m] * t1 - t0;
                t0 = t1;
                t1 = tj;
            }
            acc += gm[m] * tj;
        }
        cc[j] = acc * (2.0 / M);
    }
    cc[0] *= 0.5;
    // Chebyshev -> monomial in s = (k - kc) / h: T_{j+1} = 2 s T_j - T_{j-1}
    double mono[M], tjm1[M], tj[M], tjp1[M];
#pragma unroll
    for (int n = 0; n < M; ++n) {
        mono[n] = 0.;
        tjm1[n] = 0.;
        tj[n] = 0.;
    }
    tjm1[0] = 1.;  // T_0
    tj[1] = 1.;    // T_1
    mono[0] += cc[0];
    mono[1] += cc[1];
#pragma unroll
    for (int j = 1; j < M - 1; ++j) {
#pragma unroll
        for (int n = 0; n < M; ++n) tjp1[n] = -tjm1[n] + (n > 0 ? 2.0 * tj[n - 1] : 0.);
#pragma unroll
        for (int n = 0; n < M; ++n) {
            mono[n] += cc[j + 1] * tjp1[n];
            tjm1[n] = tj[n];
            tj[n] = tjp1[n];
        }
    }
    // Reference phase (cycles, reduced) and range-bin position at s = 0.
    const double cyc_c = a.fc * tau_c;
    const double c_ref = (cyc_c - floor(cyc_c)) + mono[0];
    const double u_c = (tau_c - a.swst) / a.dtau + mono[0] / (a.fc * a.dtau);
    // Re-expand dc(s) = sum_{n>=1} mono[n] s^n about the first pulse kw0:
    // s = s0 + j / h, j = k - kw0; coefficients a_i of j^i.
    const double s0 = ((double)kw0 - kc) / h;
    const double ih = 1.0 / h;
#pragma unroll
    for (int i = 0; i < M; ++i) {
        double acc = 0., binom = 1.;  // C(n, i) s0^(n - i), n = i..4
        double sp0 = 1.;
#pragma unroll
        for (int n = i; n < M; ++n) {
            if (n >= 1) acc += mono[n] * binom * sp0;
            // next n: C(n+1, i) = C(n, i) (n + 1) / (n + 1 - i)
            binom = binom * (double)(n + 1) / (double)(n + 1 - i);
            sp0 *= s0;
        }
        o.av[i] = acc;
    }
    double ihp = 1.;
#pragma unroll
    for (int i = 1; i < M; ++i) {
        ihp *= ih;
        o.av[i] *= ihp;
    }
    o.c_ref = c_ref;
    o.u_ref = u_c;
    const double inv_k = 1.0 / (a.fc * a.dtau);
    // |s| <= 1 on the window, so |dc| <= sum |mono[n]|
    o.bnd = inv_k * (fabs(mono[1]) + fabs(mono[2]) + fabs(mono[3]) + fabs(mono[4]));
    return o;
}

}  // namespace
}  // namespace bp
