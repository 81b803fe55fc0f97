// Split-precision coherent sum by line interpolation (gfx950, wave64).
//
// Adjacent output lines of one range column sum nearly the same terms: over
// a chunk of 64 pulses, line i's sum, with its own phase at the chunk's centre
// taken out, is a smooth function of the line index.  So a strip of up to 64
// output lines x 64 range columns is focused from a few of its lines (nodes):
//
//   strip_fit    per pixel the FP64 phase polynomial over the strip's pulses,
//                and whether the strip qualifies (below)
//   strip_nodes  per chunk the sums of the node lines (6 for strips of up to
//                32 lines, 8 above), demodulated at the chunk's centre
//   strip_lines  per line and chunk: Lagrange interpolation of the node sums
//                over the line index, the line's own FP64 phase at the
//                centre, an FP64 sum; and the corrections of the next paragraph
//   strip_ends   the pulses at the ends of the aperture that only some of the
//                strip's lines integrate, line by line
//   strip_sum    the partial sums of a pixel, added in a fixed order; strips
//                where one is not finite are left to the pixel-by-pixel sum
//
// The interpolated pulse sample s(u) is only piecewise smooth in the range
// position u: where u enters the next bin, a tap of the (truncated) kernel
// leaves and another enters.  The node sums therefore follow one cell of u per
// column and pulse, the reference line's, with the kernel's taps continued
// smoothly past its ends (each tap's weight is one degree-7 polynomial of the
// position in the cell, up to 0.33 bin past it); where a line's own cell
// differs, the difference of the two tap sets -- the tap that entered less the
// continued tap that left -- is added line by line.  u moves over the
// aperture by the range curvature alone, and equally for all columns when the
// output range spacing is the input's, so that this happens for about |y|
// pulses per crossed bin on a line y lines off the reference: 8 % of the
// pulse-line pairs at 850 km, 7.5 km/s and 4,000 pulses.
//
// Measured for 4096 x 4096 pixels of 16384 x 16384 pulses (width 8), with VALU
// instructions per pixel-pulse: fit 0.88 ms (0.1), nodes 7.4 (5.0), lines 9.6
// (3.3), ends 2.3 (0.9), sum 0.17, together 20.3 ms against 88.0 (45) pixel by
// pixel, at 1e-5 instead of 1.2e-4 relative error on noise.  The nodes are bound
// by VALU issue (1.27 instructions per SIMD and four cycles); the lines by what
// they read, their records for every chunk and the node sums in each of a strip's
// 16 line groups (36 GB past L2 at 3.8 TB/s; VALU 0.60); the ends and the fit by
// latency (0.67 and 0.26).  A 32 x 32 tile takes 0.24 ms against 2.3 for the whole
// call, because its chunks run in parallel where a wavefront walked the whole
// aperture of its pixels.  64 lines per strip and 64 pulses per chunk: strips
// of 32 lines cost the nodes 9 instructions per pixel-pulse instead of 5 and halve
// the corrections (the same sum), chunks of 32 pulses double the lines' part.
//
// Pixels whose tropospheric delays differ sit up to 2e-3 bin off the positions
// the nodes interpolate (their phases are their own); the sums of the samples'
// derivatives at four of the nodes, in such strips only, bring that in to
// first order (24 % more work in the nodes).
//
// A strip qualifies when every pixel integrates 64 pulses, no tap leaves the
// range line, lines differ by at most 0.33 bin and the phase bounds of
// bp_internal.h, the nodes reproduce every line's phase slope, and the
// columns' fractional bins agree (corrections would otherwise be needed at
// most pulses); the others take the pixel-by-pixel sum.
#include <float.h>

#include "bp_device.h"

namespace bp {
namespace {

constexpr int kLineThreads = 256;
constexpr int kCoreSegs = 4;                 // chunk ranges per line group
constexpr int kSegs = kCoreSegs + 2;         // and the aperture's two ends
constexpr int kGroupLines = 4;               // lines per wavefront of strip_lines
constexpr int kMaxGroups = kStripLines / kGroupLines;
constexpr float kMaskMargin = 0.001f;        // bins: lines between two nodes may stand
                                             // out a little (curvature of u)

// Strip t of the batch (numbered column by column inside each grid).
struct Strip {
    int64_t info, rec;     // its StripInfo; its first pixel's record
    int64_t row0, col0, width, pix0;
    int h, cols;           // output lines and columns
    float2* out;
};

__device__ inline int find_strip_grid(const OutDesc* g, int n, int64_t t)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (uniform64(g[mid].strip_seq) <= t)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

__device__ inline Strip load_strip(const OutDesc& d, int64_t t)
{
    Strip s;
    const int64_t k = t - d.strip_seq;
    const int64_t x = k / d.strips_y, y = k - x * d.strips_y;
    s.info = d.strip_info + y * d.strips_x + x;
    s.row0 = y * d.strip_rows;
    s.col0 = x * 64;
    s.width = d.map.width;
    s.h = (int)min((int64_t)d.strip_rows, d.map.length - s.row0);
    s.cols = (int)min((int64_t)64, d.map.width - s.col0);
    s.pix0 = s.row0 * s.width + s.col0;
    s.rec = d.rec_base + s.pix0;
    s.out = d.out;
    return s;
}

// Node lines of a strip of h lines: Chebyshev points stretched to its ends.
__device__ inline int node_line(int nodes, int h, int n)
{
    constexpr double x8[8] = {-1.0, -0.84775906502257351, -0.56645449735052189,
                              -0.19891236737965800, 0.19891236737965800, 0.56645449735052189,
                              0.84775906502257351, 1.0};
    constexpr double x6[6] = {-1.0, -0.73205080756887729, -0.26794919243112270,
                              0.26794919243112270, 0.73205080756887729, 1.0};
    return (int)rint(0.5 * (h - 1) * (1.0 + (nodes == 8 ? x8[n] : x6[n])));
}

__device__ inline int strip_nodes_of(int h) { return h <= 32 ? 6 : 8; }

// The nodes whose derivative sums are kept.
__device__ inline int slope_node(int nodes, int n)
{
    return nodes == 8 ? (n < 2 ? 1 + 2 * n : 2 * n) : (n == 0 ? 0 : n == 3 ? 5 : n + 1);
}

// Lagrange weight, for line i, of the n-th of `count` lines x(0) <= x(1) <=
// ... (equal lines count once).
template<class X>
__device__ inline float lagrange(int count, X&& x, int i, int n)
{
    const int xn = x(n);
    if (n > 0 && x(n - 1) == xn) return 0.f;
    double num = 1.0, den = 1.0;   // products of integers below 64^7: exact
    int prev = -1;
    for (int m = 0; m < count; ++m) {
        const int xm = x(m);
        if (xm != prev && xm != xn) {
            num *= (double)(i - xm);
            den *= (double)(xn - xm);
        }
        prev = xm;
    }
    return (float)(num / den);
}

__device__ inline float node_weight(int nodes, int h, int i, int n)
{
    return lagrange(nodes, [&](int m) { return node_line(nodes, h, m); }, i, n);
}

__device__ inline float slope_weight(int nodes, int h, int i, int n)
{
    return lagrange(kSlopeNodes, [&](int m) { return node_line(nodes, h, slope_node(nodes, m)); },
                    i, n);
}

// Phase and range of one pixel about pulse kc: p(k) = b1 (k - kc) + b2 (k -
// kc)^2 cycles from the phase at kc, and the range bin there.
struct Local {
    float b1, b2;
    double u;      // range bin at kc
    double ph;     // phase at kc, cycles
};

__device__ inline Local local_phase(const PixLine& r, double j, double inv_k)
{
    Local o;
    const double dp = fma(fma(fma(r.a4, j, r.a3), j, r.a2), j, r.a1) * j;
    o.b1 = (float)fma(fma(fma(4. * r.a4, j, 3. * r.a3), j, 2. * r.a2), j, r.a1);
    o.b2 = (float)fma(fma(6. * r.a4, j, 3. * r.a3), j, r.a2);
    o.u = (double)r.ub + fma(dp, inv_k, (double)r.uf);
    o.ph = r.p0 + dp;
    return o;
}

template<int W>
struct Cell {
    // taps of cell A start at bin A + kFirst; positions in it are measured
    // from A + kCentre
    static constexpr int kFirst = W % 2 == 0 ? 1 - W / 2 : -(W / 2);
    static constexpr double kCentre = W % 2 == 0 ? 0.5 : 0.0;
    static __device__ inline int of(double u) { return (int)(W % 2 == 0 ? ceil(u) - 1. : rint(u)); }
};

// Weight polynomials of the taps combined with the taps: s(f) = sum_d q[d]
// f^d.  The kernel is even, so taps t and W - 1 - t share coefficients up to
// the sign of the odd ones.
template<int W>
__device__ inline void farrow(const float (&c)[kLineDegree + 1][kLineTaps], const float2 (&d)[W],
                              float2 (&q)[line_degree(W) + 1])
{
    constexpr int P = W / 2;
    float2 s[P], e[P];
#pragma unroll
    for (int t = 0; t < P; ++t) {
        s[t] = make_float2(d[t].x + d[W - 1 - t].x, d[t].y + d[W - 1 - t].y);
        e[t] = make_float2(d[t].x - d[W - 1 - t].x, d[t].y - d[W - 1 - t].y);
    }
#pragma unroll
    for (int k = 0; k <= line_degree(W); ++k) {
        const float2* v = k % 2 == 0 ? s : e;
        float2 r = make_float2(c[k][0] * v[0].x, c[k][0] * v[0].y);
#pragma unroll
        for (int t = 1; t < P; ++t) {
            r.x = fmaf(c[k][t], v[t].x, r.x);
            r.y = fmaf(c[k][t], v[t].y, r.y);
        }
        if (W % 2 == 1 && k % 2 == 0) {
            r.x = fmaf(c[k][P], d[P].x, r.x);
            r.y = fmaf(c[k][P], d[P].y, r.y);
        }
        q[k] = r;
    }
}

template<int D>
__device__ inline float2 farrow_eval(const float2 (&q)[D], float f)
{
    float2 r = q[D - 1];
#pragma unroll
    for (int k = D - 2; k >= 0; --k) {
        r.x = fmaf(r.x, f, q[k].x);
        r.y = fmaf(r.y, f, q[k].y);
    }
    return r;
}

// The value and the derivative with respect to f.
template<int D>
__device__ inline float2 farrow_slope(const float2 (&q)[D], float f, float2& slope)
{
    float2 r = q[D - 1], g = make_float2(0.f, 0.f);
#pragma unroll
    for (int k = D - 2; k >= 0; --k) {
        g.x = fmaf(g.x, f, r.x);
        g.y = fmaf(g.y, f, r.y);
        r.x = fmaf(r.x, f, q[k].x);
        r.y = fmaf(r.y, f, q[k].y);
    }
    slope = g;
    return r;
}

// The tap weights at d bins past the end of a cell: the tap that entered
// (inside the kernel) and the continuation of the one that left.
__device__ inline float2 end_weights(const LineArgs& a, float d)
{
    float x = a.w_in[kEndDegree], y = a.w_out[kEndDegree];
#pragma unroll
    for (int k = kEndDegree - 1; k >= 0; --k) {
        x = fmaf(x, d, a.w_in[k]);
        y = fmaf(y, d, a.w_out[k]);
    }
    return make_float2(x, y);
}

template<int W>
__device__ inline void load_taps(const char* row, uint32_t off, float2 (&d)[W])
{
    const float2* p = reinterpret_cast<const float2*>(row + off);
#pragma unroll
    for (int t = 0; t < W; ++t) d[t] = p[t];
}

// ------------------------------------------------------------------ fit

// One workgroup per strip; a wavefront holds a line (lane = column) and takes
// eight of them.
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
void strip_fit_kernel(GeomArgs a, LineArgs l)
{
    const int64_t t = blockIdx.x;
    if (t >= uniform64(a.batch->n_strips)) return;
    const OutDesc* grids = batch_grids(a.batch);
    const OutDesc d =
        load_desc(grids, find_strip_grid(grids, __builtin_amdgcn_readfirstlane(a.batch->n_grids), t));
    const Strip st = load_strip(d, t);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = min(lane, st.cols - 1);
    __shared__ int s_red[8][5];
    __shared__ int s_bad, s_slopes;
    __shared__ float s_slope[2][kStripLines][64], s_pos[2][kStripLines][64];
    __shared__ float s_weight[kStripLines][8];

    int lo = INT_MAX, hi = INT_MIN, flo = INT_MIN, fhi = INT_MAX, ok = 1;
    for (int q = 0; q < 8; ++q) {
        const int i = wave * 8 + q;
        if (i >= st.h) break;
        const PixGeom& g = a.geom[st.rec + i * st.width + col];
        ok &= g.status == kPixOk && g.kstop - g.kstart >= kStripMinPulses;
        lo = min(lo, g.kstart);
        hi = max(hi, g.kstop);
        flo = max(flo, g.kstart);
        fhi = min(fhi, g.kstop);
    }
    lo = wave_min_i(lo);
    hi = wave_max_i(hi);
    flo = wave_max_i(flo);
    fhi = wave_min_i(fhi);
    ok = wave_min_i(ok);
    if (lane == 0) {
        s_red[wave][0] = lo;
        s_red[wave][1] = hi;
        s_red[wave][2] = flo;
        s_red[wave][3] = fhi;
        s_red[wave][4] = ok;
    }
    if (threadIdx.x == 0) s_bad = s_slopes = 0;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 8; ++w) {
        lo = min(lo, s_red[w][0]);
        hi = max(hi, s_red[w][1]);
        flo = max(flo, s_red[w][2]);
        fhi = min(fhi, s_red[w][3]);
        ok &= s_red[w][4];
    }
    const int k0 = __builtin_amdgcn_readfirstlane(lo), k1 = __builtin_amdgcn_readfirstlane(hi);
    const int f0 = __builtin_amdgcn_readfirstlane(flo), f1 = __builtin_amdgcn_readfirstlane(fhi);
    const int slot0 = f0 >> l.chunk_log2;
    const int nslots = ((f1 - 1) >> l.chunk_log2) - slot0 + 1;
    if (!__builtin_amdgcn_readfirstlane(ok) || f0 >= f1 || nslots > l.slots) {
        if (threadIdx.x == 0) {
            l.info[st.info] = StripInfo{k0, k1, f0, f1, kStripLeft, 0, 0, 0};
            atomicAdd(l.n_left, 1);
        }
        return;
    }
    // platform states at the reference pulse and the Chebyshev nodes, one
    // orbit evaluation per lane on lanes 0-5 as in the pixel-by-pixel fit
    const double kc = 0.5 * ((double)k0 + (double)(k1 - 1));
    const double hw = fmax(0.5 * (double)(k1 - 1 - k0), 0.5);
    const int m = min(lane, kFitNodes);
    const double km = m == kFitNodes ? kc : kc + hw * fit_node(m);
    V3 p, v;
    orbit_interpolate<true>(a.in_orbit, a.in_t0 + km * a.in_dt, kBorderExtrapolate, &p, &v);
    // bistatic delay (r.v - c |r|) * 2 / (|v|^2 - c^2), the factor per state
    const double fac = 2. / (dot(v, v) - kC * kC);
    const double inv_k = l.inv_k;
    const int nodes = strip_nodes_of(st.h);
    {
        const int i = threadIdx.x >> 3, n = threadIdx.x & 7;
        s_weight[i][n] = n < nodes && i < st.h ? node_weight(nodes, st.h, i, n) : 0.f;
    }
    // the range bin of the strip's first column, as a base for float positions
    const double base0 = floor((d.r0 + st.col0 * d.dr - l.in_r0) * l.inv_dr);
    bool bad = false;
    for (int q = 0; q < 8; ++q) {
        const int i = wave * 8 + q;
        if (i >= st.h) break;
        const PixGeom g = a.geom[st.rec + i * st.width + col];
        const V3 x{g.x[0], g.x[1], g.x[2]};
        auto delay = [&](int n) {
            const V3 r = x - readlane_v3(p, n);
            return (dot(r, readlane_v3(v, n)) - kC * sqrt_normal(dot(r, r))) * readlane_f64(fac, n);
        };
        const double d_c = delay(kFitNodes), tau_c = g.tau_atm + d_c;
        double gm[kFitNodes];
#pragma unroll
        for (int n = 0; n < kFitNodes; ++n) gm[n] = a.fc * (delay(n) - d_c);
        const PhaseFit f = fit_phase(a, k0, k1, tau_c, gm);
        PixLine r;
        const double u0 = f.u_ref + f.av[0] * inv_k;
        r.p0 = f.c_ref + f.av[0];
        r.a1 = f.av[1];
        r.a2 = f.av[2];
        r.a3 = f.av[3];
        r.a4 = f.av[4];
        r.ub = (int)floor(u0);
        r.uf = (float)(u0 - floor(u0));
        r.kstart = g.kstart;
        r.kstop = g.kstop;
        r.du = 0.f;
        r.pad_ = 0;
        if (lane < st.cols) l.rec[st.rec + i * st.width + lane] = r;
        // every tap of the strip's lines inside the range line, two bins off
        // their own cells included
        bad |= f.u_ref - f.bnd - (a.kwidth / 2 + 4) < 0. ||
               f.u_ref + f.bnd + (a.kwidth / 2 + 4) > (double)a.nr;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const double j = (double)((e == 0 ? f0 : f1 - 1) - k0);
            const double dp = fma(fma(fma(r.a4, j, r.a3), j, r.a2), j, r.a1) * j;
            const double sl = fma(fma(fma(4. * r.a4, j, 3. * r.a3), j, 2. * r.a2), j, r.a1);
            s_slope[e][i][lane] = (float)sl;
            s_pos[e][i][lane] = (float)(u0 + dp * inv_k - (base0 + col));
            bad |= !(fabs(sl) <= kLineMaxSlope);
        }
    }
    __syncthreads();
    const int ref = st.h / 2;
    bool slopes = false;
    const float half = 0.5f * (float)(1 << l.chunk_log2);
    const float limit = nodes == 8 ? kLineBound8 : kLineBound6;
    int line[8];
#pragma unroll
    for (int n = 0; n < 8; ++n)
        line[n] = n < nodes ? __builtin_amdgcn_readfirstlane(node_line(nodes, st.h, n)) : 0;
    for (int q = 0; q < 8; ++q) {
        const int i = wave * 8 + q;
        if (i >= st.h) break;
        float w[8], off[2];
#pragma unroll
        for (int n = 0; n < 8; ++n) w[n] = s_weight[i][n];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float sl = s_slope[e][i][lane], ps = s_pos[e][i][lane];
            const float dsl = fabsf(sl - s_slope[e][ref][lane]);
            const float dps = fabsf(ps - s_pos[e][ref][lane]);
            float rs = sl, rp = ps;
#pragma unroll
            for (int n = 0; n < 8; ++n) {
                rs = fmaf(-w[n], s_slope[e][line[n]][lane], rs);
                rp = fmaf(-w[n], s_pos[e][line[n]][lane], rp);
            }
            bad |= !(dps <= kLineMaxShift) ||
                   !(6.2831853f * half * dsl + 3.1415927f * dps <= limit) ||
                   !(6.2831853f * half * fabsf(rs) <= kLineSlopeTol);
            off[e] = rp;
            // the columns' fractional bins agree (one crossing pulse per bin
            // for the whole strip)
            const float ref_pos = s_pos[e][ref][lane];
            bad |= !(fabsf(ref_pos - __shfl(ref_pos, 0, 64)) <= kLineColumnTol);
        }
        const float du = 0.5f * (off[0] + off[1]);
        bad |= !(fabsf(off[0] - off[1]) <= kLinePosTol) ||
               !(fabsf(du) <= (l.n_sums > 8 ? kLinePosMax : kLinePosTol));
        if (fabsf(du) > kLinePosTol) slopes = true;
        if (lane < st.cols) l.rec[st.rec + i * st.width + lane].du = du;
    }
    if (bad) s_bad = 1;
    if (slopes) s_slopes = 1;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int ok = s_bad == 0 ? kStripTaken : kStripLeft;
        l.info[st.info] = StripInfo{k0, k1, f0, f1, ok, slot0, nslots, s_slopes};
        if (ok == kStripLeft) atomicAdd(l.n_left, 1);
    }
}

// ------------------------------------------------------------------ nodes

// Sums of the node lines over one chunk of one strip (one wavefront; lane =
// column), and per node the pulses at which its cell differs from the
// reference line's in some column.
template<int W, int N, bool kSlopes>
__device__ inline void node_sums(const LineArgs& a, const Strip& st, const StripInfo& in, int slot,
                                 int64_t ws, int lane)
{
    const int first = (in.slot0 + slot) << a.chunk_log2;
    const int ka = max(in.f0, first), kb = min(in.f1, first + (1 << a.chunk_log2));
    const int kc = (ka + kb) >> 1;
    const double j = (double)(kc - in.k0);
    const int col = min(lane, st.cols - 1);
    const float inv_k = (float)a.inv_k;
    float kap = (float)(ka - kc);

    // The phase from the chunk's centre is evaluated at every pulse, b1 kap +
    // b2 kap^2 with the reference line's b2 (a line's differs by 2e-9 cycles
    // per pulse^2): steps of it in FP32 would gather 1e-4 rad over 64 pulses.
    // Reference line: its cell at the first pulse.
    const Local lr = local_phase(a.rec[st.rec + (st.h / 2) * st.width + col], j, a.inv_k);
    const float b2 = lr.b2;
    const int A = Cell<W>::of(lr.u + (double)(kap * fmaf(b2, kap, lr.b1)) * a.inv_k);
    const double origin = (double)A + Cell<W>::kCentre;
    float ur = (float)(lr.u - origin);
    float b1[N], u0[N], cre[N], cim[N];
    constexpr int M = kSlopes ? kSlopeNodes : 1;
    float dre[M] = {}, dim[M] = {};
    unsigned long long cross[N];
    const float edge = 0.5f - (kSlopes ? kMaskMargin + kLinePosMax : kMaskMargin);
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const Local ln =
            local_phase(a.rec[st.rec + node_line(N, st.h, n) * st.width + col], j, a.inv_k);
        b1[n] = ln.b1;
        u0[n] = (float)(ln.u - origin);
        cre[n] = cim[n] = 0.f;
        cross[n] = 0;
    }
    uint32_t off = (uint32_t)(A + Cell<W>::kFirst) * (uint32_t)sizeof(float2);
    const char* row = reinterpret_cast<const char*>(a.rc + (int64_t)ka * a.nr);
    const int64_t stride = a.nr * (int64_t)sizeof(float2);
    for (int k = ka; k < kb; ++k, kap += 1.f) {
        const float b2k = b2 * kap;
        const float fr = fmaf(kap * (lr.b1 + b2k), inv_k, ur);
        if (__builtin_amdgcn_ballot_w64(fabsf(fr) > 0.5f) != 0) {
            // some column's reference line enters another cell
            const float s = fr > 0.5f ? 1.f : (fr < -0.5f ? -1.f : 0.f);
            ur -= s;
            off += (uint32_t)((int)s * (int)sizeof(float2));
#pragma unroll
            for (int n = 0; n < N; ++n) u0[n] -= s;
        }
        float2 x[W], q[line_degree(W) + 1];
        load_taps<W>(row, off, x);
        row += stride;
        farrow<W>(a.farrow, x, q);
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const float p = kap * (b1[n] + b2k);
            const float f = fmaf(p, inv_k, u0[n]);
            const float sn = __builtin_amdgcn_sinf(p), cs = __builtin_amdgcn_cosf(p);
            float2 s;
            bool taken = false;
#pragma unroll
            for (int m = 0; m < (kSlopes ? kSlopeNodes : 0); ++m) {
                if (slope_node(N, m) != n) continue;
                float2 g;
                s = farrow_slope(q, f, g);
                dre[m] = fmaf(g.x, cs, dre[m]);
                dre[m] = fmaf(-g.y, sn, dre[m]);
                dim[m] = fmaf(g.x, sn, dim[m]);
                dim[m] = fmaf(g.y, cs, dim[m]);
                taken = true;
            }
            if (!taken) s = farrow_eval(q, f);
            cre[n] = fmaf(s.x, cs, cre[n]);
            cre[n] = fmaf(-s.y, sn, cre[n]);
            cim[n] = fmaf(s.x, sn, cim[n]);
            cim[n] = fmaf(s.y, cs, cim[n]);
            const bool out = __builtin_amdgcn_ballot_w64(fabsf(f) > edge) != 0;
            cross[n] |= (unsigned long long)out << (k - first);
        }
    }
    const int64_t at = ws * a.slots + slot;
    float2* s = a.sums + at * (a.n_sums * 64) + lane;
#pragma unroll
    for (int n = 0; n < N; ++n) s[n * 64] = make_float2(cre[n], cim[n]);
    if (kSlopes) {
#pragma unroll
        for (int m = 0; m < M; ++m) s[(8 + m) * 64] = make_float2(dre[m], dim[m]);
    }
    if (lane == 0) {
#pragma unroll
        for (int n = 0; n < N; ++n) a.cross[at * 8 + n] = cross[n];
    }
}

template<int W>
__global__ __launch_bounds__(kLineThreads) __attribute__((amdgpu_waves_per_eu(4)))
void strip_nodes_kernel(LineArgs a)
{
    const int64_t end = min(a.s_end, uniform64(a.batch->n_strips));
    const int64_t item = (int64_t)blockIdx.x * (kLineThreads / 64) +
                         __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t ws = item / a.slots;
    const int slot = (int)(item - ws * a.slots);
    const int64_t t = a.s_begin + ws;
    if (t >= end) return;
    const OutDesc* grids = batch_grids(a.batch);
    const OutDesc d =
        load_desc(grids, find_strip_grid(grids, __builtin_amdgcn_readfirstlane(a.batch->n_grids), t));
    const Strip st = load_strip(d, t);
    const auto* in = uniform_ptr(a.info) + st.info;
    const StripInfo si{in->k0, in->k1, in->f0, in->f1, in->ok, in->slot0, in->nslots, in->slopes};
    if (!si.ok || slot >= si.nslots) return;
    const int first = (si.slot0 + slot) << a.chunk_log2;
    if (first < a.q_begin || first >= a.q_end) return;
    const int lane = threadIdx.x & 63;
    if (si.slopes) {
        if (st.h <= 32)
            node_sums<W, 6, true>(a, st, si, slot, ws, lane);
        else
            node_sums<W, 8, true>(a, st, si, slot, ws, lane);
    } else {
        if (st.h <= 32)
            node_sums<W, 6, false>(a, st, si, slot, ws, lane);
        else
            node_sums<W, 8, false>(a, st, si, slot, ws, lane);
    }
}

// ------------------------------------------------------------------ lines

using Sum64 = double2;

// The difference between a line's own taps and the continued taps of the
// reference cell, for a position f past the cell's end (zero inside it).
// `x`: bins first - 1, first, first + W - 1, first + W of the reference cell.
// (Both weights of an even kernel, a sinc's, are zero at the end itself.)
template<int W>
__device__ inline float2 cell_change(const LineArgs& a, const float2 (&x)[4], float f, bool up)
{
    const float d = fmaxf((up ? f : -f) - 0.5f, 0.f);
    float2 w = end_weights(a, d);
    if (W % 2 == 1) {
        w.x = d > 0.f ? w.x : 0.f;
        w.y = d > 0.f ? w.y : 0.f;
    }
    const float2 xi = up ? x[3] : x[0], xo = up ? x[1] : x[2];
    return make_float2(fmaf(w.x, xi.x, -w.y * xo.x), fmaf(w.x, xi.y, -w.y * xo.y));
}

template<int W>
__device__ inline void load_end_taps(const char* row, uint32_t off, float2 (&x)[4])
{
    const float2* p = reinterpret_cast<const float2*>(row + off);
    x[0] = p[-1];
    x[1] = p[0];
    x[2] = p[W - 1];
    x[3] = p[W];
}

// Chunks [c0, c1) of a group of lines: interpolated node sums and the
// corrections of the pulses at which a line's cell is not the reference's.
// Every `step`th; `add` takes each one's sums.
template<int W, int N, bool kSlopes, class Add>
__device__ inline void line_chunks(const LineArgs& a, const Strip& st, const StripInfo& in, int g,
                                   int c0, int c1, int step, int64_t ws, int lane, Add&& add)
{
    constexpr int G = kGroupLines;
    const int col = min(lane, st.cols - 1);
    const float inv_k = (float)a.inv_k;
    const PixLine* r[G];
    float w[G][N];
#pragma unroll
    for (int i = 0; i < G; ++i)
        r[i] = a.rec + st.rec + min(g * G + i, st.h - 1) * st.width + col;
    // the weights, one per lane, read back into scalar registers
    const int mine = __builtin_bit_cast(
        int, node_weight(N, st.h, min(g * G + (lane / N) % G, st.h - 1), lane % N));
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
        for (int n = 0; n < N; ++n)
            w[i][n] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(mine, i * N + n));
    // times the lines' position off the nodes', for the derivative sums
    constexpr int M = kSlopes ? kSlopeNodes : 1;
    float wd[G][M];
    if (kSlopes) {
        const int own = __builtin_bit_cast(
            int, slope_weight(N, st.h, min(g * G + (lane / M) % G, st.h - 1), lane % M));
#pragma unroll
        for (int i = 0; i < G; ++i)
#pragma unroll
            for (int m = 0; m < M; ++m)
                wd[i][m] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(own, i * M + m));
    }
    const PixLine* rr = a.rec + st.rec + (st.h / 2) * st.width + col;
    // the nodes around the group: its lines change cells no earlier than those
    int nlo = 0, nhi = N - 1;
#pragma unroll
    for (int n = 0; n < N; ++n) {
        if (node_line(N, st.h, n) <= g * G) nlo = n;
        if (node_line(N, st.h, N - 1 - n) >= min(g * G + G - 1, st.h - 1)) nhi = N - 1 - n;
    }
    nlo = __builtin_amdgcn_readfirstlane(nlo);
    nhi = __builtin_amdgcn_readfirstlane(nhi);
    for (int c = c0; c < c1; c += step) {
        const int first = (in.slot0 + c) << a.chunk_log2;
        if (first < a.q_begin || first >= a.q_end) continue;
        // the records are read anew for every chunk (kept in registers they
        // would spill)
        asm volatile("" ::: "memory");
        const int64_t at = ws * a.slots + c;
        const float2* s = a.sums + at * (a.n_sums * 64) + lane;
        float2 v[N], dv[M];
#pragma unroll
        for (int n = 0; n < N; ++n) v[n] = s[n * 64];
        if (kSlopes) {
#pragma unroll
            for (int m = 0; m < M; ++m) dv[m] = s[(8 + m) * 64];
        }
        const int ka = max(in.f0, first), kb = min(in.f1, first + (1 << a.chunk_log2));
        const int kc = (ka + kb) >> 1;
        const double j = (double)(kc - in.k0);
        float ph[G], cre[G], cim[G];
#pragma unroll
        for (int i = 0; i < G; ++i) {
            ph[i] = (float)__builtin_amdgcn_fract(
                fma(fma(fma(fma(r[i]->a4, j, r[i]->a3), j, r[i]->a2), j, r[i]->a1), j, r[i]->p0));
            float re = 0.f, im = 0.f;
#pragma unroll
            for (int n = 0; n < N; ++n) {
                re = fmaf(w[i][n], v[n].x, re);
                im = fmaf(w[i][n], v[n].y, im);
            }
            if (kSlopes) {
                float2 t = make_float2(wd[i][0] * dv[0].x, wd[i][0] * dv[0].y);
#pragma unroll
                for (int m = 1; m < M; ++m) {
                    t.x = fmaf(wd[i][m], dv[m].x, t.x);
                    t.y = fmaf(wd[i][m], dv[m].y, t.y);
                }
                const float du = r[i]->du;
                re = fmaf(du, t.x, re);
                im = fmaf(du, t.y, im);
            }
            const float sn = __builtin_amdgcn_sinf(ph[i]), cs = __builtin_amdgcn_cosf(ph[i]);
            cre[i] = fmaf(re, cs, -im * sn);
            cim[i] = fmaf(re, sn, im * cs);
        }
        uint64_t mask = (uint64_t)uniform64((int64_t)(uniform_ptr(a.cross)[at * 8 + nlo] |
                                                      uniform_ptr(a.cross)[at * 8 + nhi]));
        if (mask != 0) {
            // the reference's cell, from its position at the chunk's centre
            asm volatile("" ::: "memory");
            const Local lr = local_phase(*rr, j, a.inv_k);
            const int A = Cell<W>::of(lr.u);
            const double origin = (double)A + Cell<W>::kCentre;
            const float ur = (float)(lr.u - origin);
            float b1[G], b2[G], u0[G];
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const Local l = local_phase(*r[i], j, a.inv_k);
                b1[i] = l.b1;
                b2[i] = l.b2;
                u0[i] = (float)(l.u - origin);
            }
            const uint32_t off0 = (uint32_t)(A + Cell<W>::kFirst) * (uint32_t)sizeof(float2);
            // The next pulse at which a line of the group has changed cells, and
            // its taps' loads.  The mask is that of the nodes around: no line
            // has while the outer ones have not (to the curvature of u over
            // four lines, 1e-5 bin, and the positions off the nodes').
            const float edge = kSlopes ? 0.5f - 2.f * kLinePosMax : 0.5f;
            float kap_n = 0.f, sh_n = 0.f;
            float2 x_n[4];
            auto next = [&]() {
                while (mask != 0) {
                    const int k = first + __builtin_ctzll(mask);
                    mask &= mask - 1;
                    kap_n = (float)(k - kc);
                    sh_n = rintf(fmaf(kap_n * fmaf(lr.b2, kap_n, lr.b1), inv_k, ur));
                    const float fa = fmaf(kap_n * fmaf(b2[0], kap_n, b1[0]), inv_k, u0[0]) - sh_n;
                    const float fb =
                        fmaf(kap_n * fmaf(b2[G - 1], kap_n, b1[G - 1]), inv_k, u0[G - 1]) - sh_n;
                    if (__builtin_amdgcn_ballot_w64(fmaxf(fabsf(fa), fabsf(fb)) > edge) == 0) continue;
                    load_end_taps<W>(reinterpret_cast<const char*>(a.rc + (int64_t)k * a.nr),
                                     off0 + (uint32_t)((int)sh_n * (int)sizeof(float2)), x_n);
                    return true;
                }
                return false;
            };
            bool more = next();
            while (more) {
                const float kap = kap_n, sh = sh_n;
                const float2 x[4] = {x_n[0], x_n[1], x_n[2], x_n[3]};
                more = next();   // its loads in flight while this pulse is added
                float pk[G], f[G];
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    pk[i] = kap * fmaf(b2[i], kap, b1[i]);
                    f[i] = fmaf(pk[i], inv_k, u0[i]) - sh;
                }
                const bool up = f[0] + f[G - 1] > 0.f;
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    const float2 e = cell_change<W>(a, x, f[i], up);
                    const float sn = __builtin_amdgcn_sinf(ph[i] + pk[i]);
                    const float cs = __builtin_amdgcn_cosf(ph[i] + pk[i]);
                    cre[i] = fmaf(e.x, cs, cre[i]);
                    cre[i] = fmaf(-e.y, sn, cre[i]);
                    cim[i] = fmaf(e.x, sn, cim[i]);
                    cim[i] = fmaf(e.y, cs, cim[i]);
                }
            }
        }
        add(c, cre, cim);
    }
}

// Pulses [k_lo, k_hi) of a group of lines, each line integrating its own
// window's, evaluated line by line.
template<int W>
__device__ inline void line_ends(const LineArgs& a, const Strip& st, const StripInfo& in, int g,
                                 bool head, int lane, Sum64 (&acc)[kGroupLines])
{
    constexpr int G = kGroupLines;
    const int col = min(lane, st.cols - 1);
    const float inv_k = (float)a.inv_k;
    const PixLine* r[G];
    int ks[G], ke[G], lo = INT_MAX, hi = INT_MIN;
#pragma unroll
    for (int i = 0; i < G; ++i) {
        r[i] = a.rec + st.rec + min(g * G + i, st.h - 1) * st.width + col;
        ks[i] = r[i]->kstart;
        ke[i] = r[i]->kstop;
        lo = min(lo, ks[i]);
        hi = max(hi, ke[i]);
    }
    const int k_lo = head ? __builtin_amdgcn_readfirstlane(wave_min_i(lo)) : in.f1;
    const int k_hi = head ? in.f0 : __builtin_amdgcn_readfirstlane(wave_max_i(hi));
    for (int first = k_lo & ~63; first < k_hi; first += 64) {
        if (first < a.q_begin || first >= a.q_end) continue;
        const int ka = max(first, k_lo), kb = min(first + 64, k_hi), kc = (ka + kb) >> 1;
        const double j = (double)(kc - in.k0);
        asm volatile("" ::: "memory");   // as in line_chunks
        // cells follow the group's second line
        float kap = (float)(ka - kc);
        int A;
        {
            const Local l = local_phase(*r[1], j, a.inv_k);
            A = Cell<W>::of(l.u + (double)(kap * fmaf(l.b2, kap, l.b1)) * a.inv_k);
        }
        const double origin = (double)A + Cell<W>::kCentre;
        float b1[G], b2[G], u0[G], ph[G], cre[G], cim[G];
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const Local l = local_phase(*r[i], j, a.inv_k);
            b1[i] = l.b1;
            b2[i] = l.b2;
            u0[i] = (float)(l.u - origin);
            ph[i] = (float)__builtin_amdgcn_fract(l.ph);
            cre[i] = cim[i] = 0.f;
        }
        uint32_t off = (uint32_t)(A + Cell<W>::kFirst) * (uint32_t)sizeof(float2);
        const char* row = reinterpret_cast<const char*>(a.rc + (int64_t)ka * a.nr);
        for (int k = ka; k < kb; ++k, kap += 1.f) {
            float p[G];
#pragma unroll
            for (int i = 0; i < G; ++i) p[i] = kap * fmaf(b2[i], kap, b1[i]);
            const float fr = fmaf(p[1], inv_k, u0[1]);
            if (__builtin_amdgcn_ballot_w64(fabsf(fr) > 0.5f) != 0) {
                const float s = fr > 0.5f ? 1.f : (fr < -0.5f ? -1.f : 0.f);
                off += (uint32_t)((int)s * (int)sizeof(float2));
#pragma unroll
                for (int i = 0; i < G; ++i) u0[i] -= s;
            }
            float2 x[W], q[line_degree(W) + 1];
            load_taps<W>(row, off, x);
            farrow<W>(a.farrow, x, q);
            float f[G];
            float2 s[G];
            bool past = false;
#pragma unroll
            for (int i = 0; i < G; ++i) {
                f[i] = fmaf(p[i], inv_k, u0[i]);
                s[i] = farrow_eval(q, f[i]);
                past |= fabsf(f[i]) > 0.5f;
            }
            if (__builtin_amdgcn_ballot_w64(past) != 0) {
                float2 y[4];
                load_end_taps<W>(row, off, y);
                const bool up = f[0] + f[G - 1] > 0.f;
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    const float2 e = cell_change<W>(a, y, f[i], up);
                    s[i].x += e.x;
                    s[i].y += e.y;
                }
            }
            row += a.nr * (int64_t)sizeof(float2);
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const bool on = k >= ks[i] && k < ke[i];
                const float sn = on ? __builtin_amdgcn_sinf(ph[i] + p[i]) : 0.f;
                const float cs = on ? __builtin_amdgcn_cosf(ph[i] + p[i]) : 0.f;
                cre[i] = fmaf(s[i].x, cs, cre[i]);
                cre[i] = fmaf(-s[i].y, sn, cre[i]);
                cim[i] = fmaf(s[i].x, sn, cim[i]);
                cim[i] = fmaf(s[i].y, cs, cim[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < G; ++i) {
            acc[i].x += (double)cre[i];
            acc[i].y += (double)cim[i];
        }
    }
}

template<int W, class Add>
__device__ inline void any_chunks(const LineArgs& a, const Strip& st, const StripInfo& in, int g,
                                  int c0, int c1, int step, int64_t ws, int lane, Add&& add)
{
    if (in.slopes) {
        if (st.h <= 32)
            line_chunks<W, 6, true>(a, st, in, g, c0, c1, step, ws, lane, add);
        else
            line_chunks<W, 8, true>(a, st, in, g, c0, c1, step, ws, lane, add);
    } else {
        if (st.h <= 32)
            line_chunks<W, 6, false>(a, st, in, g, c0, c1, step, ws, lane, add);
        else
            line_chunks<W, 8, false>(a, st, in, g, c0, c1, step, ws, lane, add);
    }
}

// One wavefront per group of kGroupLines lines and segment: a quarter of the
// strip's chunks (strip_lines_kernel) or one of the aperture's ends
// (strip_ends_kernel).  Workgroups of one wavefront: the groups' work differs
// with their distance from the reference line, and a workgroup's registers
// are free only when its last wavefront ends.
template<int W, bool kEnds>
__device__ inline void group_sums(const LineArgs& a)
{
    constexpr int kFirstSeg = kEnds ? kCoreSegs : 0;
    constexpr int kNumSegs = kEnds ? kSegs - kCoreSegs : kCoreSegs;
    const int64_t end = min(a.s_end, uniform64(a.batch->n_strips));
    const int64_t item = blockIdx.x;
    const int64_t ws = item / (kNumSegs * kMaxGroups);
    const int rest = (int)(item - ws * (kNumSegs * kMaxGroups));
    const int seg = kFirstSeg + rest / kMaxGroups, g = rest % kMaxGroups;
    const int64_t t = a.s_begin + ws;
    if (t >= end) return;
    const OutDesc* grids = batch_grids(a.batch);
    const OutDesc d =
        load_desc(grids, find_strip_grid(grids, __builtin_amdgcn_readfirstlane(a.batch->n_grids), t));
    const Strip st = load_strip(d, t);
    const auto* in = uniform_ptr(a.info) + st.info;
    const StripInfo si{in->k0, in->k1, in->f0, in->f1, in->ok, in->slot0, in->nslots, in->slopes};
    if (!si.ok || g * kGroupLines >= st.h) return;
    const int lane = threadIdx.x & 63;
    Sum64 acc[kGroupLines];
#pragma unroll
    for (int i = 0; i < kGroupLines; ++i) acc[i] = make_double2(0., 0.);
    const int64_t at =
        (ws * kSegs + seg) * (kStripLines * 64) + g * kGroupLines * 64 + lane;
    if (a.carry != nullptr && !a.q_first) {
#pragma unroll
        for (int i = 0; i < kGroupLines; ++i) acc[i] = a.carry[at + i * 64];
    }
    if (kEnds) {
        line_ends<W>(a, st, si, g, seg == kCoreSegs, lane, acc);
    } else {
        const int c0 = seg * si.nslots / kCoreSegs, c1 = (seg + 1) * si.nslots / kCoreSegs;
        auto add = [&](int, const float (&cre)[kGroupLines], const float (&cim)[kGroupLines]) {
#pragma unroll
            for (int i = 0; i < kGroupLines; ++i) {
                acc[i].x += (double)cre[i];
                acc[i].y += (double)cim[i];
            }
        };
        any_chunks<W>(a, st, si, g, c0, c1, 1, ws, lane, add);
    }
    if (a.carry != nullptr) {
#pragma unroll
        for (int i = 0; i < kGroupLines; ++i) a.carry[at + i * 64] = acc[i];
    }
#pragma unroll
    for (int i = 0; i < kGroupLines; ++i)
        a.parts[at + i * 64] = make_float2((float)acc[i].x, (float)acc[i].y);
}

template<int W>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
void strip_lines_kernel(LineArgs a)
{
    if (a.few == 2 && uniform64(a.batch->n_strips) <= kFewStrips) return;
    group_sums<W, false>(a);
}

// As strip_lines_kernel, with a workgroup of four wavefronts per segment and
// group: each takes every fourth chunk and leaves its sums in LDS, then line i's
// are added by wavefront i in the order of the chunks, so that the sums do not
// depend on which kernel ran.  A single strip is 32 to 64 segments, each of 16
// chunks of 8,000 cycles of issue one after the other: 54 us for 32 x 32 pixels
// of 4,000 pulses, 27 us here.  Few wavefronts are in flight, so each has the
// registers it needs (two per SIMD; at four they spill: 31 us).
template<int W>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void strip_few_kernel(LineArgs a)
{
    constexpr int kRound = 20;   // chunks held at once
    static_assert(kGroupLines == 4, "a wavefront per line");
    __shared__ float2 s_sum[kRound][kGroupLines][64];
    const int64_t n_strips = uniform64(a.batch->n_strips);
    if (a.few == 2 && n_strips > kFewStrips) return;
    const int64_t end = min(a.s_end, n_strips);
    const int64_t item = blockIdx.x;
    const int64_t ws = item / (kCoreSegs * kMaxGroups);
    const int rest = (int)(item - ws * (kCoreSegs * kMaxGroups));
    const int seg = rest / kMaxGroups, g = rest % kMaxGroups;
    const int64_t t = a.s_begin + ws;
    if (t >= end) return;
    const OutDesc* grids = batch_grids(a.batch);
    const OutDesc d =
        load_desc(grids, find_strip_grid(grids, __builtin_amdgcn_readfirstlane(a.batch->n_grids), t));
    const Strip st = load_strip(d, t);
    const auto* in = uniform_ptr(a.info) + st.info;
    const StripInfo si{in->k0, in->k1, in->f0, in->f1, in->ok, in->slot0, in->nslots, in->slopes};
    if (!si.ok || g * kGroupLines >= st.h) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t at = (ws * kSegs + seg) * (kStripLines * 64) + (g * kGroupLines + wave) * 64 + lane;
    Sum64 acc = make_double2(0., 0.);
    if (a.carry != nullptr && !a.q_first) acc = a.carry[at];
    const int c0 = seg * si.nslots / kCoreSegs, c1 = (seg + 1) * si.nslots / kCoreSegs;
    for (int r0 = c0; r0 < c1; r0 += kRound) {
        const int r1 = min(c1, r0 + kRound);
        auto keep = [&](int c, const float (&cre)[kGroupLines], const float (&cim)[kGroupLines]) {
#pragma unroll
            for (int i = 0; i < kGroupLines; ++i)
                s_sum[c - r0][i][lane] = make_float2(cre[i], cim[i]);
        };
        any_chunks<W>(a, st, si, g, r0 + wave, r1, kGroupLines, ws, lane, keep);
        __syncthreads();
        for (int c = r0; c < r1; ++c) {
            // chunks of other parts of the pulses were passed over
            const int first = (si.slot0 + c) << a.chunk_log2;
            if (first < a.q_begin || first >= a.q_end) continue;
            const float2 v = s_sum[c - r0][wave][lane];
            acc.x += (double)v.x;
            acc.y += (double)v.y;
        }
        __syncthreads();
    }
    if (a.carry != nullptr) a.carry[at] = acc;
    a.parts[at] = make_float2((float)acc.x, (float)acc.y);
}

template<int W>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
void strip_ends_kernel(LineArgs a)
{
    group_sums<W, true>(a);
}

// The partial sums of each pixel of a strip, in segment order.  A strip with a
// sum that is not finite is left to the pixel-by-pixel sum: a NaN or an
// infinity among the pulses reaches every line of a column through the node
// sums and the corrections (never none of those that integrate it), and pixels
// whose own taps miss it keep their finite values there.
__global__ __launch_bounds__(kLineThreads) void strip_sum_kernel(LineArgs a)
{
    constexpr int kPer = kStripLines * 64 / kLineThreads / 4;   // pixels per thread
    const int64_t end = min(a.s_end, uniform64(a.batch->n_strips));
    const int64_t ws = blockIdx.x / 4;
    const int64_t t = a.s_begin + ws;
    if (t >= end) return;
    const OutDesc* grids = batch_grids(a.batch);
    const OutDesc d =
        load_desc(grids, find_strip_grid(grids, __builtin_amdgcn_readfirstlane(a.batch->n_grids), t));
    const Strip st = load_strip(d, t);
    if (!(uniform_ptr(a.info) + st.info)->ok) return;
    const float2* e = a.parts + ws * kSegs * (kStripLines * 64);
    bool bad = false;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int i = ((int)(blockIdx.x & 3) * kPer + q) * (kLineThreads / 64) + (threadIdx.x >> 6);
        const int lane = threadIdx.x & 63;
        if (i >= st.h || lane >= st.cols) continue;
        double re = 0., im = 0.;
#pragma unroll
        for (int s = 0; s < kSegs; ++s) {
            const float2 v = e[s * (kStripLines * 64) + i * 64 + lane];
            re += (double)v.x;
            im += (double)v.y;
        }
        const float2 z = make_float2((float)re, (float)im);
        bad |= !(fabsf(z.x) <= FLT_MAX && fabsf(z.y) <= FLT_MAX);
        st.out[st.pix0 + i * st.width + lane] = z;
    }
    if (__syncthreads_or(bad) && threadIdx.x == 0 &&
        atomicExch(&a.info[st.info].ok, kStripRedo) != kStripRedo)
        atomicAdd(a.n_left + 1, 1);
}

}  // namespace

// Bytes per strip of the running sums kept between parts of the pulses.
size_t line_carry_bytes() { return (size_t)kSegs * kStripLines * 64 * sizeof(double2); }

size_t line_strip_bytes(int slots, int n_sums)
{
    return (size_t)slots * (n_sums * 64 * sizeof(float2) + 8 * sizeof(unsigned long long)) +
           (size_t)kSegs * kStripLines * 64 * sizeof(float2);
}

// Workspace of n strips at `ws`: node sums, partial sums, cell-change masks.
void line_place(LineArgs& a, unsigned char* ws, int64_t n)
{
    a.sums = reinterpret_cast<float2*>(ws);
    ws += (size_t)n * a.slots * a.n_sums * 64 * sizeof(float2);
    a.parts = reinterpret_cast<float2*>(ws);
    ws += (size_t)n * kSegs * kStripLines * 64 * sizeof(float2);
    a.cross = reinterpret_cast<unsigned long long*>(ws);
}

namespace {

template<int W>
const void* width_fn(int which)
{
    switch (which) {
    case kLineNodes: return reinterpret_cast<const void*>(&strip_nodes_kernel<W>);
    case kLineLines: return reinterpret_cast<const void*>(&strip_lines_kernel<W>);
    case kLineFew: return reinterpret_cast<const void*>(&strip_few_kernel<W>);
    case kLineEnds: return reinterpret_cast<const void*>(&strip_ends_kernel<W>);
    case kLineSum: return reinterpret_cast<const void*>(&strip_sum_kernel);
    default: return reinterpret_cast<const void*>(&strip_fit_kernel);
    }
}

}  // namespace

const void* line_kernel_fn(int which, int width)
{
    return width == 8 ? width_fn<8>(which) : width == 9 ? width_fn<9>(which) : nullptr;
}

// Workgroups of each kernel for n strips.
int64_t line_grid(int which, int slots, int64_t n)
{
    constexpr int kWaves = kLineThreads / 64;
    switch (which) {
    case kLineFit: return n;
    case kLineNodes: return (n * slots + kWaves - 1) / kWaves;
    case kLineLines:
    case kLineFew: return n * kCoreSegs * kMaxGroups;
    case kLineEnds: return n * (kSegs - kCoreSegs) * kMaxGroups;
    default: return n * 4;
    }
}

hipError_t launch_strip_fit(const GeomArgs& g, const LineArgs& a, int64_t grid, hipStream_t stream)
{
    if (grid <= 0) return hipSuccess;
    hipLaunchKernelGGL(strip_fit_kernel, dim3((unsigned)grid), dim3(512), 0, stream, g, a);
    return hipGetLastError();
}

// The nodes, lines, ends and (unless more parts of the pulses follow) sum of
// the strips [a.s_begin, a.s_end).
hipError_t launch_strips(const LineArgs& a, int width, bool last, hipStream_t stream)
{
    void* kargs[] = {const_cast<LineArgs*>(&a)};
    for (int which = kLineNodes; which <= (last ? kLineSum : kLineEnds); ++which) {
        if (which == (a.few == 0 ? kLineFew : a.few == 1 ? kLineLines : kLineFit)) continue;
        const int64_t grid = line_grid(which, a.slots, a.s_end - a.s_begin);
        if (grid <= 0) continue;
        const void* fn = line_kernel_fn(which, width);
        if (fn == nullptr) return hipErrorInvalidValue;
        const int threads = which == kLineLines || which == kLineEnds ? 64 : kLineThreads;
        const hipError_t e =
            hipLaunchKernel(fn, dim3((unsigned)grid), dim3(threads), kargs, 0, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace bp
