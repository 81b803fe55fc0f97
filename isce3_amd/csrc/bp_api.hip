// C-ABI of the backprojection path: argument checks that mirror the
// reference's (focus/Backproject.cpp:77-92, pybind focus/Backproject.cpp:97-135,
// DryTroposphereModel.cpp:20-33), device uploads into a per-context grow-only
// arena, and the three-pass launch (pulse orbit, per-pixel geometry,
// coherent sum) on the caller's stream.
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <exception>
#include <string>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "../../include/isce3_amd_backproject.h"
#include "bp_internal.h"

namespace {

thread_local std::string g_msg;

int fail(int code, const std::string& msg)
{
    g_msg = msg;
    return code;
}

}  // namespace

// Shared with the range-compression entry points (rc_api.hip).
void bp_set_last_error(const std::string& msg) { g_msg = msg; }

// Every int-valued entry point ends in a catch clause that returns this, so
// no C++ exception crosses the C ABI: a failed host allocation gives
// BP_ERR_OUT_OF_MEMORY, any other exception BP_ERR_RUNTIME, with the message
// set (or cleared, if even the message cannot be stored).
int bp_host_exception() noexcept
{
    int code = BP_ERR_RUNTIME;
    try {
        try {
            throw;
        } catch (const std::bad_alloc&) {
            code = BP_ERR_OUT_OF_MEMORY;
            g_msg = "host memory allocation failed";
        } catch (const std::exception& e) {
            g_msg = std::string("host exception: ") + e.what();
        } catch (...) {
            g_msg = "unknown host exception";
        }
    } catch (...) {
        g_msg.clear();
    }
    return code;
}

int bp::usable_cpus()
{
    cpu_set_t set;
    CPU_ZERO(&set);
    if (sched_getaffinity(0, sizeof(set), &set) == 0) return std::max(1, CPU_COUNT(&set));
    return (int)std::max(1u, std::thread::hardware_concurrency());
}

namespace bp {

int check_out_block(const bp_out_block& b)
{
    const bp_grid& go = b.grid;
    if (go.length < 0 || go.width < 0) return fail(BP_ERR_INVALID_ARGUMENT, "negative grid size");
    if (go.length > INT32_MAX || go.width > INT32_MAX)
        return fail(BP_ERR_INVALID_ARGUMENT, "grid size exceeds int range");
    if (!(go.prf > 0)) return fail(BP_ERR_INVALID_ARGUMENT, "PRF must be positive");
    if (go.length * go.width > 0 && b.out_dev == nullptr)
        return fail(BP_ERR_INVALID_ARGUMENT, "out is null");
    return BP_SUCCESS;
}

}  // namespace bp

namespace {

// A device buffer.  `fixed` buffers are views of a region the library does
// not own (the static scratch of bp_backproject_noalloc): they are never
// grown or freed, and a call that needs more than they hold fails.
struct DevBuf {
    void* ptr = nullptr;
    size_t bytes = 0;
    bool fixed = false;
};

}  // namespace

// Device copies of everything a call needs besides the pulses and the output
// blocks: orbits, Doppler tables, DEM, kernel tables and (plain precision)
// the platform state at every pulse.
struct StaticData {
    DevBuf table, table2, poly, poly2, in_pos, in_vel, out_pos, out_vel, in_dop, out_dop, dem,
        pulse_pv, sinc;
    std::vector<float> poly_host, poly2_host;
    std::vector<double> table2_host;
};

// Per-pixel records, batch header + output descriptors, and the flags of one
// call ([0] any failed, [1] out of range, [2] strips the line-interpolated sum
// leaves, [3] strips done again, [8..9] update count, [16 + g] grid g failed).
struct Scratch {
    DevBuf geom, split, flags, desc;
    DevBuf strips, lines;   // line-interpolated sum: StripInfo, workspace
    DevBuf parts;           // plain sum: segment sums of small batches
};

// Buffers of the host-input path (bp_backproject_host): device pulse windows,
// band descriptors and windows, pinned staging, a copy stream and its events.
// Created on first use and kept by the context.
struct HostPath {
    DevBuf win[2];            // device copies of band pulse windows
    DevBuf band_desc;         // batch header + descriptor of every band
    DevBuf band_win;          // [kmin, kmax) of every line band (int32 pairs)
    DevBuf carry;             // running sums of a strip row taken in parts
    unsigned char* stage[2] = {nullptr, nullptr};  // pinned staging of pulse chunks
    size_t stage_bytes = 0;
    int32_t* h_win = nullptr; // pinned copy of band_win
    int32_t* h_bad = nullptr; // pinned: strips that sum pixel by pixel
    size_t h_win_words = 0;
    hipStream_t copy = nullptr;
    hipEvent_t stage_ev[2] = {nullptr, nullptr};  // copy out of staging j finished
    hipEvent_t win_ev = nullptr;                  // band windows on the host
    hipEvent_t copied_ev = nullptr;               // a band's pulses on the device
    hipEvent_t sum_ev[2] = {nullptr, nullptr};    // sum reading window buffer w finished
    std::vector<hipEvent_t> timing;               // per band: copy start/end, sum start/end
};

// A second stream for the strips that the line-interpolated sum leaves, and the
// events that part it from the call's stream and join it again.
struct Branch {
    hipStream_t s = nullptr;   // default priority
    hipEvent_t part = nullptr, fit = nullptr, join = nullptr;
    bool create()
    {
        return hipStreamCreateWithFlags(&s, hipStreamNonBlocking) == hipSuccess &&
               hipEventCreateWithFlags(&part, hipEventDisableTiming) == hipSuccess &&
               hipEventCreateWithFlags(&fit, hipEventDisableTiming) == hipSuccess &&
               hipEventCreateWithFlags(&join, hipEventDisableTiming) == hipSuccess;
    }
    void destroy()
    {
        if (part) (void)hipEventDestroy(part);
        if (fit) (void)hipEventDestroy(fit);
        if (join) (void)hipEventDestroy(join);
        if (s) (void)hipStreamDestroy(s);
    }
};

struct bp_context {
    int device = 0;
    int n_cu = 0;
    int64_t workspace_limit = -1;      // bp_context_limit_workspace
    unsigned char* scratch = nullptr;  // device address of this device's no-alloc scratch
    std::string scratch_err;           // why it is null
    StaticData st;
    Scratch sc;
    HostPath hp;
    hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
    Branch branch;
    std::vector<unsigned char> desc_host;
    std::vector<int> desc_block;
    std::vector<int32_t> flags_host;
};

namespace {

int ensure(DevBuf& b, size_t bytes)
{
    if (bytes == 0) bytes = 16;
    if (b.bytes >= bytes) return BP_SUCCESS;
    if (b.fixed)
        return fail(BP_ERR_LENGTH, "call needs " + std::to_string(bytes) +
                                       " bytes of a fixed scratch buffer of " +
                                       std::to_string(b.bytes));
    if (b.ptr) {
        (void)hipFree(b.ptr);
        b.ptr = nullptr;
        b.bytes = 0;
    }
    hipError_t e = hipMalloc(&b.ptr, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(BP_ERR_OUT_OF_MEMORY, std::string("hipMalloc failed: ") + hipGetErrorString(e));
    }
    b.bytes = bytes;
    return BP_SUCCESS;
}

int upload(DevBuf& b, const void* src, size_t bytes, hipStream_t s)
{
    int rc = ensure(b, bytes);
    if (rc != BP_SUCCESS) return rc;
    if (bytes == 0 || src == nullptr) return BP_SUCCESS;
    hipError_t e = hipMemcpyAsync(b.ptr, src, bytes, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return fail(BP_ERR_HIP, std::string("hipMemcpyAsync: ") + hipGetErrorString(e));
    return BP_SUCCESS;
}

#define BP_HIP_CHECK(expr)                                                                   \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess)                                                                \
            return fail(BP_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));       \
    } while (0)

const char* orbit_err_string(int code)
{
    switch (code) {
    case BP_ORBIT_INTERP_SIZE_ERROR: return "insufficient orbit state vectors to form interpolant";
    case BP_ORBIT_INTERP_DOMAIN_ERROR: return "interpolation point outside orbit domain";
    case BP_ORBIT_INTERP_UNKNOWN_METHOD: return "unexpected orbit interpolation method";
    default: return "orbit interpolation error";
    }
}

int check_orbit(const bp_orbit& o, const char* what)
{
    if (o.n < 2 || o.pos == nullptr || o.vel == nullptr)
        return fail(BP_ERR_INVALID_ARGUMENT, std::string(what) + ": orbit needs at least two state vectors");
    if (!(o.dt > 0.0)) return fail(BP_ERR_INVALID_ARGUMENT, std::string(what) + ": orbit spacing must be positive");
    if (o.method != BP_INTERP_HERMITE && o.method != BP_INTERP_LEGENDRE)
        return fail(BP_ERR_OUT_OF_RANGE, orbit_err_string(BP_ORBIT_INTERP_UNKNOWN_METHOD));
    const int minsv = o.method == BP_INTERP_HERMITE ? 4 : 9;
    if (o.n < minsv) return fail(BP_ERR_OUT_OF_RANGE, orbit_err_string(BP_ORBIT_INTERP_SIZE_ERROR));
    return BP_SUCCESS;
}

int check_lut(const bp_lut2d& l, const char* what)
{
    if (!l.have_data) return BP_SUCCESS;
    if (l.width < 2 || l.length < 2 || l.data == nullptr || !(l.dx != 0.0) || !(l.dy != 0.0))
        return fail(BP_ERR_INVALID_ARGUMENT, std::string(what) + ": Doppler LUT2d needs at least 2x2 samples");
    return BP_SUCCESS;
}

bp::Orbit dev_orbit(const bp_orbit& o, const DevBuf& pos, const DevBuf& vel)
{
    bp::Orbit d;
    d.t0 = o.t0;
    d.dt = o.dt;
    d.n = o.n;
    d.method = o.method;
    d.pos = static_cast<const double*>(pos.ptr);
    d.vel = static_cast<const double*>(vel.ptr);
    return d;
}

bp::Lut2d dev_lut(const bp_lut2d& l, const DevBuf& data)
{
    bp::Lut2d d;
    d.have_data = l.have_data;
    d.bounds_error = l.bounds_error;
    d.ref_value = l.ref_value;
    d.xstart = l.xstart;
    d.ystart = l.ystart;
    d.dx = l.dx;
    d.dy = l.dy;
    d.width = l.width;
    d.length = l.length;
    d.data = static_cast<const double*>(data.ptr);
    return d;
}

bp::Orbit host_orbit(const bp_orbit& o)
{
    bp::Orbit d;
    d.t0 = o.t0;
    d.dt = o.dt;
    d.n = o.n;
    d.method = o.method;
    d.pos = o.pos;
    d.vel = o.vel;
    return d;
}

bp::Lut2d host_lut(const bp_lut2d& l)
{
    bp::Lut2d d;
    d.have_data = l.have_data;
    d.bounds_error = l.bounds_error;
    d.ref_value = l.ref_value;
    d.xstart = l.xstart;
    d.ystart = l.ystart;
    d.dx = l.dx;
    d.dy = l.dy;
    d.width = l.width;
    d.length = l.length;
    d.data = l.data;
    return d;
}

// The windowed-sinc kernel of the DEM factory's Sinc2dInterpolator(8, 8192)
// (core/Sinc2dInterpolator.cpp:14-41, coefficients :105-120): the 65536
// samples of a sinc under a raised-cosine window, regrouped into 8192
// fractional rows of 8 taps, each row divided by its sum; stored as float
// (the interpolator casts each coefficient to the raster's float type).
// Built once per process.
const std::vector<float>& sinc_kernel_table()
{
    static const std::vector<float> table = [] {
        constexpr int L = bp::kSincLen, D = bp::kSincSub, n = L * D;
        const double mid = (n - 1.0) / 2.0;
        std::vector<double> f(n);
        for (int i = 0; i < n; ++i) {
            const double window = 0.5 + 0.5 * std::cos(M_PI * (i - mid) / mid);
            const double s = std::floor(i - mid) / D;
            f[i] = window * (s != 0.0 ? std::sin(M_PI * s) / (M_PI * s) : 1.0);
        }
        std::vector<float> t((size_t)n);
        for (int r = 0; r < D; ++r) {
            double sum = 0.0;
            for (int j = 0; j < L; ++j) sum += f[r + D * j];
            for (int j = 0; j < L; ++j) t[(size_t)r * L + j] = (float)(f[r + D * j] / sum);
        }
        return t;
    }();
    return table;
}

bp::Dem host_dem(const bp_dem& m)
{
    bp::Dem d;
    d.have_raster = m.have_raster;
    d.epsg = m.epsg;
    d.method = m.method;
    d.pad_ = 0;
    d.ref_height = m.ref_height;
    d.xstart = m.xstart;
    d.ystart = m.ystart;
    d.dx = m.dx;
    d.dy = m.dy;
    d.width = m.width;
    d.length = m.length;
    d.data = m.data;
    d.sinc = m.method == BP_DEM_SINC ? sinc_kernel_table().data() : nullptr;
    if (!bp::proj_init(m.epsg, &d.proj)) bp::proj_init(4326, &d.proj);
    return d;
}

bool dem_method_ok(int m)
{
    return m == BP_DEM_BILINEAR || m == BP_DEM_BICUBIC || m == BP_DEM_NEAREST ||
           m == BP_DEM_BIQUINTIC || m == BP_DEM_SINC;
}

bp::TileMap make_map(int64_t length, int64_t width, int tile_rows, int order, int lane_rows)
{
    bp::TileMap m;
    m.tile_rows = tile_rows;
    m.tile_cols = 64 / tile_rows;
    m.lane_rows = lane_rows;
    const int64_t rows = (int64_t)tile_rows * lane_rows;
    m.tiles_x = (int32_t)((width + m.tile_cols - 1) / m.tile_cols);
    m.tiles_y = (int32_t)((length + rows - 1) / rows);
    m.length = length;
    m.width = width;
    m.n_tiles = (int64_t)m.tiles_x * m.tiles_y;
    m.order = order;
    return m;
}

// Polyphase weight rows for the split kernel: row q holds the W tap weights
// at fractional offset t0 = tmin + q/Q (evaluated from the float table with
// the reference's linear interpolation, in FP64) and the difference to row q+1.
void build_polyphase(const bp_kernel& k, int width, std::vector<float>& out)
{
    const int Q = bp::kPolyphaseRows;
    const int wp = (width + 3) / 4 * 4;
    const double tmin = (width % 2 == 0) ? 0.0 : -0.5;
    const double hw = k.halfwidth;
    const double dx = hw / (k.n - 1.0);
    const float rdx = (float)(1.0 / dx);
    auto weight = [&](double x) {
        double ax = std::fabs(x);
        if (ax > hw) return 0.0;
        double axn = ax * (double)rdx;
        int i = std::min((int)std::floor(axn), k.n - 2);
        return (double)k.table[i] + (axn - i) * (double)(k.table[i + 1] - k.table[i]);
    };
    std::vector<double> w((size_t)(Q + 1) * width);
    for (int q = 0; q <= Q; ++q) {
        const double t0 = tmin + (double)q / Q;
        for (int m = 0; m < width; ++m) w[(size_t)q * width + m] = weight((m - width / 2) + t0);
    }
    // Q + 1 rows so that offsets t0 = tmin + 1 (q = Q) index a valid row
    // (whose deltas are zero) without clamping in the kernel.
    const int row = bp::poly_row_floats(width);
    out.assign((size_t)(Q + 1) * row, 0.f);
    for (int q = 0; q <= Q; ++q) {
        for (int m = 0; m < width; ++m) {
            const float w0 = (float)w[(size_t)q * width + m];
            const float w1 = q < Q ? (float)w[(size_t)(q + 1) * width + m] : w0;
            out[(size_t)q * row + m] = w0;
            out[(size_t)q * row + wp + m] = w1 - w0;
        }
    }
}

// Two-line weight table of kernel width W: Q = 2^pair_q_log2(W) rows at
// fractional offsets t0 = tmin + q/Q (tmin = 0 for even W, -1/2 for odd W, as
// the one-line table), each row pair_row_floats(W) floats, in two copies
// stored one after the other (copy o of row q at floats (2 q + o) RF): copy 0
// holds the W weights in entries 0..W-1 and a zero in entry W, copy 1 a zero
// in entry 0 and the weights in entries 1..W.  Entries interpolated in
// the sum (pair_lerp_lo .. + pair_lerp_n) hold the weight at t0 and, after the
// W + 1 entries, its difference to the weight at t0 + 1/Q; the others hold the
// weight at t0 + 1/(2Q), the middle of the row's interval.
void build_pair_table(const bp_kernel& k, int W, std::vector<float>& out)
{
    const int Q = 1 << bp::pair_q_log2(W);
    const int RF = bp::pair_row_floats(W);
    const int lo = bp::pair_lerp_lo(W), nl = bp::pair_lerp_n(W);
    const double tmin = (W % 2 == 0) ? 0.0 : -0.5;
    const double hw = k.halfwidth;
    const double dx = hw / (k.n - 1.0);
    const float rdx = (float)(1.0 / dx);
    auto weight = [&](double x) {
        double ax = std::fabs(x);
        if (ax > hw) return 0.0;
        double axn = ax * (double)rdx;
        int i = std::min((int)std::floor(axn), k.n - 2);
        return (double)k.table[i] + (axn - i) * (double)(k.table[i + 1] - k.table[i]);
    };
    out.assign((size_t)bp::pair_table_floats(W), 0.f);
    for (int o = 0; o < 2; ++o) {
        for (int q = 0; q < Q; ++q) {
            float* r = &out[((size_t)q * 2 + o) * RF];
            const double t0 = tmin + (double)q / Q;
            for (int e = 0; e <= W; ++e) {
                const int m = e - o;  // tap of entry e in this copy
                if (m < 0 || m >= W) continue;
                const double x = (m - W / 2) + t0;
                if (e >= lo && e < lo + nl) {
                    const float w0 = (float)weight(x), w1 = (float)weight(x + 1.0 / Q);
                    r[e] = w0;
                    r[W + 1 + (e - lo)] = w1 - w0;
                } else {
                    r[e] = (float)weight(x + 0.5 / Q);
                }
            }
        }
    }
}

// Least-squares polynomials of degree D over [-F, F] through samples at x with
// weights w, solved in the Chebyshev basis: the matrix [D + 1][samples] that
// takes the samples to the monomial coefficients.
template<int D>
std::vector<double> polynomial_map(double F, const std::vector<double>& x,
                                   const std::vector<double>& w)
{
    constexpr int N = D + 1;
    const int M = (int)x.size();
    std::vector<long double> row[N];   // normal matrix, then a right side per sample
    for (auto& r : row) r.assign(N + M, 0.L);
    for (int i = 0; i < M; ++i) {
        long double t[N];
        t[0] = 1.;
        if (N > 1) t[1] = x[i] / F;
        for (int k = 2; k < N; ++k) t[k] = 2 * (x[i] / F) * t[k - 1] - t[k - 2];
        for (int r = 0; r < N; ++r) {
            for (int q = 0; q < N; ++q) row[r][q] += w[i] * t[r] * t[q];
            row[r][N + i] = w[i] * t[r];
        }
    }
    for (int k = 0; k < N; ++k) {
        int piv = k;
        for (int r = k + 1; r < N; ++r)
            if (std::fabs(row[r][k]) > std::fabs(row[piv][k])) piv = r;
        std::swap(row[k], row[piv]);
        for (int r = 0; r < N; ++r) {
            if (r == k) continue;
            const long double f = row[r][k] / row[k][k];
            for (int q = k; q < N + M; ++q) row[r][q] -= f * row[k][q];
        }
    }
    // Chebyshev -> monomial
    long double basis[N][N] = {};
    basis[0][0] = 1.;
    if (N > 1) basis[1][1] = 1.;
    for (int k = 2; k < N; ++k)
        for (int n = 0; n < N; ++n)
            basis[k][n] = (n > 0 ? 2 * basis[k - 1][n - 1] : 0.L) - basis[k - 2][n];
    std::vector<double> out((size_t)N * M);
    long double f = 1.;
    for (int n = 0; n < N; ++n) {
        for (int i = 0; i < M; ++i) {
            long double c = 0.;
            for (int k = 0; k < N; ++k) c += basis[k][n] * (row[k][N + i] / row[k][k]);
            out[(size_t)n * M + i] = (double)(c * f);
        }
        f /= F;
    }
    return out;
}

// What build_line_table needs of the fits of one kernel width, the same for every
// kernel (made once per process, as every call builds its kernel's table).
template<int W>
struct LineFits {
    static constexpr int kTaps = (W + 1) / 2, kSamples = 97, kEndSamples = 33;
    static constexpr int D = bp::line_degree(W);
    static constexpr double F = 0.5 + (double)bp::kLineMaxShift, E = 0.5 * (double)bp::kLineMaxShift;
    std::vector<double> x, xe, cell[kTaps], end;
    LineFits() : x(kSamples), xe(kEndSamples)
    {
        std::vector<double> w(kSamples);
        for (int i = 0; i < kSamples; ++i) x[i] = F * std::cos(M_PI * (i + 0.5) / kSamples);
        for (int t = 0; t < kTaps; ++t) {
            for (int i = 0; i < kSamples; ++i)
                w[i] = std::fabs(t - 0.5 * (W - 1) - x[i]) <= 0.5 * W ? 1. : 1e-8;
            cell[t] = polynomial_map<D>(F, x, w);
        }
        for (int i = 0; i < kEndSamples; ++i) xe[i] = E * std::cos(M_PI * (i + 0.5) / kEndSamples);
        end = polynomial_map<bp::kEndDegree>(E, xe, std::vector<double>(kEndSamples, 1.));
    }
    static const LineFits& get()
    {
        static const LineFits fits;
        return fits;
    }
};

// Tap weight polynomials of the line-interpolated sum: tap t's weight at
// position f of its cell (0 at the centre, the cell |f| <= 1/2) continued
// smoothly to |f| <= 1/2 + kLineMaxShift, where the truncated kernel is zero
// or another tap has taken over.  False when the kernel is not smooth enough
// for them (or has another width): such kernels keep the pixel-by-pixel sum.
// The limit, 1e-4 of the kernel's peak at the worst position, keeps the sum's
// error below that of the pixel-by-pixel sum's weight table (5.4e-5 relative at
// width 8, 1.2e-4 with white noise).
template<int W>
bool fit_line_table(const bp_kernel& k, bp::LineArgs* a)
{
    using Fits = LineFits<W>;
    const Fits& fits = Fits::get();
    const double hw = k.halfwidth;
    const double dx = hw / (k.n - 1.0), rdx = 1.0 / dx;
    auto weight = [&](double ax) {
        const int i = std::min((int)(ax * rdx), k.n - 2);
        return (double)k.table[i] + (ax * rdx - i) * (double)(k.table[i + 1] - k.table[i]);
    };
    const int m = std::min(k.n - 1, 8);   // slope at the kernel's end
    const double slope = ((double)k.table[k.n - 1] - (double)k.table[k.n - 1 - m]) / (m * dx);
    float peak = 0.f;
    for (int i = 0; i < k.n; ++i) {
        if (!std::isfinite(k.table[i])) return false;
        peak = std::max(peak, std::fabs(k.table[i]));
    }
    // an even kernel's corrections take its weight at the end to be zero
    if (W % 2 == 0 && !(std::fabs(k.table[k.n - 1]) <= 1e-6 * peak)) return false;
    constexpr int D = Fits::D, M = Fits::kSamples, ME = Fits::kEndSamples;
    double c[D + 1], w0[D + 1], y[M];
    auto value = [](const double (&p)[D + 1], double f) {
        double r = p[D];
        for (int d = D - 1; d >= 0; --d) r = r * f + p[d];
        return r;
    };
    for (int t = 0; t < Fits::kTaps; ++t) {
        const double at = t - 0.5 * (W - 1);
        for (int i = 0; i < M; ++i) {
            const double ax = std::fabs(at - fits.x[i]);
            y[i] = ax <= hw ? weight(ax) : (double)k.table[k.n - 1] + slope * (ax - hw);
        }
        for (int d = 0; d <= D; ++d) {
            const double* row = &fits.cell[t][(size_t)d * M];
            c[d] = 0.;
            for (int i = 0; i < M; ++i) c[d] += row[i] * y[i];
        }
        if (2 * t + 1 == W)
            for (int d = 1; d <= D; d += 2) c[d] = 0.;   // the middle tap is even
        for (int i = 0; i <= 400; ++i) {
            const double f = Fits::F * (i / 200. - 1.), ax = std::fabs(at - f);
            if (ax <= hw && !(std::fabs(value(c, f) - weight(ax)) <= 1e-4 * peak)) return false;
        }
        for (int d = 0; d <= bp::kLineDegree; ++d) {
            a->farrow[d][t] = d <= D ? (float)c[d] : 0.f;
            if (t == 0 && d <= D) w0[d] = c[d];
        }
    }
    // weights d bins past a cell's end: the tap that entered, and the
    // continuation of the one that left
    for (int s = 0; s < 2; ++s) {
        double ce[bp::kEndDegree + 1];
        for (int d = 0; d <= bp::kEndDegree; ++d) {
            ce[d] = 0.;
            for (int i = 0; i < ME; ++i) {
                const double past = Fits::E + fits.xe[i];
                ce[d] += fits.end[(size_t)d * ME + i] * value(w0, s == 0 ? 0.5 - past : 0.5 + past);
            }
        }
        // about the cell's end: substitute x - E
        double r[bp::kEndDegree + 1] = {};
        for (int d = bp::kEndDegree; d >= 0; --d) {
            for (int q = bp::kEndDegree; q >= 0; --q)
                r[q] = (q > 0 ? r[q - 1] : 0.) - Fits::E * r[q] + (q == 0 ? ce[d] : 0.);
        }
        // to the limit of the cell's weights, which imply it for smooth kernels
        for (int i = 0; i < ME; ++i) {
            const double past = Fits::E + fits.xe[i];
            const double want = s == 0 ? weight(hw - past) : value(w0, 0.5 + past);
            double got = r[bp::kEndDegree];
            for (int d = bp::kEndDegree - 1; d >= 0; --d) got = got * past + r[d];
            if (!(std::fabs(got - want) <= 1e-4 * peak)) return false;
        }
        for (int d = 0; d <= bp::kEndDegree; ++d) (s == 0 ? a->w_in : a->w_out)[d] = (float)r[d];
    }
    return true;
}

bool build_line_table(const bp_kernel& k, int W, bp::LineArgs* a)
{
    if (2.0 * k.halfwidth != (double)W) return false;
    return W == 8 ? fit_line_table<8>(k, a) : W == 9 ? fit_line_table<9>(k, a) : false;
}

// Plain-sum table of TabulatedKernel<float> (core/Kernels.icc:137-154): entry
// i holds (t_i, t_{i+1} - t_i) as doubles with the difference formed in float,
// as the reference's evaluation forms it; entry n - 1 holds (t_{n-2} +
// (t_{n-1} - t_{n-2}), t_{n-1} - t_{n-2}), what the reference's clamp of the
// index to n - 2 evaluates for |x| at the half width.
void build_plain_table(const bp_kernel& k, std::vector<double>& out)
{
    const int n = k.n;
    out.assign((size_t)2 * n, 0.0);
    for (int i = 0; i + 1 < n; ++i) {
        out[2 * i] = (double)k.table[i];
        out[2 * i + 1] = (double)(float)(k.table[i + 1] - k.table[i]);
    }
    const double d = (double)(float)(k.table[n - 1] - k.table[n - 2]);
    out[2 * (n - 1)] = (double)k.table[n - 2] + d;
    out[2 * (n - 1) + 1] = d;
}

// The scratch region of bp_backproject_noalloc: one array per device, part of
// the library's code object, held until the process ends.  Host code never
// passes `scratch` itself (in host code the name is a stand-in, not a device
// address): bp_context_create looks up each device's address once, with that
// device current, and every use goes through that address.
// Behind the part that limits what a call may hold lies room for the strips of
// the line-interpolated sum, so that which sum a pixel takes does not depend on
// how full the first part is.
constexpr size_t kNoAllocScratchBytes = size_t(BP_NOALLOC_SCRATCH_MIB) << 20;
constexpr size_t kNoAllocLineBytes = size_t(32) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes + kNoAllocLineBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_addr[kMaxDevices] = {};

// Device address of `scratch` on the current device `device`.
int scratch_address(int device, unsigned char** addr)
{
    *addr = nullptr;
    if (device < 0 || device >= kMaxDevices)
        return fail(BP_ERR_INVALID_ARGUMENT, "device index beyond the library's device table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_addr[device] == nullptr) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            (void)hipGetLastError();
            return fail(BP_ERR_HIP, std::string("hipGetSymbolAddress of the no-alloc scratch failed: ") +
                                        hipGetErrorString(e));
        }
        g_scratch_addr[device] = static_cast<unsigned char*>(p);
    }
    *addr = g_scratch_addr[device];
    return BP_SUCCESS;
}

}  // namespace

extern "C" {

const char* bp_last_error_message(void) { return g_msg.c_str(); }

int64_t bp_scratch_bytes_per_pixel(int precision)
{
    return (int64_t)sizeof(bp::PixGeom) +
           (precision == BP_PRECISION_SPLIT ? (int64_t)sizeof(bp::PixSplit) : 0);
}

int bp_context_create(int device, bp_context** ctx)
try {
    if (ctx == nullptr) return fail(BP_ERR_INVALID_ARGUMENT, "ctx is null");
    int ndev = 0;
    hipError_t e = hipGetDeviceCount(&ndev);
    if (e != hipSuccess || ndev == 0)
        return fail(BP_ERR_HIP, "no HIP device available (isce3_amd needs an MI355X GPU)");
    if (device < 0 || device >= ndev) return fail(BP_ERR_INVALID_ARGUMENT, "invalid device index");
    BP_HIP_CHECK(hipSetDevice(device));
    auto* c = new bp_context();
    c->device = device;
    if (hipDeviceGetAttribute(&c->n_cu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
        c->n_cu < 1)
        c->n_cu = 256;
    bool made = c->branch.create();
    for (auto& ev : c->ev) made = made && hipEventCreate(&ev) == hipSuccess;
    if (!made) {
        c->branch.destroy();
        for (auto& ev : c->ev)
            if (ev) (void)hipEventDestroy(ev);
        delete c;
        return fail(BP_ERR_HIP, "hipEventCreate failed");
    }
    // a failed lookup disables bp_backproject_noalloc only
    if (scratch_address(device, &c->scratch) != BP_SUCCESS) {
        c->scratch = nullptr;
        c->scratch_err = g_msg;
        g_msg.clear();
    }
    *ctx = c;
    return BP_SUCCESS;
} catch (...) {
    return bp_host_exception();
}

}  // extern "C"

namespace {

void free_static(StaticData& s)
{
    DevBuf* bufs[] = {&s.table, &s.table2, &s.poly, &s.poly2, &s.in_pos, &s.in_vel, &s.out_pos,
                      &s.out_vel, &s.in_dop, &s.out_dop, &s.dem, &s.pulse_pv, &s.sinc};
    for (DevBuf* b : bufs)
        if (b->ptr && !b->fixed) (void)hipFree(b->ptr);
}

void free_scratch(Scratch& s)
{
    DevBuf* bufs[] = {&s.geom, &s.split, &s.flags, &s.desc, &s.strips, &s.lines, &s.parts};
    for (DevBuf* b : bufs)
        if (b->ptr && !b->fixed) (void)hipFree(b->ptr);
}

void free_host_path(HostPath& h)
{
    DevBuf* bufs[] = {&h.win[0], &h.win[1], &h.band_desc, &h.band_win, &h.carry};
    for (DevBuf* b : bufs)
        if (b->ptr && !b->fixed) (void)hipFree(b->ptr);
    for (auto* p : h.stage)
        if (p) (void)hipHostFree(p);
    if (h.h_win) (void)hipHostFree(h.h_win);
    if (h.h_bad) (void)hipHostFree(h.h_bad);
    hipEvent_t evs[] = {h.stage_ev[0], h.stage_ev[1], h.win_ev, h.copied_ev, h.sum_ev[0], h.sum_ev[1]};
    for (hipEvent_t e : evs)
        if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : h.timing)
        if (e) (void)hipEventDestroy(e);
    if (h.copy) (void)hipStreamDestroy(h.copy);
}

}  // namespace

extern "C" int bp_context_limit_workspace(bp_context* c, int64_t bytes)
{
    if (c == nullptr) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    c->workspace_limit = bytes < 0 ? -1 : bytes;
    return BP_SUCCESS;
}

extern "C" int bp_context_destroy(bp_context* c)
try {
    if (c == nullptr) return BP_SUCCESS;
    (void)hipSetDevice(c->device);
    (void)hipDeviceSynchronize();
    free_static(c->st);
    free_scratch(c->sc);
    free_host_path(c->hp);
    c->branch.destroy();
    for (auto& ev : c->ev)
        if (ev) (void)hipEventDestroy(ev);
    delete c;
    return BP_SUCCESS;
} catch (...) {
    return bp_host_exception();
}

namespace {

// Workspace of the line-interpolated sum at most; more strips run in groups.
constexpr size_t kLineBytes = size_t(1536) << 20;
// ... and that of one strip (300,000 pulses of aperture), for which every call
// has room.
constexpr size_t kStripBytes = size_t(24) << 20;
constexpr int kFlagWords = 16;  // flag words in front of the per-grid flags

// Arguments shared by every output block of a call (the raw set and its
// geometry, the output orbit/Doppler, DEM, kernel and parameters).
struct CallArgs {
    const bp_orbit* out_orbit;
    const bp_lut2d* out_doppler;
    const bp_radar_geometry* in_geometry;
    const bp_dem* dem;
    double fc, ds;
    const bp_kernel* kernel;
    int tropo;
    const bp_rdr2geo_params* r2g;
    const bp_geo2rdr_params* g2r;
    const void* in_dev;
    int precision;
};

// Validated launch options.
struct Opts {
    int tile_rows, chunk, order, blocks_per_cu, lane_rows;
    bool staged;
    // line-interpolated sum: lines per strip, at most; bins that two lines may lie
    // apart per second between them; the input's range spacing
    int strip_rows;
    double strip_shift, strip_dr;
};

// Argument rules of focus/Backproject.cpp:77-92, the pybind binding
// (focus/Backproject.cpp:97-135) and DryTroposphereModel.cpp:20-33.
// Returns the kernel width on success through *width.
int check_call(const CallArgs& a, int* width)
{
    if (!a.out_orbit || !a.out_doppler || !a.in_geometry || !a.dem || !a.kernel || !a.r2g || !a.g2r)
        return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    if (a.tropo != BP_TROPO_NODELAY && a.tropo != BP_TROPO_TSX)
        return fail(BP_ERR_INVALID_ARGUMENT, "unexpected dry troposphere model");
    if (a.precision != BP_PRECISION_PLAIN && a.precision != BP_PRECISION_SPLIT)
        return fail(BP_ERR_INVALID_ARGUMENT, "unknown precision mode");
    const bp_grid& gi = a.in_geometry->grid;
    if (gi.length < 0 || gi.width < 0) return fail(BP_ERR_INVALID_ARGUMENT, "negative grid size");
    if (gi.length > INT32_MAX || gi.width > INT32_MAX)
        return fail(BP_ERR_INVALID_ARGUMENT, "grid size exceeds int range");
    if (!(gi.prf > 0)) return fail(BP_ERR_INVALID_ARGUMENT, "PRF must be positive");
    if (!(a.fc > 0)) return fail(BP_ERR_INVALID_ARGUMENT, "center frequency must be positive");
    if (!(a.ds > 0)) return fail(BP_ERR_INVALID_ARGUMENT, "azimuth resolution must be positive");
    const bp_kernel* k = a.kernel;
    if (k->n < 2 || k->table == nullptr || !(k->halfwidth > 0))
        return fail(BP_ERR_INVALID_ARGUMENT, "kernel table needs at least two samples");
    *width = (int)std::ceil(2.0 * k->halfwidth);
    if (*width < bp::kMinKernelWidth || *width > bp::kMaxKernelWidth)
        return fail(BP_ERR_INVALID_ARGUMENT,
                    "kernel width must be in [" + std::to_string(bp::kMinKernelWidth) + ", " +
                        std::to_string(bp::kMaxKernelWidth) + "] taps (got " +
                        std::to_string(*width) + ")");
    if (k->n > (1 << 20)) return fail(BP_ERR_INVALID_ARGUMENT, "kernel table exceeds 2^20 samples");
    const bp_dem* dem = a.dem;
    if (dem->have_raster) {
        bp::Proj pj;
        if (!bp::proj_init(dem->epsg, &pj))
            return fail(BP_ERR_RUNTIME, "Unknown EPSG code (in factory): " + std::to_string(dem->epsg));
        if (!dem_method_ok(dem->method))
            return fail(BP_ERR_INVALID_ARGUMENT, "unsupported DEM interpolation method " + std::to_string(dem->method));
        if (dem->width < 4 || dem->length < 4 || dem->data == nullptr)
            return fail(BP_ERR_INVALID_ARGUMENT, "DEM raster must be at least 4x4");
    }
    int rc;
    if ((rc = check_orbit(*a.out_orbit, "output geometry")) != BP_SUCCESS) return rc;
    if ((rc = check_orbit(a.in_geometry->orbit, "input geometry")) != BP_SUCCESS) return rc;
    if ((rc = check_lut(*a.out_doppler, "output geometry")) != BP_SUCCESS) return rc;
    if ((rc = check_lut(a.in_geometry->doppler, "input geometry")) != BP_SUCCESS) return rc;
    // Pulse times must lie in the input orbit: Orbit::interpolate with the
    // default border mode throws OutOfRange (Backproject.cpp:101-106).
    const int64_t na = gi.length;
    if (na > 0) {
        const bp_orbit& io = a.in_geometry->orbit;
        const double ostart = io.t0, oend = io.t0 + (io.n - 1) * io.dt;
        const double in_dt = 1.0 / gi.prf;
        const double tf = gi.sensing_start, tl = gi.sensing_start + (na - 1) * in_dt;
        if (tf < ostart || tf > oend || tl < ostart || tl > oend)
            return fail(BP_ERR_OUT_OF_RANGE, orbit_err_string(BP_ORBIT_INTERP_DOMAIN_ERROR));
    }
    return BP_SUCCESS;
}

int check_options(const bp_options* options, Opts* o)
{
    bp_options opt{};
    if (options) opt = *options;
    o->tile_rows = opt.tile_rows == 0 ? 1 : opt.tile_rows;
    if (o->tile_rows != 1 && o->tile_rows != 2 && o->tile_rows != 4 && o->tile_rows != 8)
        return fail(BP_ERR_INVALID_ARGUMENT, "tile_rows must be 1, 2, 4 or 8");
    o->chunk = opt.chunk == 0 ? 32 : opt.chunk;
    // the split sum steps the phase by its first two differences between folds:
    // the third-difference term it leaves out grows as chunk^3
    if (o->chunk < 1 || o->chunk > BP_MAX_CHUNK)
        return fail(BP_ERR_INVALID_ARGUMENT, "chunk must be in [1, 64]");
    if (opt.fit_degree != 0 && opt.fit_degree != bp::kFitDegree)
        return fail(BP_ERR_INVALID_ARGUMENT, "fit_degree must be 4");
    if (opt.order < 0 || opt.order > 2) return fail(BP_ERR_INVALID_ARGUMENT, "order must be 0, 1 or 2");
    o->order = opt.order == 1 ? 0 : 1;
    if (opt.blocks_per_cu < 0 || opt.blocks_per_cu > 16)
        return fail(BP_ERR_INVALID_ARGUMENT, "blocks_per_cu must be in [0, 16]");
    o->blocks_per_cu = opt.blocks_per_cu;
    if (opt.staged != 0 && opt.staged != 1) return fail(BP_ERR_INVALID_ARGUMENT, "staged must be 0 or 1");
    o->staged = opt.staged == 1;
    if (opt.lane_rows < 0 || opt.lane_rows > 2) return fail(BP_ERR_INVALID_ARGUMENT, "lane_rows must be 0, 1 or 2");
    o->lane_rows = opt.lane_rows;  // 0: resolved by check_lane_rows
    o->strip_rows = bp::kStripLines;
    o->strip_shift = 0.;
    o->strip_dr = 1.;
    return BP_SUCCESS;
}

// Two lines per lane need the split kernel with gathered taps; lane_rows 0
// takes them where offered for kernel widths up to 9 (wider two-line kernels
// exceed the 128 registers of four waves per SIMD and spill, so one line per
// lane is their default).
int check_lane_rows(Opts& o, int precision, int width)
{
    const bool offered = precision == BP_PRECISION_SPLIT && !o.staged;
    if (o.staged && (precision != BP_PRECISION_SPLIT || (width != 8 && width != 9)))
        return fail(BP_ERR_INVALID_ARGUMENT, "staged 1 needs split precision and kernel width 8 or 9");
    if (o.lane_rows == 0) o.lane_rows = offered && width <= 9 ? 2 : 1;
    if (o.lane_rows == 2 && !offered)
        return fail(BP_ERR_INVALID_ARGUMENT,
                    "lane_rows 2 needs split precision and staged 0");
    return BP_SUCCESS;
}

int check_blocks(bp_out_block* blocks, int n_blocks, int64_t* npix)
{
    if (n_blocks < 0 || (n_blocks > 0 && blocks == nullptr))
        return fail(BP_ERR_INVALID_ARGUMENT, "invalid output block list");
    *npix = 0;
    for (int b = 0; b < n_blocks; ++b) {
        blocks[b].failed = 0;
        const int rc = bp::check_out_block(blocks[b]);
        if (rc != BP_SUCCESS) return rc;
        *npix += blocks[b].grid.length * blocks[b].grid.width;
    }
    return BP_SUCCESS;
}

// The strips of a grid of d.map's size and d's spacings: equal heights of at
// most o.strip_rows lines, multiples of 16 so that no wavefront tile straddles
// two.  Returns their number.  None where no full strip could qualify, by
// twice the limits: columns off the input's bins, or lines too far apart.  Such
// grids need no fit of their strips (20 us, and four kernels of nothing).
int64_t map_strips(bp::OutDesc& d, const Opts& o)
{
    const int64_t ny = (d.map.length + o.strip_rows - 1) / o.strip_rows;
    const int64_t rows = (d.map.length + ny - 1) / ny;
    d.strip_rows = (int32_t)std::min<int64_t>(o.strip_rows, (rows + 15) / 16 * 16);
    d.strips_x = (int32_t)((d.map.width + 63) / 64);
    d.strips_y = (int32_t)((d.map.length + d.strip_rows - 1) / d.strip_rows);
    const double drift =
        std::fabs(d.dr / o.strip_dr - 1.) * (double)(std::min<int64_t>(d.map.width, 64) - 1);
    const double apart = 0.5 * std::min<int64_t>(d.map.length, d.strip_rows) * d.dt * o.strip_shift;
    if (drift > 2. * (double)bp::kLineColumnTol || apart > 2. * (double)bp::kLineMaxShift) {
        d.strips_x = d.strips_y = 0;
        d.strip_info = -1;
    }
    return (int64_t)d.strips_x * d.strips_y;
}

// Header and descriptors of the non-empty blocks, written to `dst` (room for
// sizeof(BatchHeader) + max_grids descriptors); block_of_grid maps grids back.
int plan_batch(const bp_out_block* blocks, int n_blocks, const Opts& o, int32_t* d_failed,
               unsigned char* dst, int max_grids, bp::BatchHeader* hdr,
               std::vector<int>& block_of_grid)
{
    block_of_grid.clear();
    auto* descs = reinterpret_cast<bp::OutDesc*>(dst + sizeof(bp::BatchHeader));
    int64_t n_seq = 0, n_rec = 0, n_strips = 0;
    int g = 0, no_strips = 0;
    for (int b = 0; b < n_blocks; ++b) {
        const bp_grid& go = blocks[b].grid;
        if (go.length * go.width == 0) continue;
        if (g >= max_grids) return fail(BP_ERR_INVALID_ARGUMENT, "too many output blocks");
        bp::OutDesc d;
        std::memset(&d, 0, sizeof(d));
        d.map = make_map(go.length, go.width, o.tile_rows, o.order, o.lane_rows);
        d.t0 = go.sensing_start;
        d.dt = 1.0 / go.prf;
        d.r0 = go.starting_range;
        d.dr = go.range_pixel_spacing;
        d.side = go.look_side;
        d.seq_base = n_seq;
        d.rec_base = n_rec;
        d.out = static_cast<float2*>(blocks[b].out_dev);
        d.height = blocks[b].height_dev;
        d.failed = d_failed + g;
        d.strip_seq = n_strips;
        d.strip_info = n_strips;
        const int64_t strips = map_strips(d, o);
        if (strips == 0) no_strips = 1;
        n_strips += strips;
        n_seq += d.map.n_tiles;
        n_rec += go.length * go.width;
        std::memcpy(descs + g, &d, sizeof(d));
        block_of_grid.push_back(b);
        ++g;
    }
    std::memset(hdr, 0, sizeof(*hdr));
    hdr->n_seq = n_seq;
    hdr->n_groups = (n_seq + 3) / 4;
    hdr->n_geom_groups = (n_seq * o.lane_rows + 3) / 4;
    hdr->n_grids = g;
    hdr->lane_rows = o.lane_rows;
    hdr->n_strips = n_strips;
    hdr->no_strips = no_strips;
    if (hdr->n_geom_groups > INT32_MAX / 2) return fail(BP_ERR_INVALID_ARGUMENT, "too many output pixels");
    std::memcpy(dst, hdr, sizeof(*hdr));
    return BP_SUCCESS;
}

// Upload the orbits, Doppler tables, DEM and kernel tables of a call.
int upload_static(StaticData& st, const CallArgs& a, int width, hipStream_t s)
{
    int rc;
    const bp_orbit& oo = *a.out_orbit;
    const bp_orbit& io = a.in_geometry->orbit;
    const bp_lut2d& od = *a.out_doppler;
    const bp_lut2d& id = a.in_geometry->doppler;
    if ((rc = upload(st.out_pos, oo.pos, sizeof(double) * 3 * oo.n, s))) return rc;
    if ((rc = upload(st.out_vel, oo.vel, sizeof(double) * 3 * oo.n, s))) return rc;
    if ((rc = upload(st.in_pos, io.pos, sizeof(double) * 3 * io.n, s))) return rc;
    if ((rc = upload(st.in_vel, io.vel, sizeof(double) * 3 * io.n, s))) return rc;
    if ((rc = upload(st.out_dop, od.have_data ? od.data : nullptr,
                     od.have_data ? sizeof(double) * od.width * od.length : 0, s)))
        return rc;
    if ((rc = upload(st.in_dop, id.have_data ? id.data : nullptr,
                     id.have_data ? sizeof(double) * id.width * id.length : 0, s)))
        return rc;
    if ((rc = upload(st.dem, a.dem->have_raster ? a.dem->data : nullptr,
                     a.dem->have_raster ? sizeof(float) * a.dem->width * a.dem->length : 0, s)))
        return rc;
    if ((rc = upload(st.table, a.kernel->table, sizeof(float) * a.kernel->n, s))) return rc;
    const bool sinc = a.dem->have_raster && a.dem->method == BP_DEM_SINC;
    if ((rc = upload(st.sinc, sinc ? sinc_kernel_table().data() : nullptr,
                     sinc ? sizeof(float) * sinc_kernel_table().size() : 0, s)))
        return rc;
    if (a.precision == BP_PRECISION_SPLIT) {
        build_polyphase(*a.kernel, width, st.poly_host);
        if ((rc = upload(st.poly, st.poly_host.data(), sizeof(float) * st.poly_host.size(), s)))
            return rc;
        build_pair_table(*a.kernel, width, st.poly2_host);
        if ((rc = upload(st.poly2, st.poly2_host.data(), sizeof(float) * st.poly2_host.size(), s)))
            return rc;
    } else {
        build_plain_table(*a.kernel, st.table2_host);
        if ((rc = upload(st.table2, st.table2_host.data(),
                         sizeof(double) * st.table2_host.size(), s)))
            return rc;
    }
    return BP_SUCCESS;
}

// Platform position/velocity at every pulse (plain precision).
// Whether the plain sum's chunks are worth their nodes: a pixel at the swath's
// near edge keeps the cubic's tolerance.  The cubic is off
// by the fourth derivative of the phase, at most 3 v^4 / R^3 of range in a straight
// pass, times 5,666 pulses^4 (the nodes' polynomial over 4!); the third difference
// is at most 0.86 v^3 / R^2 of range.  At 5 km, 120 m/s and L band that holds from
// a PRF of 700 Hz on; at 100 Hz, where no chunk keeps the tolerance, trying cost 28 %.
bool plain_chunks(const CallArgs& a)
{
    const bp_grid& gi = a.in_geometry->grid;
    const bp_orbit& io = a.in_geometry->orbit;
    double v2 = 0.;
    for (int i = 0; i < io.n; ++i)
        v2 = std::max(v2, io.vel[3 * i] * io.vel[3 * i] + io.vel[3 * i + 1] * io.vel[3 * i + 1] +
                              io.vel[3 * i + 2] * io.vel[3 * i + 2]);
    const double r = gi.starting_range, step = std::sqrt(v2) / gi.prf;   // metres per pulse
    const double per_metre = 2. * a.fc / bp::kC;
    const double off = per_metre * 5666. * 3. * step * step * step * step / (r * r * r);
    const double eps = 2. * M_PI * per_metre * 0.86 * step * step * step / (r * r);
    return r > 0. && off <= std::max(bp::kCubicTol, bp::kCubicUlps * per_metre * r) &&
           eps <= bp::kCubicEps;
}

int pulse_states(StaticData& st, const CallArgs& a, int32_t* d_flags, hipStream_t s)
{
    if (a.precision != BP_PRECISION_PLAIN) return BP_SUCCESS;
    const bp_grid& gi = a.in_geometry->grid;
    int rc;
    if ((rc = ensure(st.pulse_pv, sizeof(double) * bp::kPulseRecDoubles * std::max<int64_t>(gi.length, 1))))
        return rc;
    if (gi.length > 0)
        BP_HIP_CHECK(bp::launch_pulse_orbit(dev_orbit(a.in_geometry->orbit, st.in_pos, st.in_vel),
                                            gi.sensing_start, 1.0 / gi.prf, (int)gi.length,
                                            static_cast<double*>(st.pulse_pv.ptr), d_flags, s));
    return BP_SUCCESS;
}

// Everything the launches of one step need, with device pointers.
struct Step {
    bp::GeomArgs ga;
    bp::SumArgs sa;
    int width, precision;
    bool staged, pair;
    int geom_grid, sum_grid;
    int32_t* flags;
    int flag_words;
    hipEvent_t ev[3];  // null: no timing
    // line-interpolated sum (split; lines false: every pixel at every pulse)
    int segs;              // plain: segments with wavefronts of their own
    bool lines;
    const Branch* branch;  // lines: strips that are left run beside them, or null
    bp::LineArgs la;
    int64_t n_strips;      // of the batch (the fit's grid)
    int64_t group_strips;  // strips the workspace holds
};

// What the line-interpolated sum needs to know before it runs: fixed by the
// input geometry, the resolution and the kernel, so that an output's result
// does not depend on what it is focused with.
struct LinePlan {
    bool on;
    int rows, chunk_log2, slots;
    double shift, dr;     // Opts::strip_shift, strip_dr
    size_t strip_bytes;
    bp::LineArgs table;   // the weight polynomials
};

// Strip height: the most lines (64, 32, 16) whose range positions stay within
// kLineMaxShift of the middle line's at the aperture's ends, where adjacent
// lines are P' / (fc dtau) bins apart, P' = v |p| / (|x| 2 ds prf) cycles per
// pulse (ds = 6 m at 7.5 km/s and 1520 Hz: 0.46; 0.28 bins over 32 lines).  A
// squint adds its Doppler's part: at 400 Hz the far end has 0.44 bins, and strips
// of 64 lines would mostly fall to the pixel-by-pixel sum.
// Chunks of 64 pulses, of 32 where a strip's lines would turn by more than
// the nodes interpolate within 64.
LinePlan plan_lines(const CallArgs& a, int width, const Opts& o)
{
    LinePlan p{};
    const bp_grid& gi = a.in_geometry->grid;
    if (a.precision != BP_PRECISION_SPLIT || o.staged || o.lane_rows != 2 || gi.length < 1 ||
        gi.width < 32 || gi.width >= (1 << 28))
        return p;
    if (!build_line_table(*a.kernel, width, &p.table)) return p;
    const bp_orbit& io = a.in_geometry->orbit;
    double vmin = INFINITY, vmax = 0., pmax = 0.;
    for (int i = 0; i < io.n; ++i) {
        const double v = std::sqrt(io.vel[3 * i] * io.vel[3 * i] + io.vel[3 * i + 1] * io.vel[3 * i + 1] +
                                   io.vel[3 * i + 2] * io.vel[3 * i + 2]);
        const double q = std::sqrt(io.pos[3 * i] * io.pos[3 * i] + io.pos[3 * i + 1] * io.pos[3 * i + 1] +
                                   io.pos[3 * i + 2] * io.pos[3 * i + 2]);
        vmin = std::min(vmin, v);
        vmax = std::max(vmax, v);
        pmax = std::max(pmax, q);
    }
    const double dt = 1.0 / gi.prf, wvl = bp::kC / a.fc;
    const double inv_k = wvl / (2.0 * gi.range_pixel_spacing);
    const double ratio = pmax / 6.33e6;   // |p| / |x|
    if (!(vmin > 0.) || !(gi.starting_range > 0.) || !(gi.range_pixel_spacing > 0.)) return p;
    // sine of the angle off broadside: half the aperture, the Doppler at a few
    // points of the input grid, and what the pulses cover
    const double half = wvl * ratio / (4.0 * a.ds);
    double fd = 0.;
    const bp::Lut2d dop = host_lut(a.in_geometry->doppler);
    for (int i = 0; i < 9; ++i)
        fd = std::max(fd, std::fabs(bp::lut2d_eval(
                              dop, gi.sensing_start + 0.5 * (i / 3) * (gi.length - 1.) * dt,
                              gi.starting_range + 0.5 * (i % 3) * (gi.width - 1.) * gi.range_pixel_spacing)));
    const double squint = 0.5 * wvl * fd / vmin;
    const double seen = squint + std::min(half, vmax * dt * gi.length / gi.starting_range);
    const double per_sine = 2.0 * vmax / wvl * inv_k;   // bins per second between lines
    const double shift = dt * per_sine * std::max(half, squint > 0. ? seen : 0.);
    p.shift = per_sine * seen;
    p.dr = gi.range_pixel_spacing;
    for (p.rows = bp::kStripLines; p.rows >= 16; p.rows /= 2)
        if (0.5 * p.rows * shift * 1.05 <= (double)bp::kLineMaxShift) break;
    if (p.rows < 16) return p;
    const double turn = 2.0 * vmax * vmax * dt * dt / (wvl * gi.starting_range);
    const double x64 = 2. * M_PI * 32. * 0.5 * p.rows * turn + M_PI * 0.5 * p.rows * shift;
    p.chunk_log2 = x64 <= 0.98 * (p.rows > 32 ? bp::kLineBound8 : bp::kLineBound6) ? 6 : 5;
    const double rmax = 1.02 * (gi.starting_range + gi.width * gi.range_pixel_spacing);
    const double pulses = std::min((double)gi.length, wvl * rmax * ratio / (2. * a.ds) / vmin / dt + 8.);
    p.slots = (int)(pulses / (1 << p.chunk_log2)) + 3;
    p.table.n_sums = 8 + (a.tropo != BP_TROPO_NODELAY ? bp::kSlopeNodes : 0);
    p.strip_bytes = bp::line_strip_bytes(p.slots, p.table.n_sums);
    p.on = p.strip_bytes <= kStripBytes;
    return p;
}

void use_plan(Opts& o, const LinePlan& p)
{
    if (!p.on) return;
    o.strip_rows = p.rows;
    o.strip_shift = p.shift;
    o.strip_dr = p.dr;
}

// Segments of the plain sum that get wavefronts of their own (0: none).  The
// chip holds 4,096 of its wavefronts: 256 x 256 pixels are 1,024, each with
// 512 pulses to sum one after the other, and 301 x 1003 pixels are 4,816, so that
// a second round runs 18% full.  By segments these take 0.34 instead of
// 0.50 ms and 5.8 instead of 8.3 ms.  From four rounds on (kPlainWaves) the
// last one costs less than the segments' sums, which are kept while they fit
// kPartBytes.
constexpr int64_t kPlainWaves = 16384;
constexpr size_t kPartBytes = size_t(256) << 20;

// The lesser of a workspace bound and the context's own limit (none below 0).
size_t limited(size_t bytes, int64_t limit)
{
    return limit < 0 ? bytes : std::min(bytes, (size_t)limit);
}

int plain_segments(const CallArgs& a, int64_t n_seq, int64_t n_rec, int64_t limit)
{
    if (a.precision != BP_PRECISION_PLAIN || n_seq >= kPlainWaves) return 0;
    const int64_t segs = (a.in_geometry->grid.length + bp::kPlainSeg - 1) / bp::kPlainSeg;
    if (segs < 2 || segs > 65535 ||
        (double)segs * n_rec * sizeof(double2) > (double)limited(kPartBytes, limit))
        return 0;
    return (int)segs;
}

// Pixels whose segment sums a scene holds (0: no segments of their own).
int64_t scene_part_records(const CallArgs& a, int64_t max_pixels, int64_t limit)
{
    const int64_t length = a.in_geometry->grid.length;
    if (a.precision != BP_PRECISION_PLAIN || length <= bp::kPlainSeg) return 0;
    const int64_t segs = (length + bp::kPlainSeg - 1) / bp::kPlainSeg;
    return std::min({max_pixels, kPlainWaves * 64,
                     (int64_t)(limited(kPartBytes, limit) / (segs * sizeof(double2)))});
}

// Strips of max_pixels pixels in max_blocks blocks at most: a block of l x w
// pixels has ceil(l / rows) ceil(w / 64) <= l w / rows + 1, rows <= 64.
int64_t most_strips(int64_t max_pixels, int max_blocks, int rows)
{
    return max_pixels / rows + std::min<int64_t>(max_blocks, max_pixels);
}

// ... and those that a scene has workspace for at a time: more than blocks of
// some hundred pixels a side need; narrower ones run in groups.
int64_t scene_strips(int64_t max_pixels, int max_blocks, int rows)
{
    return std::min(most_strips(max_pixels, max_blocks, rows),
                    max_pixels / (rows * 64) * 5 / 4 + 2 * std::min(max_blocks, 64) + 8);
}

// Strips whose workspace is taken at once for n of them, beside the StripInfo
// of `records` strips.
int64_t line_group(const LinePlan& p, int64_t n, int64_t records, int64_t limit)
{
    const int64_t left = (int64_t)limited(kLineBytes, limit) -
                         (limit < 0 ? 0 : (int64_t)sizeof(bp::StripInfo) * records);
    return std::min<int64_t>(n, std::max<int64_t>(left / (int64_t)p.strip_bytes, 1));
}

// StripInfo for `records` strips and workspace for n, or as many of them at once
// as limit and device have room for: their number.  Results do not depend on
// it, but for a device without room for a single strip (0.3 to 0.5 MB), where the
// call sums pixel by pixel (0).
int64_t alloc_lines(const LinePlan& p, int64_t n, int64_t records, int64_t limit, Scratch& sc)
{
    if (ensure(sc.strips, sizeof(bp::StripInfo) * records) != BP_SUCCESS) return 0;
    for (int64_t group = line_group(p, n, records, limit); group > 0; group /= 2)
        if (ensure(sc.lines, p.strip_bytes * group) == BP_SUCCESS) return group;
    return 0;
}

// Point a step at the line-interpolated sum with a workspace of `group`
// strips.
void set_lines(struct Step& sp, const LinePlan& p, const Scratch& sc, const CallArgs& a, int64_t n,
               int64_t group);

void build_step(Step& sp, const StaticData& st, const Scratch& sc, const CallArgs& a, int width,
                const Opts& o, int n_cu)
{
    const bp_grid& gi = a.in_geometry->grid;
    const double swst = 2. * gi.starting_range / bp::kC;
    const double dtau = 2. * gi.range_pixel_spacing / bp::kC;
    const auto* batch = static_cast<const bp::BatchHeader*>(sc.desc.ptr);
    int32_t* d_flags = static_cast<int32_t*>(sc.flags.ptr);

    bp::Dem ddem = host_dem(*a.dem);
    ddem.data = static_cast<const float*>(st.dem.ptr);
    ddem.sinc = static_cast<const float*>(st.sinc.ptr);

    bp::GeomArgs& ga = sp.ga;
    std::memset(&ga, 0, sizeof(ga));
    ga.batch = batch;
    ga.in_side = gi.look_side;
    ga.kwidth = width;
    ga.nr = (int32_t)gi.width;
    ga.in_t0 = gi.sensing_start;
    ga.in_dt = 1.0 / gi.prf;
    ga.na = (int32_t)gi.length;
    ga.tropo = a.tropo;
    ga.swst = swst;
    ga.dtau = dtau;
    ga.wvl = bp::kC / a.fc;
    ga.fc = a.fc;
    ga.ds = a.ds;
    ga.out_orbit = dev_orbit(*a.out_orbit, st.out_pos, st.out_vel);
    ga.in_orbit = dev_orbit(a.in_geometry->orbit, st.in_pos, st.in_vel);
    ga.out_dop = dev_lut(*a.out_doppler, st.out_dop);
    ga.in_dop = dev_lut(a.in_geometry->doppler, st.in_dop);
    ga.dem = ddem;
    ga.r2g = {a.r2g->tol_height, a.r2g->look_min, a.r2g->look_max};
    ga.g2r.tol_aztime = a.g2r->tol_aztime;
    ga.g2r.have_time_start = a.g2r->have_time_start;
    ga.g2r.have_time_end = a.g2r->have_time_end;
    ga.g2r.time_start = a.g2r->time_start;
    ga.g2r.time_end = a.g2r->time_end;
    ga.want_split = a.precision == BP_PRECISION_SPLIT;
    ga.geom = static_cast<bp::PixGeom*>(sc.geom.ptr);
    ga.split = static_cast<bp::PixSplit*>(sc.split.ptr);
    ga.flags = d_flags;
    ga.updates = reinterpret_cast<unsigned long long*>(d_flags + 8);

    bp::SumArgs& sa = sp.sa;
    std::memset(&sa, 0, sizeof(sa));
    sa.batch = batch;
    sa.nr = gi.width;
    sa.swst = swst;
    sa.dtau = dtau;
    sa.fc = a.fc;
    sa.inv_k = 1.0 / (a.fc * dtau);
    sa.zscale = (float)(-(double)bp::kPolyphaseRows * sa.inv_k);
    sa.halfwidth = a.kernel->halfwidth;
    sa.rdx = (float)(1.0 / (a.kernel->halfwidth / (a.kernel->n - 1.0)));
    sa.ntab = a.kernel->n;
    sa.chunk = o.chunk;
    {
        const double n = (double)o.chunk;
        sa.fold_c[0] = n;
        sa.fold_c[1] = n * (n - 1.) / 2.;
        sa.fold_c[2] = n * (n - 1.) * (n - 2.) / 6.;
        sa.fold_c[3] = n * (n - 1.) * (n - 2.) * (n - 3.) / 24.;
    }
    sa.rc = static_cast<const float2*>(a.in_dev);
    sa.pulse_pv = static_cast<const double*>(st.pulse_pv.ptr);
    sa.geom = static_cast<const bp::PixGeom*>(sc.geom.ptr);
    sa.split = static_cast<const bp::PixSplit*>(sc.split.ptr);
    sa.table = static_cast<const float*>(st.table.ptr);
    sa.poly = static_cast<const float*>(st.poly.ptr);
    sa.poly2 = static_cast<const float*>(st.poly2.ptr);
    sa.zscale2 = (float)(-(double)(1 << bp::pair_q_log2(width)) * sa.inv_k);
    sa.inv_dtau = 1.0 / dtau;
    sa.exact_width = 2.0 * a.kernel->halfwidth == (double)width;
    sa.tab2 = static_cast<const double2*>(st.table2.ptr);
    sa.chunks = a.precision == BP_PRECISION_PLAIN && plain_chunks(a);

    sp.width = width;
    sp.precision = a.precision;
    sp.staged = o.staged;
    sp.pair = o.lane_rows == 2;
    const int per_cu = o.blocks_per_cu > 0 ? o.blocks_per_cu
                                           : bp::sum_blocks_per_cu(a.precision, width, o.staged, sp.pair);
    sp.sum_grid = (n_cu * per_cu + 7) / 8 * 8;  // persistent split grid
    sp.geom_grid = 0;
    sp.flags = d_flags;
    sp.flag_words = 0;
    sp.ev[0] = sp.ev[1] = sp.ev[2] = nullptr;
    sp.lines = false;
    sp.branch = nullptr;
    sp.segs = 0;
}

void set_lines(Step& sp, const LinePlan& p, const Scratch& sc, const CallArgs& a, int64_t n,
               int64_t group)
{
    const bp_grid& gi = a.in_geometry->grid;
    bp::LineArgs& la = sp.la;
    la = p.table;
    la.batch = sp.sa.batch;
    la.rec = reinterpret_cast<bp::PixLine*>(sc.split.ptr);
    la.info = static_cast<bp::StripInfo*>(sc.strips.ptr);
    la.n_left = sp.flags + 2;
    la.rc = sp.sa.rc;
    la.nr = gi.width;
    la.inv_k = sp.sa.inv_k;
    la.in_r0 = gi.starting_range;
    la.inv_dr = 1.0 / gi.range_pixel_spacing;
    la.slots = p.slots;
    la.chunk_log2 = p.chunk_log2;
    la.s_begin = 0;
    la.s_end = group;
    la.q_begin = INT32_MIN;
    la.q_end = INT32_MAX;
    la.few = std::min(n, group) <= bp::kFewStrips ? 1 : 0;
    bp::line_place(la, static_cast<unsigned char*>(sc.lines.ptr), group);
    sp.lines = true;
    sp.n_strips = n;
    sp.group_strips = group;
    sp.ga.strips = la.info;
    sp.sa.strips = la.info;
    sp.ga.strip_pass = sp.sa.strip_pass = bp::kPassLeft | bp::kPassRedo;
    sp.sa.n_left = la.n_left;
}

// The coherent sum of a step over the descriptors at `batch` (`groups` groups of
// four wavefront tiles), reading pulse k at rc + k * nr.
int enqueue_sum(const Step& sp, const bp::BatchHeader* batch, const float2* rc, int groups,
                int64_t n_strips, hipStream_t s)
{
    bp::SumArgs sa = sp.sa;
    sa.batch = batch;
    sa.rc = rc;
    bp::GeomArgs ga = sp.ga;
    ga.batch = batch;
    if (sp.lines) {
        // The strips in groups of the workspace's size; beside them the strips
        // that did not qualify, whose pixels walk their aperture alone (1.4 ms
        // however few they are: behind the line sum a tile of 310 x 290 pixels with
        // a column of such strips took 4.80 ms, with none of its strips taken 4.46);
        // then those that met samples that are not finite.  The strips wait for the
        // other stream's fit, so that its sum, next there, has its long wavefronts
        // placed first, evenly over the SIMDs: 512 x 512 pixels of which most strips
        // are left 7.9 ms when the line sum came first, 5.0 so.
        ga.strip_pass = sa.strip_pass = bp::kPassLeft | bp::kPassRedo;
        if (sp.branch) {
            ga.strip_pass = sa.strip_pass = bp::kPassLeft;
            const hipStream_t o = sp.branch->s;
            BP_HIP_CHECK(hipEventRecord(sp.branch->part, s));
            BP_HIP_CHECK(hipStreamWaitEvent(o, sp.branch->part, 0));
            BP_HIP_CHECK(bp::launch_fit(ga, groups, o));
            BP_HIP_CHECK(hipEventRecord(sp.branch->fit, o));
            BP_HIP_CHECK(bp::launch_sum_split(sa, sp.width, sp.sum_grid, sp.staged, sp.pair, o));
            BP_HIP_CHECK(hipEventRecord(sp.branch->join, o));
            BP_HIP_CHECK(hipStreamWaitEvent(s, sp.branch->fit, 0));
            ga.strip_pass = sa.strip_pass = bp::kPassRedo;
        }
        bp::LineArgs la = sp.la;
        la.batch = batch;
        la.rc = rc;
        for (int64_t s0 = 0; s0 < n_strips; s0 += sp.group_strips) {
            const int64_t n = std::min(sp.group_strips, n_strips - s0);
            la.s_begin = s0;
            la.s_end = s0 + n;
            BP_HIP_CHECK(bp::launch_strips(la, sp.width, true, s));
        }
        if (sp.branch) BP_HIP_CHECK(hipStreamWaitEvent(s, sp.branch->join, 0));
        BP_HIP_CHECK(bp::launch_fit(ga, groups, s));
    }
    if (sp.precision == BP_PRECISION_PLAIN)
        BP_HIP_CHECK(bp::launch_sum_plain(sa, sp.width, groups, sp.segs, s));
    else
        BP_HIP_CHECK(bp::launch_sum_split(sa, sp.width, sp.sum_grid, sp.staged, sp.pair, s));
    return BP_SUCCESS;
}

// Enqueue the launches of one step: clear the flags, per-pixel geometry,
// coherent sum (with optional event records around the two passes).
int enqueue_step(const Step& sp, int groups, hipStream_t s)
{
    BP_HIP_CHECK(bp::launch_clear(sp.flags, sp.flag_words, s));
    if (sp.ev[0]) BP_HIP_CHECK(hipEventRecord(sp.ev[0], s));
    BP_HIP_CHECK(bp::launch_geometry(sp.ga, sp.geom_grid, s));
    if (sp.lines)
        BP_HIP_CHECK(bp::launch_strip_fit(sp.ga, sp.la, bp::line_grid(bp::kLineFit, 0, sp.n_strips), s));
    else if (sp.precision == BP_PRECISION_SPLIT)
        BP_HIP_CHECK(bp::launch_fit(sp.ga, groups, s));
    if (sp.ev[1]) BP_HIP_CHECK(hipEventRecord(sp.ev[1], s));
    const int rc = enqueue_sum(sp, sp.sa.batch, sp.sa.rc, groups, sp.n_strips, s);
    if (rc != BP_SUCCESS) return rc;
    if (sp.ev[2]) BP_HIP_CHECK(hipEventRecord(sp.ev[2], s));
    return BP_SUCCESS;
}

// Read the flags of a finished step into the caller's outputs.
int finish_step(const int32_t* hflags, int n_grids, const std::vector<int>& block_of_grid,
                bp_out_block* blocks, const hipEvent_t* ev, int* any_failed, bp_stats* stats)
{
    unsigned long long hupd = 0;
    std::memcpy(&hupd, hflags + 8, sizeof(hupd));
    for (int g = 0; g < n_grids; ++g) blocks[block_of_grid[g]].failed = hflags[kFlagWords + g] != 0;
    if (stats) {
        float ms = 0.f;
        if (ev[1]) {
            BP_HIP_CHECK(hipEventElapsedTime(&ms, ev[0], ev[1]));
            stats->geometry_ms = ms;
            BP_HIP_CHECK(hipEventElapsedTime(&ms, ev[1], ev[2]));
            stats->sum_ms = ms;
        }
        if (ev[0] && ev[2]) {  // calls without events report no times
            BP_HIP_CHECK(hipEventElapsedTime(&ms, ev[0], ev[2]));
            stats->step_ms = ms;
        }
        stats->updates = (int64_t)hupd;
        stats->any_failed = hflags[0] != 0;
    }
    if (hflags[1]) return fail(BP_ERR_OUT_OF_RANGE, orbit_err_string(BP_ORBIT_INTERP_DOMAIN_ERROR));
    if (any_failed) *any_failed = hflags[0] != 0;
    return hflags[0] ? BP_FAILED_TO_CONVERGE : BP_SUCCESS;
}

// Shared implementation of bp_backproject and bp_backproject_blocks: every
// output block shares the output orbit and Doppler, the input geometry, DEM,
// kernel and parameters; the pixels of all blocks are focused by one geometry
// launch and one coherent-sum launch.
// `carve`, when given, places the call's buffers in a fixed region instead of
// the context's grow-only arena (bp_backproject_noalloc).
struct Carve;
int carve_call(Carve& cv, const CallArgs& a, int width, int n_blocks, int64_t npix,
               StaticData& st, Scratch& sc);
int64_t carve_lines(Carve& cv, const LinePlan& p, int64_t n_strips, Scratch& sc);
int carve_parts(Carve& cv, size_t bytes, Scratch& sc);

int run_blocks(bp_context* c, const CallArgs& a, bp_out_block* blocks, int n_blocks,
               const bp_options* options, void* stream, int* any_failed, bp_stats* stats,
               Carve* carve = nullptr)
{
    if (any_failed) *any_failed = 0;
    if (stats) std::memset(stats, 0, sizeof(*stats));
    if (!c) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    int width = 0, rc;
    if ((rc = check_call(a, &width)) != BP_SUCCESS) return rc;
    int64_t npix = 0;
    if ((rc = check_blocks(blocks, n_blocks, &npix)) != BP_SUCCESS) return rc;
    Opts o;
    if ((rc = check_options(options, &o)) != BP_SUCCESS) return rc;
    if ((rc = check_lane_rows(o, a.precision, width)) != BP_SUCCESS) return rc;
    const bp_grid& gi = a.in_geometry->grid;
    if (npix > 0 && gi.length * gi.width > 0 && a.in_dev == nullptr)
        return fail(BP_ERR_INVALID_ARGUMENT, "in is null");
    LinePlan lp = plan_lines(a, width, o);
    use_plan(o, lp);
    StaticData fixed_st;
    Scratch fixed_sc;
    if (carve && (rc = carve_call(*carve, a, width, n_blocks, npix, fixed_st, fixed_sc)) != BP_SUCCESS)
        return rc;
    if (npix == 0) return BP_SUCCESS;
    StaticData& st = carve ? fixed_st : c->st;
    Scratch& sc = carve ? fixed_sc : c->sc;

    BP_HIP_CHECK(hipSetDevice(c->device));
    hipStream_t s = static_cast<hipStream_t>(stream);

    const int n_flag = kFlagWords + n_blocks;
    if ((rc = ensure(sc.flags, sizeof(int32_t) * n_flag))) return rc;
    c->desc_host.assign(sizeof(bp::BatchHeader) + sizeof(bp::OutDesc) * std::max(n_blocks, 1), 0);
    bp::BatchHeader hdr;
    if ((rc = plan_batch(blocks, n_blocks, o, static_cast<int32_t*>(sc.flags.ptr) + kFlagWords,
                         c->desc_host.data(), n_blocks, &hdr, c->desc_block)) != BP_SUCCESS)
        return rc;
    const int64_t n_rec = npix;

    int segs = plain_segments(a, hdr.n_seq, n_rec, c->workspace_limit);
    if (segs > 0) {
        const size_t bytes = sizeof(double2) * (size_t)segs * n_rec;
        if (carve ? carve_parts(*carve, bytes, sc) : ensure(sc.parts, bytes)) segs = 0;
        hdr.plain_segs = segs;
        std::memcpy(c->desc_host.data(), &hdr, sizeof(hdr));
    }
    if ((rc = upload_static(st, a, width, s))) return rc;
    if ((rc = upload(sc.desc, c->desc_host.data(), c->desc_host.size(), s))) return rc;
    if ((rc = ensure(sc.geom, sizeof(bp::PixGeom) * n_rec))) return rc;
    if (a.precision == BP_PRECISION_SPLIT && (rc = ensure(sc.split, sizeof(bp::PixSplit) * n_rec)))
        return rc;
    int64_t group = 0;
    if (lp.on && hdr.n_strips > 0) {
        if (carve) {
            group = carve_lines(*carve, lp, hdr.n_strips, sc);
        } else {
            group = alloc_lines(lp, hdr.n_strips, hdr.n_strips, c->workspace_limit, sc);
        }
    }
    BP_HIP_CHECK(bp::launch_clear(static_cast<int32_t*>(sc.flags.ptr), n_flag, s));
    if ((rc = pulse_states(st, a, static_cast<int32_t*>(sc.flags.ptr), s))) return rc;

    Step sp;
    build_step(sp, st, sc, a, width, o, c->n_cu);
    if (group > 0) {
        set_lines(sp, lp, sc, a, hdr.n_strips, group);
        sp.branch = &c->branch;
    }
    if (segs > 0) {
        sp.segs = segs;
        sp.sa.parts = static_cast<double2*>(sc.parts.ptr);
        sp.sa.parts_stride = n_rec;
    }
    sp.geom_grid = (int)hdr.n_geom_groups;
    sp.flag_words = 0;  // cleared above, before the pulse states
    if (stats)
        for (int i = 0; i < 3; ++i) sp.ev[i] = c->ev[i];
    if ((rc = enqueue_step(sp, (int)hdr.n_groups, s))) {
        (void)hipStreamSynchronize(c->branch.s);   // nothing of the call runs on
        return rc;
    }

    c->flags_host.assign(n_flag, 0);
    BP_HIP_CHECK(hipMemcpyAsync(c->flags_host.data(), sc.flags.ptr, sizeof(int32_t) * n_flag,
                                hipMemcpyDeviceToHost, s));
    BP_HIP_CHECK(hipStreamSynchronize(s));
    return finish_step(c->flags_host.data(), hdr.n_grids, c->desc_block, blocks, c->ev,
                       any_failed, stats);
}

// A bump allocator over a fixed device region: every buffer of a call starts
// on a 256-byte boundary; a call that does not fit fails before any launch.
struct Carve {
    unsigned char* base;
    size_t cap;
    size_t used = 0;
    int take(DevBuf& b, size_t bytes)
    {
        if (bytes == 0) bytes = 16;  // as ensure()
        const size_t off = (used + 255) & ~size_t(255);
        if (off > cap || bytes > cap - off) {
            used = cap + 1;  // mark the call as too large
            return BP_ERR_LENGTH;
        }
        b.ptr = base + off;
        b.bytes = bytes;
        b.fixed = true;
        used = off + bytes;
        return BP_SUCCESS;
    }
};

// Buffers of one bp_backproject_noalloc call, of the sizes upload_static,
// pulse_states and run_blocks ask for (a buffer that came out smaller would
// fail in ensure(), never overrun).
int carve_call(Carve& cv, const CallArgs& a, int width, int n_blocks, int64_t npix,
               StaticData& st, Scratch& sc)
{
    const bp_orbit& oo = *a.out_orbit;
    const bp_orbit& io = a.in_geometry->orbit;
    const bp_lut2d& od = *a.out_doppler;
    const bp_lut2d& id = a.in_geometry->doppler;
    const bool split = a.precision == BP_PRECISION_SPLIT;
    const int64_t na = std::max<int64_t>(a.in_geometry->grid.length, 1);
    const struct {
        DevBuf* b;
        double bytes;  // double: sizes of absurd inputs must not wrap
    } want[] = {
        {&sc.flags, 4.0 * (kFlagWords + n_blocks)},
        {&sc.desc, (double)sizeof(bp::BatchHeader) + (double)sizeof(bp::OutDesc) * std::max(n_blocks, 1)},
        {&st.out_pos, 24.0 * oo.n},
        {&st.out_vel, 24.0 * oo.n},
        {&st.in_pos, 24.0 * io.n},
        {&st.in_vel, 24.0 * io.n},
        {&st.out_dop, od.have_data ? 8.0 * od.width * od.length : 0.0},
        {&st.in_dop, id.have_data ? 8.0 * id.width * id.length : 0.0},
        {&st.dem, a.dem->have_raster ? 4.0 * a.dem->width * a.dem->length : 0.0},
        {&st.sinc, a.dem->have_raster && a.dem->method == BP_DEM_SINC
                       ? 4.0 * bp::kSincLen * bp::kSincSub : 0.0},
        {&st.table, 4.0 * a.kernel->n},
        {&st.poly, split ? 4.0 * (bp::kPolyphaseRows + 1) * bp::poly_row_floats(width) : 0.0},
        {&st.poly2, split ? 4.0 * bp::pair_table_floats(width) : 0.0},
        {&st.table2, split ? 0.0 : 16.0 * a.kernel->n},
        {&st.pulse_pv, split ? 0.0 : 8.0 * bp::kPulseRecDoubles * na},
        {&sc.geom, (double)sizeof(bp::PixGeom) * npix},
        {&sc.split, split ? (double)sizeof(bp::PixSplit) * npix : 0.0},
    };
    double total = 0.0;
    for (const auto& w : want) total += std::ceil(std::max(w.bytes, 16.0) / 256.0) * 256.0;
    if (total > (double)cv.cap)
        return fail(BP_ERR_LENGTH,
                    "bp_backproject_noalloc: the call needs " + std::to_string((long long)total) +
                        " bytes of scratch (output records " +
                        std::to_string((long long)bp_scratch_bytes_per_pixel(a.precision)) +
                        " bytes per pixel, plus orbit, Doppler, DEM and kernel tables); the "
                        "library's fixed scratch holds " + std::to_string(cv.cap) + " bytes");
    for (const auto& w : want)
        if (cv.take(*w.b, (size_t)w.bytes) != BP_SUCCESS)
            return fail(BP_ERR_LENGTH, "bp_backproject_noalloc: scratch layout overflow");
    return BP_SUCCESS;
}

// Segment sums of the plain sum in what a no-alloc call's buffers leave (the
// sums are the same without them).
int carve_parts(Carve& cv, size_t bytes, Scratch& sc)
{
    if (cv.used > cv.cap || bytes + 256 > cv.cap - cv.used) return BP_ERR_LENGTH;
    return cv.take(sc.parts, bytes);
}

// Workspace of the line-interpolated sum in what a no-alloc call's buffers
// leave and the room kept for it, which holds a strip of any call and the
// StripInfo of all that its records allow (16 lines of one pixel each).
int64_t carve_lines(Carve& cv, const LinePlan& p, int64_t n_strips, Scratch& sc)
{
    static_assert(kStripBytes + sizeof(bp::StripInfo) * (kNoAllocScratchBytes /
                  (sizeof(bp::PixGeom) + sizeof(bp::PixSplit)) / 16 + 1) + 1024 <= kNoAllocLineBytes,
                  "room for a strip");
    cv.cap = kNoAllocScratchBytes + kNoAllocLineBytes;
    const size_t info = sizeof(bp::StripInfo) * (size_t)n_strips;
    if (cv.used > cv.cap || info + p.strip_bytes + 512 > cv.cap - cv.used) return 0;
    const int64_t group =
        std::min<int64_t>(n_strips, (int64_t)((cv.cap - cv.used - info - 512) / p.strip_bytes));
    if (cv.take(sc.strips, info) != BP_SUCCESS ||
        cv.take(sc.lines, p.strip_bytes * group) != BP_SUCCESS)
        return 0;
    return group;
}

// ------------------------------------------------------------ host input
//
// Range-compressed pulses in host memory (an array or a memory map of a
// raster file): the geometry pass runs first, the union [kmin, kmax) of the
// pixels' pulse windows comes back per band of tile rows, and only those
// pulses are copied to the device, in chunks of at most `batch` pulses through
// two pinned staging buffers on a copy stream (the host reads chunk j + 1
// while chunk j is copied).  When the window of the whole block exceeds the
// device budget, the block is focused in bands of output lines with smaller
// windows; a band starts on a tile row, so its wavefront tiles, records and
// per-pixel arithmetic are those of the whole block and every result equals
// the resident call's.  Bands alternate between two window buffers when two
// fit the budget, so the copy of band b + 1 overlaps the sum of band b.

constexpr size_t kStageBytes = size_t(64) << 20;   // per pinned staging buffer

int host_path_init(HostPath& h)
{
    if (h.copy) return BP_SUCCESS;
    BP_HIP_CHECK(hipStreamCreateWithFlags(&h.copy, hipStreamNonBlocking));  // default priority
    hipEvent_t* evs[] = {&h.stage_ev[0], &h.stage_ev[1], &h.win_ev, &h.copied_ev, &h.sum_ev[0],
                         &h.sum_ev[1]};
    for (hipEvent_t* e : evs) BP_HIP_CHECK(hipEventCreateWithFlags(e, hipEventDisableTiming));
    return BP_SUCCESS;
}

int ensure_pinned(unsigned char*& p, size_t& have, size_t bytes)
{
    if (have >= bytes && p) return BP_SUCCESS;
    if (p) (void)hipHostFree(p);
    p = nullptr;
    have = 0;
    if (hipHostMalloc(reinterpret_cast<void**>(&p), bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        p = nullptr;
        return fail(BP_ERR_OUT_OF_MEMORY, "hipHostMalloc of pulse staging failed");
    }
    have = bytes;
    return BP_SUCCESS;
}

// memcpy of `bytes` from src to dst, split over up to 8 host threads for
// large copies (reading a memory-mapped raster is the slow side).
void host_copy(unsigned char* dst, const unsigned char* src, size_t bytes)
{
    const size_t kPerThread = size_t(16) << 20;
    unsigned nt = (unsigned)std::min<size_t>(8, (bytes + kPerThread - 1) / kPerThread);
    nt = std::max(1u, std::min(nt, (unsigned)bp::usable_cpus()));
    if (nt == 1) {
        std::memcpy(dst, src, bytes);
        return;
    }
    const size_t part = (bytes + nt - 1) / nt;
    std::vector<std::thread> th;
    for (unsigned t = 1; t < nt; ++t) {
        const size_t o = std::min(bytes, t * part), n = std::min(bytes - o, part);
        try {
            th.emplace_back([=] { std::memcpy(dst + o, src + o, n); });
        } catch (...) {
            std::memcpy(dst + o, src + o, n);  // no thread: copy here
        }
    }
    std::memcpy(dst, src, std::min(bytes, part));
    for (auto& x : th) x.join();
}

struct Band {
    int64_t r0, r1;   // output lines
    int32_t k0, k1;   // pulses [k0, k1) (k0 >= k1: none)
    // kWhole: both sums; kPart: the line-interpolated sum of one strip row
    // over the pulses in [k0, k1) of its window (first, last: its first and
    // last part); kTiles: the strips that sum pixel by pixel
    enum Kind { kWhole, kPart, kTiles } kind = kWhole;
    bool first = false, last = false;
};

int run_host(bp_context* c, const CallArgs& a, bp_out_block* blk, int64_t batch,
             int64_t max_window_bytes, const bp_options* options, void* stream, int* any_failed,
             bp_stats* stats, bp_host_stats* hstats)
{
    if (any_failed) *any_failed = 0;
    if (stats) std::memset(stats, 0, sizeof(*stats));
    if (hstats) std::memset(hstats, 0, sizeof(*hstats));
    if (!c) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    int width = 0, rc;
    if ((rc = check_call(a, &width)) != BP_SUCCESS) return rc;
    if (batch < 1) return fail(BP_ERR_DOMAIN, "batch size must be > 0");
    if (max_window_bytes < 0) return fail(BP_ERR_INVALID_ARGUMENT, "max_window_bytes must be >= 0");
    int64_t npix = 0;
    if ((rc = check_blocks(blk, 1, &npix)) != BP_SUCCESS) return rc;
    Opts o;
    if ((rc = check_options(options, &o)) != BP_SUCCESS) return rc;
    if ((rc = check_lane_rows(o, a.precision, width)) != BP_SUCCESS) return rc;
    const bp_grid& gi = a.in_geometry->grid;
    if (npix > 0 && gi.length * gi.width > 0 && a.in_dev == nullptr)
        return fail(BP_ERR_INVALID_ARGUMENT, "in is null");
    if (npix == 0) return BP_SUCCESS;
    const LinePlan lp = plan_lines(a, width, o);
    use_plan(o, lp);

    BP_HIP_CHECK(hipSetDevice(c->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    HostPath& hp = c->hp;
    if ((rc = host_path_init(hp))) return rc;
    // a call that fails after enqueueing work drains both streams before it
    // returns, so that the next call never refills buffers still being read
    struct Drain {
        hipStream_t a, b;
        bool armed = true;
        ~Drain()
        {
            if (armed) {
                (void)hipStreamSynchronize(a);
                (void)hipStreamSynchronize(b);
            }
        }
    } drain{s, hp.copy};

    const int n_flag = kFlagWords + 1;
    if ((rc = ensure(c->sc.flags, sizeof(int32_t) * n_flag))) return rc;
    c->desc_host.assign(sizeof(bp::BatchHeader) + sizeof(bp::OutDesc), 0);
    bp::BatchHeader hdr;
    if ((rc = plan_batch(blk, 1, o, static_cast<int32_t*>(c->sc.flags.ptr) + kFlagWords,
                         c->desc_host.data(), 1, &hdr, c->desc_block)) != BP_SUCCESS)
        return rc;
    bp::OutDesc whole;
    std::memcpy(&whole, c->desc_host.data() + sizeof(bp::BatchHeader), sizeof(whole));

    if ((rc = upload_static(c->st, a, width, s))) return rc;
    if ((rc = upload(c->sc.desc, c->desc_host.data(), c->desc_host.size(), s))) return rc;
    if ((rc = ensure(c->sc.geom, sizeof(bp::PixGeom) * npix))) return rc;
    if (a.precision == BP_PRECISION_SPLIT && (rc = ensure(c->sc.split, sizeof(bp::PixSplit) * npix)))
        return rc;
    const int64_t group =
        lp.on && hdr.n_strips > 0 ? alloc_lines(lp, hdr.n_strips, hdr.n_strips, c->workspace_limit, c->sc) : 0;
    BP_HIP_CHECK(bp::launch_clear(static_cast<int32_t*>(c->sc.flags.ptr), n_flag, s));
    if ((rc = pulse_states(c->st, a, static_cast<int32_t*>(c->sc.flags.ptr), s))) return rc;

    Step sp;
    build_step(sp, c->st, c->sc, a, width, o, c->n_cu);
    sp.geom_grid = (int)hdr.n_geom_groups;
    if (group > 0) set_lines(sp, lp, c->sc, a, hdr.n_strips, group);

    // geometry, the band windows (read back while the fit runs), the fit
    const int band_rows = whole.map.tile_rows * whole.map.lane_rows;
    const int64_t length = whole.map.length, owidth = whole.map.width;
    const int64_t n_tr = (length + band_rows - 1) / band_rows;
    if (stats) BP_HIP_CHECK(hipEventRecord(c->ev[0], s));
    BP_HIP_CHECK(bp::launch_geometry(sp.ga, sp.geom_grid, s));
    if ((rc = ensure(hp.band_win, sizeof(int32_t) * 2 * n_tr))) return rc;
    BP_HIP_CHECK(bp::launch_band_window(static_cast<const bp::PixGeom*>(c->sc.geom.ptr), length,
                                        owidth, band_rows, n_tr,
                                        static_cast<int32_t*>(hp.band_win.ptr), s));
    if (hp.h_win_words < (size_t)(2 * n_tr)) {
        unsigned char* p = reinterpret_cast<unsigned char*>(hp.h_win);
        size_t have = hp.h_win_words * sizeof(int32_t);
        if ((rc = ensure_pinned(p, have, sizeof(int32_t) * 2 * n_tr))) {
            hp.h_win = nullptr;
            hp.h_win_words = 0;
            return rc;
        }
        hp.h_win = reinterpret_cast<int32_t*>(p);
        hp.h_win_words = have / sizeof(int32_t);
    }
    BP_HIP_CHECK(hipMemcpyAsync(hp.h_win, hp.band_win.ptr, sizeof(int32_t) * 2 * n_tr,
                                hipMemcpyDeviceToHost, s));
    if (sp.lines) {
        BP_HIP_CHECK(bp::launch_strip_fit(sp.ga, sp.la, bp::line_grid(bp::kLineFit, 0, sp.n_strips), s));
        if (hp.h_bad == nullptr)
            BP_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&hp.h_bad), sizeof(int32_t),
                                       hipHostMallocDefault));
        BP_HIP_CHECK(hipMemcpyAsync(hp.h_bad, sp.la.n_left, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    }
    BP_HIP_CHECK(hipEventRecord(hp.win_ev, s));
    // (with strips the fit follows them, in enqueue_sum)
    if (a.precision == BP_PRECISION_SPLIT && !sp.lines)
        BP_HIP_CHECK(bp::launch_fit(sp.ga, (int)hdr.n_groups, s));
    if (stats) BP_HIP_CHECK(hipEventRecord(c->ev[1], s));
    BP_HIP_CHECK(hipEventSynchronize(hp.win_ev));

    // bands whose union window fits the budget: of whole strips (the
    // line-interpolated sum) or of tile rows
    const size_t line_bytes = sizeof(float) * 2 * (size_t)gi.width;
    size_t budget = (size_t)max_window_bytes;
    if (budget == 0) {
        size_t free_b = 0, total_b = 0;
        BP_HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
        budget = free_b / 2;
    }
    // the window of lines [r0, r1), r0 a multiple of the tile rows
    auto window = [&](int64_t r0, int64_t r1) {
        Band w{r0, r1, INT32_MAX, INT32_MIN};
        for (int64_t q = r0 / band_rows; q < (r1 + band_rows - 1) / band_rows; ++q) {
            if (hp.h_win[2 * q] >= hp.h_win[2 * q + 1]) continue;
            w.k0 = std::min(w.k0, hp.h_win[2 * q]);
            w.k1 = std::max(w.k1, hp.h_win[2 * q + 1]);
        }
        return w;
    };
    auto fits = [&](const Band& w) {
        return w.k0 >= w.k1 || (size_t)(w.k1 - w.k0) * line_bytes <= budget;
    };
    for (int64_t t = 0; t < n_tr; ++t) {
        const Band w = window(t * band_rows, std::min(length, (t + 1) * (int64_t)band_rows));
        if (!fits(w))
            return fail(BP_ERR_LENGTH, "the pulse window of " + std::to_string(band_rows) +
                                           " output lines (" + std::to_string(w.k1 - w.k0) +
                                           " pulses) exceeds max_window_bytes");
    }
    std::vector<Band> bands;
    // bands of `unit` lines at a time from [r0, r1)
    auto cut = [&](int64_t r0, int64_t r1, int unit, Band::Kind kind) {
        Band cur{r0, r0, INT32_MAX, INT32_MIN, kind};
        for (int64_t r = r0; r < r1; r += unit) {
            Band w = window(r, std::min(r1, r + unit));
            Band both = cur;
            both.k0 = std::min(cur.k0, w.k0);
            both.k1 = std::max(cur.k1, w.k1);
            if (cur.r1 > cur.r0 && !fits(both)) {
                bands.push_back(cur);
                cur = Band{r, r, w.k0, w.k1, kind};
            } else {
                cur = both;
            }
            cur.r1 = w.r1;
        }
        if (cur.r1 > cur.r0) bands.push_back(cur);
    };
    // pulses of a part: whole 64-pulse chunks
    const int64_t part = (int64_t)(budget / line_bytes) / 64 * 64;
    std::vector<std::pair<int64_t, int64_t>> part_rows;   // strip rows taken in parts
    if (sp.lines) {
        const int sr = whole.strip_rows;
        int64_t r = 0;
        while (r < length) {
            int64_t e = r;   // strip rows that fit the budget one by one
            while (e < length && fits(window(e, std::min(length, e + sr)))) e = std::min(length, e + sr);
            if (e > r) cut(r, e, sr, Band::kWhole);
            r = e;
            if (r >= length) break;
            // a strip row whose window is larger: its pulses in parts, and
            // what does not qualify in bands of tile rows
            const Band w = window(r, std::min(length, r + sr));
            if (part < bp::kStripMinPulses) {
                // the budget holds no window that a strip qualifies with
                sp.lines = false;
                break;
            }
            part_rows.emplace_back(r, w.r1);
            for (int64_t q = w.k0 / 64 * 64; q < w.k1; q += part) {
                Band b{r, w.r1, (int32_t)std::max<int64_t>(q, w.k0),
                       (int32_t)std::min<int64_t>(q + part, w.k1), Band::kPart};
                b.first = q <= w.k0;
                b.last = q + part >= w.k1;
                bands.push_back(b);
            }
            if (*hp.h_bad > 0) cut(r, w.r1, band_rows, Band::kTiles);
            r = w.r1;
        }
        if (!sp.lines) {
            // the pixel-by-pixel sum in bands of tile rows
            bands.clear();
            part_rows.clear();
            sp.ga.strips = nullptr;
            sp.sa.strips = nullptr;
            BP_HIP_CHECK(bp::launch_fit(sp.ga, (int)hdr.n_groups, s));
        }
    }
    if (!sp.lines) cut(0, length, band_rows, Band::kWhole);
    if (!part_rows.empty() && (rc = ensure(hp.carry, bp::line_carry_bytes() * whole.strips_x))) return rc;
    const bool timed = stats != nullptr || hstats != nullptr;
    int64_t h2d = 0, pulses = 0;
    size_t n_bands = 0;
    double sum_ms = 0., copy_ms = 0.;
    for (bool again = false;; again = true) {
        drain.armed = true;
        size_t max_band = 16;
        for (const Band& b : bands)
            if (b.k0 < b.k1) max_band = std::max(max_band, (size_t)(b.k1 - b.k0) * line_bytes);
        const int nbuf = bands.size() > 1 && 2 * max_band <= budget ? 2 : 1;
        for (int w = 0; w < nbuf; ++w)
            if ((rc = ensure(hp.win[w], max_band))) return rc;
        const int64_t chunk_lines = std::max<int64_t>(
            1, std::min<int64_t>(batch, (int64_t)(kStageBytes / std::max<size_t>(line_bytes, 1))));
        {
            size_t have = hp.stage_bytes, have1 = hp.stage_bytes;
            const size_t want = (size_t)chunk_lines * line_bytes;
            if ((rc = ensure_pinned(hp.stage[0], have, want))) return rc;
            if ((rc = ensure_pinned(hp.stage[1], have1, want))) return rc;
            hp.stage_bytes = std::min(have, have1);
        }

        // descriptors of every band: the whole block's, cut to the band's lines
        const size_t stride = (sizeof(bp::BatchHeader) + sizeof(bp::OutDesc) + 255) & ~size_t(255);
        std::vector<unsigned char> bdesc(stride * bands.size(), 0);
        std::vector<int> band_groups(bands.size());
        std::vector<int64_t> band_strips(bands.size());
        for (size_t b = 0; b < bands.size(); ++b) {
            bp::OutDesc d = whole;
            const int64_t r0 = bands[b].r0;
            d.map = make_map(bands[b].r1 - r0, owidth, o.tile_rows, o.order, o.lane_rows);
            d.t0 = whole.t0 + r0 * whole.dt;
            d.seq_base = 0;
            d.rec_base = whole.rec_base + r0 * owidth;
            d.out = whole.out + r0 * owidth;
            d.height = whole.height ? whole.height + r0 * owidth : nullptr;
            d.strip_seq = 0;
            d.strip_info = whole.strip_info + r0 / whole.strip_rows * whole.strips_x;
            d.strips_y = (int32_t)((d.map.length + d.strip_rows - 1) / d.strip_rows);
            bp::BatchHeader h;
            std::memset(&h, 0, sizeof(h));
            h.n_seq = d.map.n_tiles;
            h.n_groups = (h.n_seq + 3) / 4;
            h.n_geom_groups = (h.n_seq * o.lane_rows + 3) / 4;
            h.n_grids = 1;
            h.lane_rows = o.lane_rows;
            h.n_strips = (int64_t)d.strips_x * d.strips_y;
            std::memcpy(bdesc.data() + b * stride, &h, sizeof(h));
            std::memcpy(bdesc.data() + b * stride + sizeof(h), &d, sizeof(d));
            band_groups[b] = (int)h.n_groups;
            band_strips[b] = h.n_strips;
        }
        if ((rc = upload(hp.band_desc, bdesc.data(), bdesc.size(), s))) return rc;

        while (timed && hp.timing.size() < 4 * bands.size()) {
            hipEvent_t e;
            BP_HIP_CHECK(hipEventCreate(&e));
            hp.timing.push_back(e);
        }
        // copies on the copy stream (they write only the context's window
        // buffers, which no earlier call still reads: every call ends with both
        // streams drained), sums on the caller's stream
        const unsigned char* src = static_cast<const unsigned char*>(a.in_dev);
        int64_t chunk_no = 0;
        bool used[2] = {false, false};
        for (size_t b = 0; b < bands.size(); ++b) {
            const Band& bd = bands[b];
            const int w = (int)(b % nbuf);
            unsigned char* dwin = static_cast<unsigned char*>(hp.win[w].ptr);
            if (used[w]) BP_HIP_CHECK(hipStreamWaitEvent(hp.copy, hp.sum_ev[w], 0));
            if (timed) BP_HIP_CHECK(hipEventRecord(hp.timing[4 * b], hp.copy));
            for (int64_t k = bd.k0; k < bd.k1; k += chunk_lines) {
                const int64_t n = std::min<int64_t>(chunk_lines, bd.k1 - k);
                const int j = (int)(chunk_no++ & 1);
                // staging j is free once its previous copy has finished
                BP_HIP_CHECK(hipEventSynchronize(hp.stage_ev[j]));
                const size_t bytes = (size_t)n * line_bytes;
                host_copy(hp.stage[j], src + (size_t)k * line_bytes, bytes);
                BP_HIP_CHECK(hipMemcpyAsync(dwin + (size_t)(k - bd.k0) * line_bytes, hp.stage[j],
                                            bytes, hipMemcpyHostToDevice, hp.copy));
                BP_HIP_CHECK(hipEventRecord(hp.stage_ev[j], hp.copy));
                h2d += (int64_t)bytes;
            }
            if (bd.k0 < bd.k1) pulses += bd.k1 - bd.k0;
            if (timed) BP_HIP_CHECK(hipEventRecord(hp.timing[4 * b + 1], hp.copy));
            BP_HIP_CHECK(hipEventRecord(hp.copied_ev, hp.copy));
            BP_HIP_CHECK(hipStreamWaitEvent(s, hp.copied_ev, 0));
            // pulse k of the band at dwin + (k - k0) * line_bytes; the sum reads
            // only pulses of its pixels' windows, all inside [k0, k1)
            const int64_t k0 = bd.k0 < bd.k1 ? bd.k0 : 0;
            const float2* rc_base = reinterpret_cast<const float2*>(
                reinterpret_cast<uintptr_t>(dwin) - (uintptr_t)((size_t)k0 * line_bytes));
            const auto* batch_b = reinterpret_cast<const bp::BatchHeader*>(
                static_cast<unsigned char*>(hp.band_desc.ptr) + b * stride);
            if (timed) BP_HIP_CHECK(hipEventRecord(hp.timing[4 * b + 2], s));
            if (bd.kind == Band::kPart) {
                bp::LineArgs la = sp.la;
                la.batch = batch_b;
                la.rc = rc_base;
                la.q_begin = bd.k0 / 64 * 64;
                la.q_end = bd.k1;
                la.q_first = bd.first;
                for (int64_t s0 = 0; s0 < band_strips[b]; s0 += sp.group_strips) {
                    la.s_begin = s0;
                    la.s_end = std::min(band_strips[b], s0 + sp.group_strips);
                    la.carry = reinterpret_cast<double2*>(static_cast<unsigned char*>(hp.carry.ptr) +
                                                          bp::line_carry_bytes() * s0);
                    BP_HIP_CHECK(bp::launch_strips(la, sp.width, bd.last, s));
                }
            } else if ((rc = enqueue_sum(sp, batch_b, rc_base, band_groups[b],
                                         bd.kind == Band::kTiles ? 0 : band_strips[b], s))) {
                return rc;
            }
            if (timed) BP_HIP_CHECK(hipEventRecord(hp.timing[4 * b + 3], s));
            BP_HIP_CHECK(hipEventRecord(hp.sum_ev[w], s));
            used[w] = true;
        }
        if (stats) BP_HIP_CHECK(hipEventRecord(c->ev[2], s));

        c->flags_host.assign(n_flag, 0);
        BP_HIP_CHECK(hipMemcpyAsync(c->flags_host.data(), c->sc.flags.ptr, sizeof(int32_t) * n_flag,
                                    hipMemcpyDeviceToHost, s));
        BP_HIP_CHECK(hipStreamSynchronize(s));
        BP_HIP_CHECK(hipStreamSynchronize(hp.copy));
        drain.armed = false;
        n_bands += bands.size();
        if (timed) {
            for (size_t b = 0; b < bands.size(); ++b) {
                float ms = 0.f;
                BP_HIP_CHECK(hipEventElapsedTime(&ms, hp.timing[4 * b], hp.timing[4 * b + 1]));
                copy_ms += ms;
                BP_HIP_CHECK(hipEventElapsedTime(&ms, hp.timing[4 * b + 2], hp.timing[4 * b + 3]));
                sum_ms += ms;
            }
        }
        // strips taken in parts met samples that are not finite, and no bands of
        // tile rows followed them: those rows once more, pixel by pixel
        if (again || part_rows.empty() || *hp.h_bad > 0 || c->flags_host[3] == 0) break;
        bands.clear();
        for (const auto& r : part_rows) cut(r.first, r.second, band_rows, Band::kTiles);
    }
    if (hstats) {
        hstats->h2d_bytes = h2d;
        hstats->window_pulses = pulses;
        hstats->bands = (int32_t)n_bands;
        hstats->copy_ms = copy_ms;
    }
    const hipEvent_t ev[3] = {stats ? c->ev[0] : nullptr, nullptr, stats ? c->ev[2] : nullptr};
    rc = finish_step(c->flags_host.data(), hdr.n_grids, c->desc_block, blk, ev, any_failed, stats);
    if (stats && c->ev[1]) {
        float ms = 0.f;
        BP_HIP_CHECK(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
        stats->geometry_ms = ms;
        stats->sum_ms = sum_ms;
    }
    return rc;
}

}  // namespace

extern "C" int bp_backproject_host(bp_context* c, const bp_radar_geometry* og,
                                   const bp_radar_geometry* ig, const bp_dem* dem, double fc,
                                   double ds, const bp_kernel* kernel, int dry_tropo_model,
                                   const bp_rdr2geo_params* r2g, const bp_geo2rdr_params* g2r,
                                   const void* in_host, int64_t batch, int64_t max_window_bytes,
                                   void* out_dev, float* height_dev, int precision,
                                   const bp_options* options, void* stream, int* any_failed,
                                   bp_stats* stats, bp_host_stats* host_stats)
try {
    if (any_failed) *any_failed = 0;
    if (!og) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    bp_out_block blk;
    std::memset(&blk, 0, sizeof(blk));
    blk.grid = og->grid;
    blk.out_dev = out_dev;
    blk.height_dev = height_dev;
    CallArgs a{&og->orbit, &og->doppler, ig, dem, fc, ds, kernel, dry_tropo_model, r2g, g2r,
               in_host, precision};
    return run_host(c, a, &blk, batch, max_window_bytes, options, stream, any_failed, stats,
                    host_stats);
} catch (...) {
    return bp_host_exception();
}

extern "C" int64_t bp_workspace_bytes(const bp_radar_geometry* ig, double fc, double ds,
                                      const bp_kernel* kernel, int dry_tropo_model, int precision,
                                      int64_t max_pixels, int max_blocks, int scene, int64_t limit)
try {
    // the rules of check_call that the plans below rely on
    if (ig == nullptr || kernel == nullptr || !(ig->grid.prf > 0) || !(fc > 0) || !(ds > 0) ||
        kernel->n < 2 || kernel->table == nullptr || !(kernel->halfwidth > 0) || max_pixels < 1 ||
        max_blocks < 1)
        return fail(BP_ERR_INVALID_ARGUMENT, "invalid argument");
    int rc;
    if ((rc = check_orbit(ig->orbit, "input geometry")) != BP_SUCCESS) return rc;
    if ((rc = check_lut(ig->doppler, "input geometry")) != BP_SUCCESS) return rc;
    CallArgs a{nullptr, nullptr, ig, nullptr, fc, ds, kernel, dry_tropo_model, nullptr, nullptr,
               nullptr, precision};
    if (precision == BP_PRECISION_PLAIN) {
        const int64_t segs = (ig->grid.length + bp::kPlainSeg - 1) / bp::kPlainSeg;
        return scene_part_records(a, max_pixels, limit) * segs * (int64_t)sizeof(double2);
    }
    Opts two{};
    two.lane_rows = 2;
    const LinePlan p = plan_lines(a, (int)std::ceil(2.0 * kernel->halfwidth), two);
    if (!p.on) return 0;
    const int64_t most = most_strips(max_pixels, max_blocks, p.rows);
    const int64_t n = scene ? scene_strips(max_pixels, max_blocks, p.rows) : most;
    return (int64_t)sizeof(bp::StripInfo) * most +
           (int64_t)p.strip_bytes * line_group(p, n, most, limit);
} catch (...) {
    return bp_host_exception();
}

// ------------------------------------------------------------------ scenes

// One raw set kept resident with everything its tile requests share, scratch
// for up to max_pixels output pixels in up to max_blocks blocks, and one HIP
// graph per launch configuration.  The graph of a step copies the batch
// header and descriptors from pinned host memory, clears the flags with a
// kernel, runs the geometry and sum kernels (persistent grids that read the
// batch counts from the device header) between event records, and copies the
// flags back to pinned host memory; a request only rewrites the pinned
// descriptors and replays the graph.
struct bp_scene {
    bp_context* ctx = nullptr;
    CallArgs args{};
    int width = 0;
    int64_t max_pixels = 0;
    int max_blocks = 0;
    StaticData st;
    Scratch sc;
    // copies of the caller's structs that CallArgs points to
    bp_orbit out_orbit{};
    bp_lut2d out_doppler{};
    bp_radar_geometry in_geometry{};
    bp_dem dem{};
    bp_kernel kernel{};
    bp_rdr2geo_params r2g{};
    bp_geo2rdr_params g2r{};
    unsigned char* h_desc = nullptr;   // pinned: header + max_blocks descriptors
    int32_t* h_flags = nullptr;        // pinned: kFlagWords + max_blocks words
    hipStream_t cap = nullptr;         // capture stream (default priority)
    Branch branch;
    // Strips were left by the last batch: the next one is launched kernel by kernel,
    // with the strips that are left beside the others.  In a graph the second branch
    // takes 17 us (one strip) to 44 us (25) longer to replay, and its long wavefronts
    // share SIMDs where the line sum's are placed first (512 x 512 pixels with a
    // column of such strips: 7.4 ms instead of 4.8); a graph without it puts 0.3 ms of
    // line sum before them.  Results are the same either way.
    bool left = false;
    hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
    std::vector<int> block_of_grid;
    LinePlan lines{};          // line-interpolated sum (lane_rows 2)
    int64_t line_group = 0;    // strips the scene holds workspace for at a time
    int64_t part_records = 0;  // plain: pixels whose segment sums the scene holds
    // A kernel node whose grid follows the batch, with its captured launch
    // parameters: the geometry pass (geometry groups), fit and plain sum (tile
    // groups; the plain sum by segments), strip fit (strips), and the kernels of
    // the line-interpolated
    // sum (the strips of their group, from first on, at most count).
    enum Kind { kGeom, kTiles, kPlain, kStrips };   // kStrips + a LineKernel for the others
    struct GridNode {
        hipGraphNode_t node;
        hipKernelNodeParams params;
        Kind kind;
        int64_t first, count;
    };
    struct Graph {
        int chunk, blocks_per_cu, lane_rows;
        bool staged;
        int64_t groups;   // of line_group strips, 0 without the line-interpolated sum
        hipGraph_t graph;
        hipGraphExec_t exec;
        std::vector<GridNode> nodes;
    };
    std::vector<Graph> graphs;
};

namespace {

void destroy_graphs(bp_scene* sc)
{
    for (auto& g : sc->graphs) {
        if (g.exec) (void)hipGraphExecDestroy(g.exec);
        if (g.graph) (void)hipGraphDestroy(g.graph);
    }
    sc->graphs.clear();
}

void destroy_scene(bp_scene* sc)
{
    destroy_graphs(sc);
    free_static(sc->st);
    free_scratch(sc->sc);
    if (sc->h_desc) (void)hipHostFree(sc->h_desc);
    if (sc->h_flags) (void)hipHostFree(sc->h_flags);
    for (auto& ev : sc->ev)
        if (ev) (void)hipEventDestroy(ev);
    if (sc->cap) (void)hipStreamDestroy(sc->cap);
    sc->branch.destroy();
    delete sc;
}

// Capture the step of one launch configuration, for up to `groups` groups of
// strips.
int capture_graph(bp_scene* sc, const Opts& o, int64_t groups, bp_scene::Graph* out)
{
    bp_context* c = sc->ctx;
    Step sp;
    build_step(sp, sc->st, sc->sc, sc->args, sc->width, o, c->n_cu);
    if (groups > 0) {
        set_lines(sp, sc->lines, sc->sc, sc->args, groups * sc->line_group, sc->line_group);
        if (sp.la.few == 0) sp.la.few = 2;   // replayed with any count up to the groups'
    }
    if (sc->part_records > 0) {
        sp.sa.parts = static_cast<double2*>(sc->sc.parts.ptr);
        sp.sa.parts_stride = sc->part_records;
    }
    // the geometry, fit and plain-sum grids are set per replay to the batch's
    // group counts (bp_scene_focus); one workgroup at capture
    const int cap_grid = 1;
    sp.geom_grid = cap_grid;
    sp.flag_words = kFlagWords + sc->max_blocks;
    // no event records inside the graph: a replay is timed as a whole by
    // events recorded around the launch
    const size_t desc_bytes = sizeof(bp::BatchHeader) + sizeof(bp::OutDesc) * sc->max_blocks;

    hipStream_t s = sc->cap;
    BP_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    int rc = BP_SUCCESS;
    hipError_t e = hipMemcpyAsync(sc->sc.desc.ptr, sc->h_desc, desc_bytes, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) rc = fail(BP_ERR_HIP, std::string("hipMemcpyAsync: ") + hipGetErrorString(e));
    if (rc == BP_SUCCESS) rc = enqueue_step(sp, cap_grid, s);
    if (rc == BP_SUCCESS) {
        e = hipMemcpyAsync(sc->h_flags, sc->sc.flags.ptr, sizeof(int32_t) * (kFlagWords + sc->max_blocks),
                           hipMemcpyDeviceToHost, s);
        if (e != hipSuccess) rc = fail(BP_ERR_HIP, std::string("hipMemcpyAsync: ") + hipGetErrorString(e));
    }
    hipGraph_t g = nullptr;
    e = hipStreamEndCapture(s, &g);
    if (rc != BP_SUCCESS) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return fail(BP_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    // find the kernel nodes whose grid follows the batch
    out->nodes.clear();
    size_t n_nodes = 0;
    e = hipGraphGetNodes(g, nullptr, &n_nodes);
    std::vector<hipGraphNode_t> nodes(n_nodes);
    if (e == hipSuccess && n_nodes) e = hipGraphGetNodes(g, nodes.data(), &n_nodes);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(g);
        return fail(BP_ERR_HIP, std::string("hipGraphGetNodes: ") + hipGetErrorString(e));
    }
    const bool pair = o.lane_rows == 2;
    const void* geo_fn = bp::kernel_fn(bp::dem_generic(host_dem(sc->dem)) ? 4 : 0, sc->width,
                                       o.staged, pair);
    const bool plain = sc->args.precision == BP_PRECISION_PLAIN;
    const void* tile_fn = bp::kernel_fn(plain ? (sp.sa.chunks ? 1 : 6) : 3, sc->width, o.staged, pair);
    const void* total_fn = plain && sc->part_records > 0 ? bp::kernel_fn(5, sc->width, false, false)
                                                         : nullptr;
    for (hipGraphNode_t nd : nodes) {
        hipGraphNodeType type;
        if (hipGraphNodeGetType(nd, &type) != hipSuccess || type != hipGraphNodeTypeKernel) continue;
        hipKernelNodeParams p{};
        if (hipGraphKernelNodeGetParams(nd, &p) != hipSuccess) continue;
        bp_scene::GridNode gn{nd, p, bp_scene::kGeom, 0, 0};
        if (p.func == geo_fn) {
            out->nodes.push_back(gn);
        } else if (p.func == tile_fn) {
            gn.kind = plain ? bp_scene::kPlain : bp_scene::kTiles;
            out->nodes.push_back(gn);
        } else if (total_fn != nullptr && p.func == total_fn) {
            gn.kind = bp_scene::kTiles;
            out->nodes.push_back(gn);
        } else if (sp.lines) {
            for (int which = bp::kLineFit; which <= bp::kLineSum; ++which) {
                if (p.func != bp::line_kernel_fn(which, sc->width)) continue;
                gn.kind = (bp_scene::Kind)(bp_scene::kStrips + which);
                if (which != bp::kLineFit) {
                    const auto* la = static_cast<const bp::LineArgs*>(p.kernelParams[0]);
                    gn.first = la->s_begin;
                    gn.count = la->s_end - la->s_begin;
                }
                out->nodes.push_back(gn);
            }
        }
    }
    const size_t per_group = sp.lines && sp.la.few == 2 ? 5 : 4;
    const size_t want = 2 + (total_fn ? 1 : 0) + (sp.lines ? 1 + per_group * (size_t)groups : 0);
    if (out->nodes.size() != want) {
        (void)hipGraphDestroy(g);
        return fail(BP_ERR_HIP, "captured step is missing its kernel nodes");
    }
    hipGraphExec_t x = nullptr;
    e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(g);
        return fail(BP_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
    }
    out->chunk = o.chunk;
    out->blocks_per_cu = o.blocks_per_cu;
    out->lane_rows = o.lane_rows;
    out->staged = o.staged;
    out->groups = groups;
    out->graph = g;
    out->exec = x;
    return BP_SUCCESS;
}

// The step of a batch launched kernel by kernel.
int launch_scene(bp_scene* sc, const Opts& o, const bp::BatchHeader& hdr, hipStream_t s)
{
    Step sp;
    build_step(sp, sc->st, sc->sc, sc->args, sc->width, o, sc->ctx->n_cu);
    set_lines(sp, sc->lines, sc->sc, sc->args, hdr.n_strips, sc->line_group);
    sp.branch = &sc->branch;
    sp.geom_grid = (int)hdr.n_geom_groups;
    sp.flag_words = kFlagWords + sc->max_blocks;
    BP_HIP_CHECK(hipMemcpyAsync(sc->sc.desc.ptr, sc->h_desc,
                                sizeof(bp::BatchHeader) + sizeof(bp::OutDesc) * hdr.n_grids,
                                hipMemcpyHostToDevice, s));
    const int rc = enqueue_step(sp, (int)hdr.n_groups, s);
    if (rc != BP_SUCCESS) return rc;
    BP_HIP_CHECK(hipMemcpyAsync(sc->h_flags, sc->sc.flags.ptr, sizeof(int32_t) * sp.flag_words,
                                hipMemcpyDeviceToHost, s));
    return BP_SUCCESS;
}

}  // namespace

extern "C" {

int bp_scene_create(bp_context* c, const bp_orbit* out_orbit, const bp_lut2d* out_doppler,
                    const bp_radar_geometry* in_geometry, const bp_dem* dem, double fc,
                    double ds, const bp_kernel* kernel, int dry_tropo_model,
                    const bp_rdr2geo_params* rdr2geo, const bp_geo2rdr_params* geo2rdr,
                    const void* in_dev, int precision, int64_t max_pixels, int max_blocks,
                    bp_scene** scene)
try {
    if (scene == nullptr || c == nullptr) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    *scene = nullptr;
    CallArgs a{out_orbit, out_doppler, in_geometry, dem, fc, ds, kernel, dry_tropo_model,
               rdr2geo, geo2rdr, in_dev, precision};
    int width = 0, rc;
    if ((rc = check_call(a, &width)) != BP_SUCCESS) return rc;
    if (max_pixels < 1 || max_blocks < 1 || max_blocks > (1 << 20))
        return fail(BP_ERR_INVALID_ARGUMENT, "max_pixels and max_blocks must be positive");
    const bp_grid& gi = in_geometry->grid;
    if (gi.length * gi.width > 0 && in_dev == nullptr) return fail(BP_ERR_INVALID_ARGUMENT, "in is null");
    BP_HIP_CHECK(hipSetDevice(c->device));

    auto* sc = new bp_scene();
    sc->ctx = c;
    sc->width = width;
    sc->max_pixels = max_pixels;
    sc->max_blocks = max_blocks;
    sc->out_orbit = *out_orbit;
    sc->out_doppler = *out_doppler;
    sc->in_geometry = *in_geometry;
    sc->dem = *dem;
    sc->kernel = *kernel;
    sc->r2g = *rdr2geo;
    sc->g2r = *geo2rdr;
    sc->args = CallArgs{&sc->out_orbit, &sc->out_doppler, &sc->in_geometry, &sc->dem, fc, ds,
                        &sc->kernel, dry_tropo_model, &sc->r2g, &sc->g2r, in_dev, precision};
    auto bail = [&](int code) {
        destroy_scene(sc);
        return code;
    };
    if (hipStreamCreateWithFlags(&sc->cap, hipStreamNonBlocking) != hipSuccess || !sc->branch.create())
        return bail(fail(BP_ERR_HIP, "hipStreamCreate failed"));
    for (auto& ev : sc->ev)
        if (hipEventCreate(&ev) != hipSuccess) return bail(fail(BP_ERR_HIP, "hipEventCreate failed"));
    const size_t desc_bytes = sizeof(bp::BatchHeader) + sizeof(bp::OutDesc) * max_blocks;
    const size_t flag_bytes = sizeof(int32_t) * (kFlagWords + max_blocks);
    if (hipHostMalloc(reinterpret_cast<void**>(&sc->h_desc), desc_bytes, hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc(reinterpret_cast<void**>(&sc->h_flags), flag_bytes, hipHostMallocDefault) != hipSuccess)
        return bail(fail(BP_ERR_OUT_OF_MEMORY, "hipHostMalloc failed"));
    std::memset(sc->h_desc, 0, desc_bytes);
    std::memset(sc->h_flags, 0, flag_bytes);
    if ((rc = ensure(sc->sc.desc, desc_bytes))) return bail(rc);
    if ((rc = ensure(sc->sc.flags, flag_bytes))) return bail(rc);
    if ((rc = ensure(sc->sc.geom, sizeof(bp::PixGeom) * max_pixels))) return bail(rc);
    if (precision == BP_PRECISION_SPLIT && (rc = ensure(sc->sc.split, sizeof(bp::PixSplit) * max_pixels)))
        return bail(rc);
    hipStream_t s = sc->cap;
    if ((rc = upload_static(sc->st, sc->args, width, s))) return bail(rc);
    if (hipMemsetAsync(sc->sc.flags.ptr, 0, flag_bytes, s) != hipSuccess)
        return bail(fail(BP_ERR_HIP, "hipMemsetAsync failed"));
    if ((rc = pulse_states(sc->st, sc->args, static_cast<int32_t*>(sc->sc.flags.ptr), s))) return bail(rc);
    if (const int64_t n = scene_part_records(sc->args, max_pixels, c->workspace_limit)) {
        const int64_t segs = (in_geometry->grid.length + bp::kPlainSeg - 1) / bp::kPlainSeg;
        if (ensure(sc->sc.parts, sizeof(double2) * segs * n) == BP_SUCCESS) sc->part_records = n;
    }
    {
        Opts two{};
        two.lane_rows = 2;
        sc->lines = plan_lines(sc->args, width, two);
        if (sc->lines.on)
            sc->line_group = alloc_lines(sc->lines, scene_strips(max_pixels, max_blocks, sc->lines.rows),
                                         most_strips(max_pixels, max_blocks, sc->lines.rows),
                                         c->workspace_limit, sc->sc);
        sc->lines.on = sc->line_group > 0;
    }
    int32_t oor = 0;
    if (hipMemcpyAsync(&oor, static_cast<int32_t*>(sc->sc.flags.ptr) + 1, sizeof(oor),
                       hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return bail(fail(BP_ERR_HIP, "scene upload failed"));
    if (oor) return bail(fail(BP_ERR_OUT_OF_RANGE, orbit_err_string(BP_ORBIT_INTERP_DOMAIN_ERROR)));
    *scene = sc;
    return BP_SUCCESS;
} catch (...) {
    return bp_host_exception();
}

int bp_scene_destroy(bp_scene* sc)
try {
    if (sc == nullptr) return BP_SUCCESS;
    (void)hipSetDevice(sc->ctx->device);
    (void)hipStreamSynchronize(sc->cap);
    destroy_scene(sc);
    return BP_SUCCESS;
} catch (...) {
    return bp_host_exception();
}

}  // extern "C"

namespace bp {
int scene_device(const bp_scene* s) { return s->ctx->device; }
int64_t scene_max_pixels(const bp_scene* s) { return s->max_pixels; }
int scene_max_blocks(const bp_scene* s) { return s->max_blocks; }
}  // namespace bp

extern "C" {

int bp_scene_focus(bp_scene* sc, bp_out_block* blocks, int n_blocks, const bp_options* options,
                   void* stream, int* any_failed, bp_stats* stats)
try {
    if (any_failed) *any_failed = 0;
    if (stats) std::memset(stats, 0, sizeof(*stats));
    if (sc == nullptr) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    int rc;
    int64_t npix = 0;
    if ((rc = check_blocks(blocks, n_blocks, &npix)) != BP_SUCCESS) return rc;
    if (npix > sc->max_pixels)
        return fail(BP_ERR_INVALID_ARGUMENT, "request of " + std::to_string(npix) +
                                                 " pixels exceeds the scene's max_pixels");
    Opts o;
    if ((rc = check_options(options, &o)) != BP_SUCCESS) return rc;
    if ((rc = check_lane_rows(o, sc->args.precision, sc->width)) != BP_SUCCESS) return rc;
    if (npix == 0) return BP_SUCCESS;
    BP_HIP_CHECK(hipSetDevice(sc->ctx->device));
    hipStream_t s = static_cast<hipStream_t>(stream);
    // strips in groups of the scene's workspace; graphs for powers of two of them
    int64_t groups = 0;
    if (sc->lines.on && o.lane_rows == 2 && !o.staged) {
        use_plan(o, sc->lines);
        int64_t n_strips = 0;
        for (int b = 0; b < n_blocks; ++b) {
            bp::OutDesc d;
            d.map.length = blocks[b].grid.length;
            d.map.width = blocks[b].grid.width;
            d.dt = 1.0 / blocks[b].grid.prf;
            d.dr = blocks[b].grid.range_pixel_spacing;
            if (d.map.length * d.map.width > 0) n_strips += map_strips(d, o);
        }
        if (n_strips > 0)
            for (groups = 1; groups * sc->line_group < n_strips;) groups *= 2;
    }

    const bool replayed = groups == 0 || !sc->left;
    bp_scene::Graph* g = nullptr;
    for (auto& x : sc->graphs)
        if (x.chunk == o.chunk && x.blocks_per_cu == o.blocks_per_cu && x.staged == o.staged &&
            x.lane_rows == o.lane_rows && x.groups == groups)
            g = &x;
    if (g == nullptr && replayed) {
        bp_scene::Graph ng{};
        if ((rc = capture_graph(sc, o, groups, &ng)) != BP_SUCCESS) return rc;
        sc->graphs.push_back(ng);
        g = &sc->graphs.back();
    }
    // the previous replay has finished (every focus call waits for its step),
    // so the pinned descriptors are free to rewrite
    bp::BatchHeader hdr;
    if ((rc = plan_batch(blocks, n_blocks, o, static_cast<int32_t*>(sc->sc.flags.ptr) + kFlagWords,
                         sc->h_desc, sc->max_blocks, &hdr, sc->block_of_grid)) != BP_SUCCESS)
        return rc;
    if (sc->part_records > 0 && npix <= sc->part_records) {
        hdr.plain_segs = plain_segments(sc->args, hdr.n_seq, npix, -1);
        std::memcpy(sc->h_desc, &hdr, sizeof(hdr));
    }
    for (size_t i = 0; replayed && i < g->nodes.size(); ++i) {
        const bp_scene::GridNode& gn = g->nodes[i];
        const int64_t n = std::min(std::max<int64_t>(hdr.n_strips - gn.first, 0), gn.count);
        int64_t grid;
        switch (gn.kind) {
        case bp_scene::kGeom: grid = hdr.n_geom_groups; break;
        case bp_scene::kTiles: case bp_scene::kPlain: grid = hdr.n_groups; break;
        case bp_scene::kStrips: grid = hdr.n_strips; break;
        default: grid = bp::line_grid(gn.kind - bp_scene::kStrips, sc->lines.slots, n); break;
        }
        hipKernelNodeParams p = gn.params;
        p.gridDim = dim3((unsigned)std::max<int64_t>(grid, 1),
                         gn.kind == bp_scene::kPlain ? (unsigned)std::max(hdr.plain_segs, 1) : 1u);
        BP_HIP_CHECK(hipGraphExecKernelNodeSetParams(g->exec, gn.node, &p));
    }
    if (stats) BP_HIP_CHECK(hipEventRecord(sc->ev[0], s));
    if (replayed) {
        BP_HIP_CHECK(hipGraphLaunch(g->exec, s));
    } else if ((rc = launch_scene(sc, o, hdr, s)) != BP_SUCCESS) {
        (void)hipStreamSynchronize(sc->branch.s);   // nothing of the call runs on
        (void)hipStreamSynchronize(s);
        return rc;
    }
    if (stats) BP_HIP_CHECK(hipEventRecord(sc->ev[2], s));
    BP_HIP_CHECK(hipStreamSynchronize(s));
    if (groups > 0)
        sc->left = sc->h_flags[2] + hdr.no_strips > 0 && sc->h_flags[2] < hdr.n_strips;
    const hipEvent_t ev[3] = {sc->ev[0], nullptr, sc->ev[2]};
    return finish_step(sc->h_flags, hdr.n_grids, sc->block_of_grid, blocks, ev, any_failed, stats);
} catch (...) {
    return bp_host_exception();
}

int bp_backproject(bp_context* c, const bp_radar_geometry* og, const bp_radar_geometry* ig,
                   const bp_dem* dem, double fc, double ds, const bp_kernel* kernel,
                   int dry_tropo_model, const bp_rdr2geo_params* r2g,
                   const bp_geo2rdr_params* g2r, const void* in_dev, void* out_dev,
                   float* height_dev, int precision, const bp_options* options, void* stream,
                   int* any_failed, bp_stats* stats)
try {
    if (any_failed) *any_failed = 0;
    if (!og) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    bp_out_block blk;
    std::memset(&blk, 0, sizeof(blk));
    blk.grid = og->grid;
    blk.out_dev = out_dev;
    blk.height_dev = height_dev;
    CallArgs a{&og->orbit, &og->doppler, ig, dem, fc, ds, kernel, dry_tropo_model, r2g, g2r,
               in_dev, precision};
    return run_blocks(c, a, &blk, 1, options, stream, any_failed, stats);
} catch (...) {
    return bp_host_exception();
}

int bp_backproject_noalloc(bp_context* c, const bp_radar_geometry* og,
                           const bp_radar_geometry* ig, const bp_dem* dem, double fc, double ds,
                           const bp_kernel* kernel, int dry_tropo_model,
                           const bp_rdr2geo_params* r2g, const bp_geo2rdr_params* g2r,
                           const void* in_dev, void* out_dev, float* height_dev, int precision,
                           const bp_options* options, void* stream, int* any_failed,
                           bp_stats* stats)
try {
    if (any_failed) *any_failed = 0;
    if (!og || !c) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    if (c->scratch == nullptr)
        return fail(BP_ERR_HIP, "bp_backproject_noalloc: no scratch address for this context's "
                                "device (" + c->scratch_err + ")");
    bp_out_block blk;
    std::memset(&blk, 0, sizeof(blk));
    blk.grid = og->grid;
    blk.out_dev = out_dev;
    blk.height_dev = height_dev;
    CallArgs a{&og->orbit, &og->doppler, ig, dem, fc, ds, kernel, dry_tropo_model, r2g, g2r,
               in_dev, precision};
    Carve cv{c->scratch, kNoAllocScratchBytes};
    return run_blocks(c, a, &blk, 1, options, stream, any_failed, stats, &cv);
} catch (...) {
    return bp_host_exception();
}

int bp_backproject_blocks(bp_context* c, const bp_orbit* out_orbit, const bp_lut2d* out_doppler,
                          bp_out_block* blocks, int n_blocks, const bp_radar_geometry* ig,
                          const bp_dem* dem, double fc, double ds, const bp_kernel* kernel,
                          int dry_tropo_model, const bp_rdr2geo_params* r2g,
                          const bp_geo2rdr_params* g2r, const void* in_dev, int precision,
                          const bp_options* options, void* stream, int* any_failed,
                          bp_stats* stats)
try {
    CallArgs a{out_orbit, out_doppler, ig, dem, fc, ds, kernel, dry_tropo_model, r2g, g2r,
               in_dev, precision};
    return run_blocks(c, a, blocks, n_blocks, options, stream, any_failed, stats);
} catch (...) {
    return bp_host_exception();
}

// ------------------------------------------------------------ host helpers

int bp_orbit_interpolate(const bp_orbit* orbit, double t, int border, double* pos, double* vel)
try {
    if (!orbit || !pos || !vel) return BP_NULL_DEREFERENCE;
    bp::V3 p{bp::qnan(), bp::qnan(), bp::qnan()}, v = p;
    int st = bp::orbit_interpolate(host_orbit(*orbit), t, border, &p, &v);
    pos[0] = p.x; pos[1] = p.y; pos[2] = p.z;
    vel[0] = v.x; vel[1] = v.y; vel[2] = v.z;
    return st;
} catch (...) {
    return bp_host_exception();
}

void bp_lonlat_to_xyz(double a, double e2, const double* llh, double* xyz)
{
    bp::V3 r = bp::lonlat_to_xyz(a, e2, bp::V3{llh[0], llh[1], llh[2]});
    xyz[0] = r.x; xyz[1] = r.y; xyz[2] = r.z;
}

void bp_xyz_to_lonlat(double a, double e2, const double* xyz, double* llh)
{
    bp::V3 r = bp::xyz_to_lonlat(a, e2, bp::V3{xyz[0], xyz[1], xyz[2]});
    llh[0] = r.x; llh[1] = r.y; llh[2] = r.z;
}

double bp_dem_interpolate_lonlat(const bp_dem* dem, double lon, double lat)
{
    return bp::dem_interpolate_lonlat(host_dem(*dem), lon, lat);
}

double bp_dem_interpolate_xy(const bp_dem* dem, double x, double y)
{
    return bp::dem_interpolate_xy(host_dem(*dem), x, y);
}

int bp_proj_forward(int epsg, const double* llh, double* xyz)
try {
    bp::Proj p;
    if (llh == nullptr || xyz == nullptr) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    if (!bp::proj_init(epsg, &p))
        return fail(BP_ERR_INVALID_ARGUMENT, "Unknown EPSG code (in factory): " + std::to_string(epsg));
    bp::V3 out;
    if (!bp::proj_forward(p, bp::ld3(llh), &out)) return 1;
    xyz[0] = out.x; xyz[1] = out.y; xyz[2] = out.z;
    return 0;
} catch (...) {
    return bp_host_exception();
}

int bp_proj_inverse(int epsg, const double* xyz, double* llh)
try {
    bp::Proj p;
    if (llh == nullptr || xyz == nullptr) return fail(BP_ERR_INVALID_ARGUMENT, "null argument");
    if (!bp::proj_init(epsg, &p))
        return fail(BP_ERR_INVALID_ARGUMENT, "Unknown EPSG code (in factory): " + std::to_string(epsg));
    bp::V3 out;
    if (!bp::proj_inverse(p, bp::ld3(xyz), &out)) return 1;
    llh[0] = out.x; llh[1] = out.y; llh[2] = out.z;
    return 0;
} catch (...) {
    return bp_host_exception();
}

double bp_lut2d_eval(const bp_lut2d* lut, double y, double x)
{
    return bp::lut2d_eval(host_lut(*lut), y, x);
}

void bp_sincos_turns(double t, double* s, double* c)
{
    double ss = 0., cc = 0.;
    bp::sincos_turns(t, &ss, &cc);
    if (s) *s = ss;
    if (c) *c = cc;
}

double bp_knab_eval(double width, double bandwidth, double x)
{
    return bp::knab_eval(x, std::fabs(width / 2.0), bandwidth);
}

int bp_tabulate_knab(double width, double bandwidth, int n, float* table)
try {
    if (n < 2 || table == nullptr) return fail(BP_ERR_INVALID_ARGUMENT, "Require table size >= 2.");
    if (!(bandwidth > 0.0 && bandwidth < 1.0))
        return fail(BP_ERR_RUNTIME, "Require 0 < bandwidth < 1");
    const double hw = std::fabs(width / 2.0);
    const double dx = hw / (n - 1.0);
    for (int i = 0; i < n; ++i) table[i] = (float)bp::knab_eval(i * dx, hw, bandwidth);
    return BP_SUCCESS;
} catch (...) {
    return bp_host_exception();
}

int bp_rdr2geo_bracket(double aztime, double slant_range, double doppler, const bp_orbit* orbit,
                       const bp_dem* dem, double wavelength, int side,
                       const bp_rdr2geo_params* params, double* xyz)
try {
    bp::V3 x{bp::qnan(), bp::qnan(), bp::qnan()};
    bp::R2GParams p{params->tol_height, params->look_min, params->look_max};
    int st = bp::rdr2geo_bracket(aztime, slant_range, doppler, host_orbit(*orbit), host_dem(*dem),
                                 wavelength, side, p, &x);
    xyz[0] = x.x; xyz[1] = x.y; xyz[2] = x.z;
    return st;
} catch (...) {
    return bp_host_exception();
}

int bp_geo2rdr_bracket(const double* xyz, const bp_orbit* orbit, const bp_lut2d* doppler,
                       double wavelength, int side, const bp_geo2rdr_params* params,
                       double* aztime, double* range)
try {
    bp::G2RParams p;
    p.tol_aztime = params->tol_aztime;
    p.have_time_start = params->have_time_start;
    p.have_time_end = params->have_time_end;
    p.time_start = params->time_start;
    p.time_end = params->time_end;
    return bp::geo2rdr_bracket(bp::V3{xyz[0], xyz[1], xyz[2]}, host_orbit(*orbit),
                               host_lut(*doppler), wavelength, side, p, aztime, range);
} catch (...) {
    return bp_host_exception();
}

}  // extern "C"
