// Internal device-side data layout shared by the geometry pass, the
// coherent-sum kernels and the host launcher.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/isce3_amd_backproject.h"
#include "bp_math.h"

namespace bp {

// Per-pixel status values written by the geometry pass.
enum PixStatus : int32_t {
    kPixOk = 0,
    kPixRdr2GeoFailed = 1,   // output NaN, height NaN (Backproject.cpp:146-152)
    kPixGeo2RdrFailed = 2,   // output NaN, height valid (Backproject.cpp:167-170)
    kPixOutOfRange = 3,      // orbit domain error; the call raises OutOfRange
    kPixOutside = 4,         // padding lane outside the output grid
};

// Result of the per-pixel geometry pass consumed by the plain FP64 sum:
// target ECEF position, dry-troposphere delay and pulse window [kstart, kstop).
struct alignas(16) PixGeom {
    double x[3];
    double tau_atm;
    int32_t kstart, kstop;
    int32_t status;
    int32_t pad_;
};

// Per-pixel record of the split-precision sum.  The pulse phase in cycles,
// P(k), is a degree-4 polynomial in the pulse index fitted in FP64; the sum
// kernel steps it pulse by pulse from the wavefront's first pulse kw0 by FP64
// forward differences, P += d1; d1 += d2, and every `chunk` pulses adds the
// terms of d3 and d4 those steps left out (binomial coefficients of chunk).
// The polyphase coordinate z = fma((float)P, zscale, zoff) >= 0, with the
// global zscale = -Q/(fc dtau), gives the first tap c0 = cbase - (floor(z) >>
// log2 Q) and the weight row floor(z) & (Q - 1) + fract(z).
struct alignas(16) PixSplit {
    double p0;               // P(kw0)
    double d1, d2, d3, d4;   // forward differences of P at kw0
    float zoff;
    int32_t cbase;
    int32_t kstart, kstop;
    int32_t status;
    int32_t edge;            // nonzero: some tap of the window may leave [0, nr)
};

static_assert(sizeof(PixGeom) == 48, "PixGeom layout");
static_assert(sizeof(PixSplit) == 64, "PixSplit layout");

constexpr int kFitDegree = 4;        // delay polynomial degree of the split path
constexpr int kPolyphaseLog2 = 9;
constexpr int kPolyphaseRows = 1 << kPolyphaseLog2;  // fractional-offset rows of the split weight table
constexpr int kMaxTableLds = 8192;   // plain path keeps tables up to this size in LDS

// One polyphase weight row of the split sum: the W tap weights (padded to a
// multiple of 4), the same number of deltas to the next row, and for W <= 8
// four floats of padding.  Rows are read as float4 at data-dependent row
// offsets; an 80-byte stride spreads their starts over all LDS banks.
__host__ __device__ constexpr int poly_row_floats(int w)
{
    return 2 * ((w + 3) / 4 * 4) + (((w + 3) / 4 * 4) % 8 == 0 ? 4 : 0);
}

// Pixel tiling of one output grid: each 64-lane wavefront of the sum owns a
// tile of (tile_rows * lane_rows) x (64 / tile_rows) output pixels; lane l
// holds the lane_rows vertically adjacent pixels of lane row l / tile_cols and
// column l % tile_cols.
struct TileMap {
    int32_t tile_rows, tile_cols;
    int32_t tiles_x, tiles_y;
    int64_t length, width;      // output grid
    int64_t n_tiles;            // wavefront tiles of this grid
    int32_t order;              // sum-kernel tile sequence: 0 row-major, 1 column-major
    int32_t lane_rows;          // output lines per lane: 1, or 2 (split sum, W = 8)
};

// Interpolation kernel widths (taps, ceil of the kernel width) with built
// coherent-sum kernels.
constexpr int kMinKernelWidth = 2;
constexpr int kMaxKernelWidth = 16;

// Two-line weight table of kernel width W (split sum with lane_rows = 2):
// Q = 2^pair_q_log2(W) rows at fractional offsets tmin + q/Q, each holding
// the W + 1 entries of a (W + 1)-bin window followed by the differences to the
// next row of entries [pair_lerp_lo(W), pair_lerp_lo(W) + pair_lerp_n(W)),
// padded to whole float4s, in two copies -- the W weights followed by a zero
// (copy 0) or preceded by one (copy 1), copy 1 of a row right after its copy
// 0.  A pixel reads row floor(Q t) and
// interpolates the entries that have differences linearly between the rows;
// entries without differences hold the weight at the middle of the row's
// interval.  Q is the largest power of two up to 512 that keeps the table
// within 64 KB of LDS, so that two 512-thread workgroups fit one CU.
// Entries interpolated between rows: the BP_PAIR_LERP_N central ones (all
// W + 1 when W + 1 <= BP_PAIR_LERP_N).  The outer taps of the kernel change
// slowly with the offset, so their half-row offset error costs little: on the
// config-1 block (width 8, 512 rows) 5 interpolated entries give 5.4e-5
// relative and 4.5e-5 rad RMS phase error against the FP64 oracle, 7 give
// 2.0e-5, all 9 (256 rows) 2.7e-6, at 91.1 / 93.4 / 96.3 ms for the sum.
#ifndef BP_PAIR_LERP_N
#define BP_PAIR_LERP_N 5
#endif
__host__ __device__ constexpr int pair_lerp_n(int w) { return BP_PAIR_LERP_N < w + 1 ? BP_PAIR_LERP_N : w + 1; }
__host__ __device__ constexpr int pair_lerp_lo(int w) { return (w + 1 - pair_lerp_n(w)) / 2; }
__host__ __device__ constexpr int pair_row_floats(int w)
{
    return (w + 1 + pair_lerp_n(w) + 3) / 4 * 4;
}
__host__ __device__ constexpr int pair_q_log2(int w)
{
    int q = 9;
    while (q > 4 && 2 * (1 << q) * pair_row_floats(w) * 4 > 65536) --q;
    return q;
}
__host__ __device__ constexpr int pair_table_floats(int w)
{
    return 2 * (1 << pair_q_log2(w)) * pair_row_floats(w);
}

// Doubles per pulse of the plain sum's per-pulse record: platform position
// (3), velocity (3), 2 / (|v|^2 - c^2) (the bistatic delay's factor) and the
// position's difference from the cubic of its chunk.
constexpr int kPulseRecDoubles = 8;

// The plain sum takes pulses in chunks of kPlainChunk (absolute multiples) and
// interpolates a pixel's delay between four of them (near the Chebyshev points
// of the chunk).
constexpr int kPlainChunk = 64;
constexpr int kPlainNode[4] = {2, 19, 44, 61};
// A pulse's position less the cubic through the nodes' positions, kPosQ
// steps per metre in three 21-bit fields, or kPosNone in a chunk where some do
// not fit (2.4e-7 m) or that the data's end cuts off: delays are evaluated there.
constexpr double kPosQ = 4398046511104.0;  // 2^42
constexpr unsigned long long kPosNone = 1ull << 63;
// How far the cubic may be off the delay (cycles): a few roundings of the phase
// itself, 8 / 2^53 of fc tau (4e-8 rad at 850 km and L band), and no less than
// 6e-9 rad.
constexpr double kCubicUlps = 8. / 9007199254740992.;
constexpr double kCubicTol = 1e-9;
// Largest third difference of the phase (radians), whose phasor 1 + i eps is
// good to 2e-8 at the chunk's end (eps^2 / 2 times 64^3 / 6); 7e-9 at 850 km, 7.5
// km/s, 1520 Hz and L band, and beyond 2e-7 only where the phase rounds to more.
constexpr double kCubicEps = 9e-7;

// One output grid of a (batched) call.  Wavefront tiles of all grids are
// numbered consecutively: grid g owns [seq_base, seq_base + map.n_tiles).
struct OutDesc {
    TileMap map;
    double t0, dt, r0, dr;      // sensing start, 1/PRF, starting range, spacing
    int32_t side;               // look side
    int32_t pad_;
    int64_t seq_base;           // first global wavefront tile of this grid
    int64_t rec_base;           // first per-pixel record of this grid
    float2* out;                // complex64 [length x width]
    float* height;              // optional float32 [length x width]
    int32_t* failed;            // per-grid flag: some pixel failed to converge
    // strips of the line-interpolated split sum (none: strip_info < 0): strip_rows
    // x 64 pixels, row
    // (y, x) of strips with its StripInfo at strip_info + y strips_x + x; the
    // batch's strips are numbered consecutively, column by column in a grid
    int32_t strip_rows, strips_x, strips_y, pad2_;
    int64_t strip_seq;          // first strip of this grid in the batch
    int64_t strip_info;         // StripInfo of this grid's strip (0, 0)
};

// Counts of one (batched) call, stored on the device directly in front of its
// output descriptors, so that the kernels read them at run time and a
// captured step replays with new counts.
struct BatchHeader {
    int64_t n_seq;              // wavefront tiles of all grids
    int64_t n_groups;           // groups of four tiles (plain-sum and fit workgroups)
    int64_t n_geom_groups;      // groups of four geometry wavefronts (lane_rows per tile)
    int32_t n_grids;
    int32_t lane_rows;
    int64_t n_strips;           // strips of all grids
    int32_t plain_segs;         // plain sum: segments summed by their own
                                // wavefronts, 0: each wavefront takes them all
    int32_t no_strips;          // some grid has none
};
static_assert(sizeof(BatchHeader) == 48, "BatchHeader layout");

// Pulses per segment of the plain sum: 512 pulses still give four wavefronts a
// tile, and the table's copy to LDS is 1% of a segment's work.
constexpr int kPlainSeg = 128;
static_assert(kPlainSeg % kPlainChunk == 0, "segments of whole chunks");

// Line-interpolated split sum (bp_lines.hip).
constexpr int kStripLines = 64;      // lines per strip, at most
// degree of the tap weight polynomials in the cell: 7 for even kernels, 8 for
// odd ones, whose taps end away from a zero of the sinc (worst weight error
// 9e-6 and 2e-6 of the peak for the widths 8 and 9; 5.5e-5 for 9 at degree 7)
constexpr int kLineDegree = 8;
__host__ __device__ constexpr int line_degree(int w) { return w % 2 == 0 ? 7 : 8; }
constexpr int kLineTaps = 5;         // distinct taps of an even kernel, widths up to 9
constexpr int kEndDegree = 4;        // weights of the taps at a cell's end
// Limits a strip has to keep, at the ends of its lines' common pulses:
constexpr float kLineMaxShift = 0.33f;   // bins between a line and the reference line
constexpr double kLineMaxSlope = 1.0;    // cycles per pulse
// Pulses of each of its pixels, at least: with fewer the pixel-by-pixel sum is
// short anyway, and host pulses in parts of whole chunks need as many.
constexpr int kStripMinPulses = 64;
// phase (rad) a line gathers over half a chunk against the reference line,
// plus pi times its bins off: what the 6 or 8 nodes interpolate (the residue
// is x^N / (N! 2^(N-1)) at most: 1.5e-4 for x = 2.4 and N = 8, 1.2e-4 for x =
// 1.15 and N = 6, each ten times smaller as an average over the chunk, the
// lines and the band)
constexpr float kLineBound8 = 2.65f, kLineBound6 = 1.35f;
constexpr float kLineSlopeTol = 1e-4f;   // rad: a line's phase off the nodes' at a chunk's end
// A line's position off the nodes' (bins), where pixels differ by their
// tropospheric delay: up to kLinePosTol it is left out (1.6e-4 of a sample in
// the middle of the band, a tenth of that over a strip's lines), up to
// kLinePosMax the sums of the samples' derivatives at four nodes bring it in.
// It has to be the same at both ends of the aperture to kLinePosTol.
constexpr float kLinePosTol = 1e-4f, kLinePosMax = 3e-3f;
constexpr int kSlopeNodes = 4;
constexpr float kLineColumnTol = 0.06f;  // bins: fractional positions of the columns

// What becomes of a strip: left to the pixel-by-pixel sum by its fit, taken by
// the line-interpolated sum, or taken and, with sums that are not finite, done
// again by the pixel-by-pixel sum.
enum StripState : int32_t { kStripLeft = 0, kStripTaken = 1, kStripRedo = 2 };
// The strips that a launch of the pixel-by-pixel sum (and of its fit) takes.
enum StripPass : int32_t { kPassLeft = 1, kPassRedo = 2 };

// Pulses of a strip: k0 .. k1 by some pixel, f0 .. f1 by all; chunks of
// 2^chunk_log2 pulses (absolute multiples) from slot0.
struct StripInfo {
    int32_t k0, k1, f0, f1;
    int32_t ok;              // StripState
    int32_t slot0, nslots;
    int32_t slopes;          // the lines' positions need the samples' derivatives
};

// Per-pixel record of the line-interpolated sum (in the place of PixSplit):
// the phase in cycles p0 + a1 j + .. + a4 j^4, j = k - k0, and the range bin
// ub + uf + (phase - p0) / (fc dtau).
struct alignas(16) PixLine {
    double p0, a1, a2, a3, a4;
    float uf;
    int32_t ub;
    int32_t kstart, kstop;
    float du;                // bins off the position the nodes interpolate
    int32_t pad_;
};
static_assert(sizeof(PixLine) == 64, "PixLine layout");

struct LineArgs {
    const BatchHeader* batch;
    PixLine* rec;
    StripInfo* info;
    int32_t* n_left;                     // strips left to the pixel-by-pixel sum, and done again
    const float2* rc;                    // range-compressed pulses [na x nr]
    int64_t nr;
    double inv_k;                        // 1 / (fc dtau): cycles -> range bins
    double in_r0, inv_dr;                // input grid: starting range, 1 / spacing
    int64_t s_begin, s_end;              // strips of this launch
    // Pulses in device memory a part at a time: the chunks that begin in
    // [q_begin, q_end), multiples of 64, with the running FP64 sums of
    // strip_lines kept in `carry` between the parts (null: all at once).
    int32_t q_begin, q_end, q_first, pad_;
    double2* carry;                      // [strip][segment][64 lines][64]
    int32_t slots;                       // chunks per strip in the workspace
    int32_t chunk_log2;
    int32_t n_sums;                      // sums per chunk: 8 nodes, and with a
                                         // tropospheric delay kSlopeNodes slopes
    float2* sums;                        // [strip][slot][n_sums][64]
    float2* parts;                       // [strip][segment][64 lines][64]
    unsigned long long* cross;           // [strip][slot][8 nodes]
    float farrow[kLineDegree + 1][kLineTaps];
    float w_in[kEndDegree + 1], w_out[kEndDegree + 1];
    int32_t few;                // lines kernel: 0 for many strips, 1 for up to
                                // kFewStrips, 2 chosen by the batch's count
};

__host__ __device__ inline const OutDesc* batch_grids(const BatchHeader* b)
{
    return reinterpret_cast<const OutDesc*>(b + 1);
}

struct GeomArgs {
    const BatchHeader* batch;   // device: header then OutDesc[n_grids]
    int32_t want_split;
    int32_t in_side;
    int32_t kwidth;             // interpolation kernel width W (taps)
    int32_t nr;                 // range samples per pulse
    double in_t0, in_dt;
    int32_t na, tropo;
    double swst, dtau;
    double wvl, fc, ds;
    Orbit out_orbit, in_orbit;  // device pointers
    Lut2d out_dop, in_dop;      // device pointers
    Dem dem;                    // device pointers
    R2GParams r2g;
    G2RParams g2r;
    PixGeom* geom;              // plain records (always written)
    PixSplit* split;            // split records (when want_split)
    int32_t* flags;             // [0] any failed, [1] out of range, [2] strips
                                // left to the pixel-by-pixel split sum, [3] done again
    unsigned long long* updates;
    const StripInfo* strips;    // line-interpolated sum's strips, or null
    int32_t strip_pass;         // StripPass bits of this launch
};

struct SumArgs {
    const BatchHeader* batch;   // device: header then OutDesc[n_grids]
    int32_t chunk;
    int32_t ntab;
    int64_t nr;                 // range samples per pulse
    double swst, dtau, fc;
    double inv_k;               // 1 / (fc * dtau): cycles -> range bins
    double halfwidth;           // kernel half width
    float rdx;                  // float(1/dx) of the tabulated kernel
    float zscale;               // -Q * inv_k (split polyphase coordinate per cycle)
    const float2* rc;           // range-compressed pulses [na x nr]
    const double* pulse_pv;     // per-pulse records [na x kPulseRecDoubles]
    const PixGeom* geom;
    const PixSplit* split;
    const float* table;         // tabulated kernel (plain)
    const float* poly;          // polyphase weights (split): (rows+1) x poly_row_floats(W)
    const float* poly2;         // two-line weights (split, lane_rows 2): pair_table_floats(W)
    float zscale2;              // -2^pair_q_log2(W) * inv_k
    int32_t exact_width;        // plain: 2 * halfwidth == W (no tap lies past the half width)
    double inv_dtau;            // 1 / dtau
    const double2* tab2;        // plain: (t_i, t_{i+1} - t_i) per table entry, as doubles
    double fold_c[4];           // split: n, C(n,2), C(n,3), C(n,4) for n = chunk
    const StripInfo* strips;    // split: strips of the line-interpolated sum, or null
    const int32_t* n_left;      // strips left, and done again
    int32_t strip_pass;         // StripPass bits of this launch
    double2* parts;             // plain: segment sums [segment][record], or null
    int64_t parts_stride;       // records per segment
    int32_t chunks;             // plain: delays by chunks of pulses (the kernel's choice)
};

// Host launchers (defined in bp_kernels.hip).  `grid` is the number of
// workgroups: the geometry and plain-sum kernels take one group of four tiles
// per workgroup (grid >= n_groups; extra workgroups return at once), the
// split kernel walks the wavefront tiles persistently.
hipError_t launch_pulse_orbit(const Orbit& orbit, double t0, double dt, int na, double* pv,
                              int32_t* flags, hipStream_t stream);
hipError_t launch_clear(int32_t* words, int n, hipStream_t stream);
hipError_t launch_geometry(const GeomArgs& args, int grid, hipStream_t stream);
hipError_t launch_fit(const GeomArgs& args, int grid, hipStream_t stream);
hipError_t launch_sum_plain(const SumArgs& args, int width, int grid, int segs, hipStream_t stream);
hipError_t launch_sum_split(const SumArgs& args, int width, int grid, bool staged, bool pair,
                            hipStream_t stream);
int sum_blocks_per_cu(int precision, int width, bool staged, bool pair);
// Strips up to which a segment of a line group gets four wavefronts instead of
// one.  Whole calls on tiles of 1, 4, 16 and 25 strips (32, 128, 256 and 300
// pixels square, 4,000 pulses): 221, 302, 394 and 461 us with four, 251, 356, 400
// and 443 us with one.
constexpr int kFewStrips = 16;

// Line-interpolated split sum (bp_lines.hip): workspace bytes per strip and
// its placement, kernels and their grids.
enum LineKernel : int { kLineFit = 0, kLineNodes, kLineLines, kLineFew, kLineEnds, kLineSum };
size_t line_strip_bytes(int slots, int n_sums);
size_t line_carry_bytes();
void line_place(LineArgs& a, unsigned char* ws, int64_t n_strips);
const void* line_kernel_fn(int which, int width);
int64_t line_grid(int which, int slots, int64_t n_strips);
hipError_t launch_strip_fit(const GeomArgs& g, const LineArgs& a, int64_t grid, hipStream_t stream);
hipError_t launch_strips(const LineArgs& a, int width, bool last, hipStream_t stream);
// [kmin, kmax) of each band of band_rows output lines (n_bands workgroups).
hipError_t launch_band_window(const PixGeom* geom, int64_t length, int64_t width, int band_rows,
                              int64_t n_bands, int32_t* win, hipStream_t stream);
// Host-side handle of a kernel (0 geometry, 4 geometry for generic DEMs,
// 1 plain sum, 6 with a delay per pulse, 5 its segments' total, 2 split sum, 3 fit),
// as graph kernel nodes report it.
const void* kernel_fn(int which, int width, bool staged, bool pair);

// CPUs the calling thread may run on (its affinity mask; threads it starts
// inherit the mask), at least 1.
int usable_cpus();

// Scene facts the serving queue needs (bp_api.hip).
int scene_device(const struct bp_scene* scene);
// Argument rules of one output block (shape, PRF, output buffer), shared by
// the batched calls and the serving queue's admission; returns BP_SUCCESS or
// a negative code with the thread's message set.
int check_out_block(const bp_out_block& block);
int64_t scene_max_pixels(const struct bp_scene* scene);
int scene_max_blocks(const struct bp_scene* scene);

}  // namespace bp
