"""Workloads of the framework through its public entry points, for timing and
for comparing outputs.

``listed()`` gives the workloads, ``draw(rng)`` more of the same ranges,
``prepare(case, seed)`` what a program holds before the call (device tensors,
geometries, compressors, scenes), ``run(state)`` one pass, ``work(case)`` the
bytes and operations a pass cannot do without, ``exact(case, seed)`` the same
outputs in 64-bit arithmetic by plain torch.

The radar is the synthetic L-band stripmap of isce3_amd.sim: a straight track
at 747 km and 7.5 km/s, PRF 1520 Hz, 6.25 m range spacing, near range 850 km,
wavelength 0.2384 m.  Pulses are range compressed: unit point targets, speckle
in 0.8 of the band and white receiver noise.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from isce3_amd import focus, presum, rslc
from isce3_amd.container import RadarGeometry
from isce3_amd.core import KnabKernel, LUT2d, Orbit, TabulatedKernelF32, speed_of_light
from isce3_amd.geometry import DEMInterpolator
from isce3_amd.product import RadarGridParameters
from isce3_amd.sim import EPOCH

C = speed_of_light
WAVELENGTH = 0.2384
FC = C / WAVELENGTH
PRF, DR, R0 = 1520.0, 6.25, 850e3
ALTITUDE, SPEED, EARTH_A = 747e3, 7500.0, 6378137.0
EARTH_E2 = 0.006694379990141317
BANDWIDTH, TABLE = 0.8, 2048
FLAT_HEIGHT = 120.0        # without relief, and outside the raster
DEV = "cuda:0"

FLOPS_PER_UPDATE = 101     # algorithmic flops of one pixel-pulse update


def listed():
    return [
        # The reference's default precision on a small scene: a user's first
        # call, a single chip around a few targets (every pulse integrated).
        dict(name="chip plain 256x256", op="backproject", precision="plain", na=512, nr=2048,
             rows=256, cols=256, ds=6.0, width=8, dem="flat", tropo="nodelay", doppler=0.0,
             height=True),
        # One processing block as the RSLC workflow asks for it: kernel width
        # 9, biquintic DEM, TSX troposphere, native Doppler; odd sizes.
        dict(name="block plain 301x1003", op="backproject", precision="plain", na=5000, nr=2500,
             rows=301, cols=1003, ds=6.0, width=9, dem="biquintic", tropo="tsx", doppler=40.0,
             height=True),
        # The full-size block (16384 x 16384 pulses) in both precisions.
        dict(name="full plain 4096x4096", op="backproject", precision="plain", na=16384, nr=16384,
             rows=4096, cols=4096, ds=6.0, width=8, dem="bilinear", tropo="nodelay", doppler=0.0,
             height=False),
        dict(name="full split 4096x4096", op="backproject", precision="split", na=16384, nr=16384,
             rows=4096, cols=4096, ds=6.0, width=8, dem="bilinear", tropo="nodelay", doppler=0.0,
             height=False),
        # Tile requests of the serving layer against a resident raw set: the
        # smallest request, where latency counts, and a middling odd one.
        dict(name="tile split 32x32", op="scene", precision="split", na=8192, nr=16384, tiles=1,
             side_min=32, side_max=32, aspect=1.0, ds=6.0, width=8, dem="bilinear",
             tropo="nodelay", doppler=0.0),
        dict(name="tile split 310x290", op="scene", precision="split", na=8192, nr=16384, tiles=1,
             side_min=300, side_max=300, aspect=1.07, ds=6.0, width=9, dem="bilinear",
             tropo="tsx", doppler=0.0),
        # A batch of uneven tiles of one raw set, focused by one call.
        dict(name="batch split 12 tiles", op="blocks", precision="split", na=8192, nr=16384,
             tiles=12, side_min=64, side_max=700, aspect=2.0, ds=6.0, width=8, dem="bilinear",
             tropo="nodelay", doppler=0.0),
        # Range compression: a full raw set, a few short pulses, and pulses
        # with a chirp too long for the fused transforms.
        dict(name="rangecomp 16384x15000", op="rangecomp", batch=16384, n=15000, chirp=961,
             mode="Same"),
        dict(name="rangecomp 48x2049", op="rangecomp", batch=48, n=2049, chirp=65, mode="Full"),
        dict(name="rangecomp 300x30000 long", op="rangecomp", batch=300, n=30000, chirp=10001,
             mode="Valid"),
        # Gap filling and resampling of dithered pulses to the uniform grid.
        dict(name="presum 16384x16384", op="presum", na=16384, nr=16384, gap=20, dither=0.15,
             length=12.0),
        # Finishing a focused block for storage: range correction,
        # statistics, half-precision encoding.
        dict(name="rslc 4095x16383 c32", op="rslc", rows=4095, cols=16383, encoding="complex32",
             range_cor=True, prior=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["backproject", "backproject", "scene", "scene", "blocks", "rangecomp",
                     "rangecomp", "presum", "rslc", "rslc"])
    if op in ("backproject", "scene", "blocks"):
        case = dict(op=op, precision=rng.choice(["plain", "split"]), ds=rng.choice([6.0, 6.0, 9.0]),
                    width=rng.choice([8, 9]), dem=rng.choice(["flat", "bilinear"]),
                    tropo=rng.choice(["nodelay", "tsx"]), doppler=0.0)
        if op == "backproject":
            case.update(na=rng.randint(4000, 8192), nr=rng.randint(2048, 6000),
                        rows=_log_int(rng, 32, 1024), cols=_log_int(rng, 32, 1024),
                        height=rng.choice([True, False]))
        else:
            case.update(na=rng.randint(4096, 8192), nr=rng.randint(6000, 16384),
                        tiles=1 if op == "scene" else rng.randint(4, 16),
                        side_min=0, side_max=0, aspect=rng.choice([1.0, 1.5, 2.0]))
            if op == "scene":
                case.update(precision="split")
                case["side_min"] = case["side_max"] = _log_int(rng, 32, 1024)
            else:
                case.update(side_min=64, side_max=_log_int(rng, 100, 512))
        return case
    if op == "rangecomp":
        n = _log_int(rng, 500, 40000)
        return dict(op=op, batch=max(1, min(8192, _log_int(rng, 16, 4096 * 15000 // n))), n=n,
                    chirp=2 * (_log_int(rng, 33, max(34, min(n, 2000))) // 2) + 1,
                    mode=rng.choice(["Full", "Valid", "Same"]))
    if op == "presum":
        return dict(op=op, na=_log_int(rng, 500, 6000), nr=_log_int(rng, 1000, 16384),
                    gap=rng.randint(0, 60), dither=rng.choice([0.1, 0.15, 0.25]),
                    length=rng.choice([8.0, 12.0, 16.0]))
    return dict(op=op, rows=_log_int(rng, 64, 8192), cols=_log_int(rng, 300, 16384),
                encoding=rng.choice(["complex64", "complex32", "complex64_zero_mantissa"]),
                range_cor=rng.choice([True, True, False]), prior=rng.choice([True, False]))


# ---------------------------------------------------------------- inputs

def _generator(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


def _complex_normal(shape, gen, variance=1.0):
    x = torch.randn(tuple(shape), dtype=torch.complex64, device=DEV, generator=gen)
    return x.mul_(math.sqrt(variance))


def _grids(case):
    """Input grid and the grid that outputs are cut from, both centred in
    azimuth on t = 0; outputs keep clear of the swath's ends."""
    na, nr = case["na"], case["nr"]
    in_grid = RadarGridParameters(-0.5 * na / PRF, WAVELENGTH, PRF, R0, DR, "right", na, nr, EPOCH)
    if case["op"] == "backproject":
        rows, cols = case["rows"], case["cols"]
    else:
        rows, cols = na // 2, 3 * nr // 4
    out_grid = RadarGridParameters(-0.5 * rows / PRF, WAVELENGTH, PRF,
                                   R0 + 0.5 * (nr - cols) * DR, DR, "right", rows, cols, EPOCH)
    return in_grid, out_grid


def _tiles(case, seed):
    """(row, column, lines, samples) of each output of a case, in the grid
    that outputs are cut from."""
    _, g = _grids(case)
    if case["op"] == "backproject":
        return [(0, 0, g.length, g.width)]
    rng = np.random.default_rng([int(seed), 5])
    # the sides are the case's: positions alone follow the seed
    shape = np.random.default_rng([case["tiles"], case["side_min"], case["side_max"]])
    out = []
    for _ in range(case["tiles"]):
        side = math.exp(shape.uniform(math.log(case["side_min"]), math.log(case["side_max"])))
        a = case["aspect"] if case["tiles"] == 1 else shape.uniform(1 / case["aspect"], case["aspect"])
        nl = int(min(g.length, max(1, round(side * math.sqrt(a)))))
        nw = int(min(g.width, max(1, round(side / math.sqrt(a)))))
        out.append((int(rng.integers(0, g.length - nl + 1)), int(rng.integers(0, g.width - nw + 1)),
                    nl, nw))
    return out


def _orbit_arrays():
    t = -50.0 + 10.0 * np.arange(11)
    p0 = np.array([EARTH_A + ALTITUDE, 0.0, 0.0])
    v = np.array([0.0, 0.0, SPEED])
    return t, p0[None, :] + t[:, None] * v[None, :], np.repeat(v[None, :], 11, axis=0)


def _dem_arrays(case, seed):
    """Fractal relief of 100 m (Hurst exponent 0.8, 30 m posting) around the
    middle of the outputs: (raster, x0, y0, step) in degrees, or None."""
    if case["dem"] == "flat":
        return None
    n = 1024
    rng = np.random.default_rng([int(seed), 7])
    k = np.hypot(np.fft.fftfreq(n)[None, :], np.fft.fftfreq(n)[:, None])
    k[0, 0] = np.inf
    spec = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) * k ** -1.8
    z = np.real(np.fft.ifft2(spec))
    z *= 100.0 / z.std()
    # ground point under the middle: slant range r, height 0 on a sphere
    r = R0 + 0.5 * case["nr"] * DR
    a = EARTH_A + ALTITUDE
    # right-looking and northbound: the swath lies east of the track
    lon = math.degrees(math.acos((a * a + EARTH_A ** 2 - r * r) / (2 * a * EARTH_A)))
    d = 30.0 / (EARTH_A * math.pi / 180.0)
    return z.astype(np.float32), lon - 0.5 * n * d, -0.5 * n * d, d


def _pulses(case, seed, in_grid, out_grid):
    """Range-compressed pulses [na, nr] on the GPU."""
    na, nr = in_grid.length, in_grid.width
    gen = _generator(seed, 1)
    raw = torch.empty((na, nr), dtype=torch.complex64, device=DEV)
    keep = (torch.fft.fftfreq(nr, device=DEV).abs() <= 0.5 * BANDWIDTH).to(torch.float32)
    for k in range(0, na, 2048):
        x = _complex_normal((min(2048, na - k), nr), gen, 0.05 / BANDWIDTH)
        raw[k:k + 2048] = torch.fft.ifft(torch.fft.fft(x) * keep)
        raw[k:k + 2048] += _complex_normal(x.shape, gen, 0.01)
    # point targets seen over the synthetic aperture
    rng = np.random.default_rng([int(seed), 3])
    tk = in_grid.sensing_start + torch.arange(na, dtype=torch.float64, device=DEV) / PRF
    taps = torch.arange(-16, 17, device=DEV)
    for _ in range(12):
        t = out_grid.sensing_start + rng.uniform(0, out_grid.length) / PRF
        r = out_grid.starting_range + rng.uniform(0, out_grid.width) * DR
        s = SPEED * (tk - t)
        rr = torch.sqrt(r * r + s * s)
        tau = 2.0 * (SPEED * s + C * rr) / (C * C - SPEED * SPEED)
        seen = (s.abs() / rr <= 1.5 * WAVELENGTH / (4.0 * case["ds"])).to(torch.float64)
        u = (tau - 2.0 * R0 / C) / (2.0 * DR / C)
        j = torch.round(u).long()[:, None] + taps[None, :]
        x = u[:, None] - j
        resp = torch.sinc(BANDWIDTH * x) * torch.cos(0.5 * math.pi * x / 17.0).clamp(min=0)
        ph = torch.polar(seen, -2.0 * math.pi * torch.frac(FC * tau))
        # the responses stay inside the line: outputs keep clear of its ends
        raw.scatter_add_(1, j.clamp(0, nr - 1), (resp * ph[:, None]).to(torch.complex64))
    return raw


def _doppler(case, in_grid):
    if case["doppler"] == 0.0:
        return LUT2d()
    fd = case["doppler"]
    xs = R0 + DR * np.array([-10.0, in_grid.width + 10.0])
    ys = np.array([-49.0, 49.0])
    return LUT2d(xs, ys, fd + 0.05 * ys[:, None] + 1e-4 * (xs[None, :] - R0))


def _chirp(case):
    m = case["chirp"]
    # an up-chirp over 0.8 of the sampling rate
    t = (np.arange(m) - (m - 1) / 2)
    return np.exp(1j * math.pi * 0.8 / m * t * t).astype(np.complex64)


def _presum_inputs(case, seed):
    nt, nr = case["na"], case["nr"]
    rng = np.random.default_rng([int(seed), 9])
    t = np.sort((np.arange(nt) - nt / 2) / PRF + rng.uniform(-1, 1, nt) * case["dither"] / PRF)
    gap = case["gap"]
    g = 200 + (np.arange(nt) * 997) % (nr - 400)
    sw = np.zeros((2, nt, 2), np.int64)
    sw[0, :, 1] = g
    sw[1, :, 0], sw[1, :, 1] = np.minimum(g + gap, nr), nr
    xs = R0 + DR * np.array([-10.0, nr + 10.0])
    ys = t[0] + np.array([-1.0, 12.0])
    fd = 50 + 20.0 * (ys[:, None] - t[0]) + 1e-4 * (xs[None, :] - R0)
    return t, sw, xs, ys, fd


def prepare(case, seed):
    op = case["op"]
    if op in ("backproject", "scene", "blocks"):
        in_grid, out_grid = _grids(case)
        t, pos, vel = _orbit_arrays()
        orbit = Orbit.from_arrays(EPOCH, float(t[0]), 10.0, pos, vel)
        dem = DEMInterpolator(FLAT_HEIGHT, "biquintic" if case["dem"] == "biquintic" else "bilinear")
        arrays = _dem_arrays(case, seed)
        if arrays is not None:
            z, x0, y0, d = arrays
            dem.load_dem_array(z, x0, y0, d, d)
        kernel = TabulatedKernelF32(KnabKernel(float(case["width"]), BANDWIDTH), TABLE)
        raw = _pulses(case, seed, in_grid, out_grid)
        doppler = _doppler(case, in_grid)
        grids = [out_grid.offset_and_resize(*x) for x in _tiles(case, seed)]
        st = dict(case=case, raw=raw, orbit=orbit, dem=dem, kernel=kernel, grids=grids,
                  in_geometry=RadarGeometry(in_grid, orbit, doppler),
                  out_geometries=[RadarGeometry(g, orbit, LUT2d()) for g in grids],
                  outs=[torch.empty(g.shape, dtype=torch.complex64, device=DEV) for g in grids],
                  height=(torch.empty(grids[0].shape, dtype=torch.float32, device=DEV)
                          if case.get("height") else None))
        if op == "scene":
            st["scene"] = focus.Scene(raw, st["in_geometry"], orbit, LUT2d(), dem, FC, case["ds"],
                                      kernel, case["tropo"], precision=case["precision"],
                                      max_pixels=sum(g.size for g in grids),
                                      max_blocks=len(grids))
        return st
    if op == "rangecomp":
        comp = focus.RangeComp(_chirp(case), case["n"], maxbatch=case["batch"],
                               mode=getattr(focus.RangeComp.Mode, case["mode"]))
        x = _complex_normal((case["batch"], case["n"]), _generator(seed, 2))
        return dict(case=case, comp=comp, x=x,
                    y=torch.empty((case["batch"], comp.output_size), dtype=torch.complex64,
                                  device=DEV))
    if op == "presum":
        t, sw, xs, ys, fd = _presum_inputs(case, seed)
        ot, pos, vel = _orbit_arrays()
        grid = RadarGridParameters(t[0], WAVELENGTH, PRF, R0, DR, "right", case["na"], case["nr"],
                                   EPOCH)
        return dict(case=case, t=t, sw=sw, grid=grid, lut=LUT2d(xs, ys, fd),
                    orbit=Orbit.from_arrays(EPOCH, float(ot[0]), 10.0, pos, vel),
                    raw=_complex_normal((case["na"], case["nr"]), _generator(seed, 4)))
    shape = (case["rows"], case["cols"])
    z, rc, prior = _rslc_inputs(case, seed)
    return dict(case=case, finisher=rslc.BlockFinisher(shape[0] * shape[1]), z=z, rc=rc,
                prior=prior)


def _rslc_inputs(case, seed):
    shape = (case["rows"], case["cols"])
    gen = _generator(seed, 6)
    z = _complex_normal(shape, gen, 4.0)
    # a focused block is NaN where the geometry has no solution
    z[:, :3] = complex(float("nan"), float("nan"))
    rc = prior = None
    if case["range_cor"]:
        ph = torch.rand(shape[1:], device=DEV, generator=gen, dtype=torch.float64) * 2 * math.pi
        rc = torch.polar(torch.ones_like(ph), ph).to(torch.complex64)
    if case["prior"]:
        prior = _complex_normal(shape, gen)
    return z, rc, prior


# ---------------------------------------------------------------- one pass

def run(st):
    case = st["case"]
    op = case["op"]
    if op == "backproject":
        focus.backproject(st["outs"][0], st["out_geometries"][0], st["raw"], st["in_geometry"],
                          st["dem"], FC, case["ds"], st["kernel"], case["tropo"],
                          height=st["height"], precision=case["precision"])
        return st["outs"] if st["height"] is None else [st["outs"][0], st["height"]]
    if op == "scene":
        st["scene"].focus(st["outs"], st["grids"])
        return st["outs"]
    if op == "blocks":
        focus.backproject_blocks(st["outs"], st["out_geometries"], st["raw"], st["in_geometry"],
                                 st["dem"], FC, case["ds"], st["kernel"], case["tropo"],
                                 precision=case["precision"])
        return st["outs"]
    if op == "rangecomp":
        st["comp"].rangecompress(st["y"], st["x"])
        return st["y"]
    if op == "presum":
        return presum.resample(st["raw"], st["t"], st["grid"], st["sw"], st["orbit"], st["lut"],
                               L=case["length"])
    # the finisher updates the block in place: a block's values keep their
    # size from pass to pass (the range correction is a rotation), and what
    # was stored before is added to the block as it was focused
    z = st["z"] if st["prior"] is None else st["z"].clone()
    enc, stats = st["finisher"].finish(z, range_cor=st["rc"], prior=st["prior"],
                                       data_type=case["encoding"])
    figures = torch.tensor([v for p in (stats.real, stats.imag)
                            for v in (p.min, p.max, p.mean, p.sample_stddev)], dtype=torch.float32)
    out = dict(z=z, n_valid=stats.n_valid, stats=figures)
    if case["encoding"] == "complex32":
        out["encoded"] = enc.view(torch.int32)
    return out


# ---------------------------------------------------------------- accounting

def _updates(case):
    """Pixel-pulse updates of a case and the samples they touch."""
    cpi = WAVELENGTH * (R0 + 0.5 * case["nr"] * DR) * (1 + ALTITUDE / EARTH_A) / (2 * case["ds"])
    pulses = min(case["na"], cpi / SPEED * PRF)
    _, g = _grids(case)
    upd = px = touched = 0.0
    for _, _, nl, nw in _tiles(case, 0):
        px += nl * nw
        upd += nl * nw * pulses
        touched += min(case["na"], pulses + nl) * min(case["nr"], nw + 20)
    return upd, px, min(touched, float(case["na"]) * case["nr"])


def work(case):
    op = case["op"]
    if op in ("backproject", "scene", "blocks"):
        upd, px, touched = _updates(case)
        return dict(bytes=8 * touched + 8 * px + (4 * px if case.get("height") else 0),
                    flops=FLOPS_PER_UPDATE * upd)
    if op == "rangecomp":
        m, n, b = case["chirp"], case["n"], case["batch"]
        out = {"Full": n + m - 1, "Valid": abs(n - m) + 1, "Same": n}[case["mode"]]
        full = n + m - 1
        return dict(bytes=8.0 * b * (n + out), flops=b * full * (10 * math.log2(full) + 6))
    if op == "presum":
        n = float(case["na"]) * case["nr"]
        taps = 2 * case["length"] / SPEED * PRF
        return dict(bytes=16 * n, flops=n * taps * 12)
    n = float(case["rows"]) * case["cols"]
    store = case["range_cor"] or case["prior"] or case["encoding"] == "complex64_zero_mantissa"
    return dict(bytes=n * (8 + (8 if store else 0) + (8 if case["prior"] else 0) +
                           (4 if case["encoding"] == "complex32" else 0)), flops=n * 14)


# ---------------------------------------------------------------- 64 bits

def _knab_table(width):
    """The tabulated kernel's float32 samples (Knab's window times a sinc)."""
    hw = width / 2.0
    x = hw / (TABLE - 1.0) * np.arange(TABLE)
    c = math.pi * hw * (1.0 - BANDWIDTH)
    win = np.cosh(c * np.sqrt(np.maximum(1.0 - (x / hw) ** 2, 0.0))) / math.cosh(c)
    return torch.from_numpy((win * np.sinc(x)).astype(np.float32)).to(DEV).double()


def _tap_weights(width, table, x0):
    """Weights [..., width] of taps at offsets x0, x0 + 1, ...: linear
    interpolation of the table at |x|."""
    x = (x0[..., None] + torch.arange(width, dtype=torch.float64, device=DEV)).abs()
    a = x * ((TABLE - 1.0) / (width / 2.0))
    i = a.floor().clamp(max=TABLE - 2).long()
    t0 = table[i]
    w = t0 + (a - i) * (table[i + 1] - t0)
    return torch.where(x <= width / 2.0, w, torch.zeros_like(w))


def _spline_weights(f):
    """Weights of six samples at -1 .. 4 in their natural cubic spline at f,
    0 <= f < 1."""
    system, right = np.eye(6), np.zeros((6, 6))
    for k in range(1, 5):
        system[k, k - 1:k + 2] = (1 / 6, 2 / 3, 1 / 6)
        right[k, k - 1:k + 2] = (1, -2, 1)
    second = np.linalg.solve(system, right)   # second derivatives per sample value
    g = 1 - f
    out = [float(second[1, k]) * (g ** 3 - g) / 6 + float(second[2, k]) * (f ** 3 - f) / 6
           for k in range(6)]
    out[1], out[2] = out[1] + g, out[2] + f
    return out


def _ground(case, seed, t, r):
    """Zero-Doppler ground points of (t, r) [lines, samples]: (distance from
    the Earth's centre, ellipsoidal height, the vector to the zero-Doppler
    platform times the ellipsoid's normal, sine of the latitude)."""
    arrays = _dem_arrays(case, seed)
    e2 = EARTH_E2
    p = torch.tensor([EARTH_A + ALTITUDE, 0.0, 0.0], dtype=torch.float64, device=DEV)
    t, r = torch.broadcast_tensors(t[:, None], r[None, :])
    pz = SPEED * t

    def point(look):
        # the plane across the track: down is towards the axis, right is east
        return p[0] - r * torch.cos(look), r * torch.sin(look)

    def geodetic(x, y):
        q = torch.sqrt(x * x + y * y)
        lat = torch.atan2(pz, q * (1 - e2))
        for _ in range(6):
            n = EARTH_A / torch.sqrt(1 - e2 * torch.sin(lat) ** 2)
            h = q / torch.cos(lat) - n
            lat = torch.atan2(pz, q * (1 - e2 * n / (n + h)))
        n = EARTH_A / torch.sqrt(1 - e2 * torch.sin(lat) ** 2)
        h = q / torch.cos(lat) - n
        return torch.atan2(y, x), lat, h

    def terrain(lon, lat):
        if arrays is None:
            return torch.full_like(lon, FLAT_HEIGHT)
        z, x0, y0, d = arrays
        z = torch.from_numpy(z).to(DEV).double()
        col = (lon * 180 / math.pi - x0) / d
        row = (lat * 180 / math.pi - y0) / d
        n = z.shape[0]
        inside = (row.floor() >= 2) & (row.floor() < n - 1) & (col.floor() >= 2) & \
            (col.floor() < n - 1)
        col, row = col.clamp(0, n - 2), row.clamp(0, n - 2)
        i, j = row.floor().long().clamp(max=n - 2), col.floor().long().clamp(max=n - 2)
        if case["dem"] == "biquintic":
            wr, wc = _spline_weights(row - i), _spline_weights(col - j)
            h = torch.zeros_like(lon)
            for a in range(6):
                ia = (i - 2 + a).clamp(0, n - 2) + 1
                for b in range(6):
                    h += wr[a] * wc[b] * z[ia, (j - 2 + b).clamp(0, n - 2) + 1]
        else:
            fr, fc = row - i, col - j
            h = (z[i, j] * (1 - fr) * (1 - fc) + z[i, j + 1] * (1 - fr) * fc +
                 z[i + 1, j] * fr * (1 - fc) + z[i + 1, j + 1] * fr * fc)
        return torch.where(inside, h, torch.full_like(h, FLAT_HEIGHT))

    # bisection on the look angle: height above the terrain grows with it
    lo, hi = torch.zeros_like(r), torch.full_like(r, 0.5 * math.pi)
    for _ in range(52):
        mid = 0.5 * (lo + hi)
        x, y = point(mid)
        lon, lat, h = geodetic(x, y)
        above = h - terrain(lon, lat) > 0
        hi, lo = torch.where(above, mid, hi), torch.where(above, lo, mid)
    x, y = point(0.5 * (lo + hi))
    lon, lat, h = geodetic(x, y)
    n_hat = (torch.cos(lat) * torch.cos(lon), torch.cos(lat) * torch.sin(lon), torch.sin(lat))
    up = (p[0] - x) * n_hat[0] - y * n_hat[1]
    return torch.sqrt(x * x + y * y + pz * pz), h, up, n_hat[2]


def _exact_windows(case, seed, in_grid, t, r):
    """First and past-the-last pulse, tropospheric delay and height of every
    pixel [lines, samples]."""
    dist, h, up, sin_lat = _ground(case, seed, t, r)
    # native Doppler (zero, or a plane): seen s metres ahead of closest approach
    t, r = torch.broadcast_tensors(t[:, None], r[None, :])
    s = torch.zeros_like(r)
    for _ in range(30 if case["doppler"] else 0):
        rho = torch.sqrt(r * r + s * s)
        fd = case["doppler"] + 0.05 * (t - s / SPEED) + 1e-4 * (rho - R0)
        s = fd * WAVELENGTH * rho / (2.0 * SPEED)
    tn = t - s / SPEED
    rho = torch.sqrt(r * r + s * s)
    plat = torch.sqrt((EARTH_A + ALTITUDE) ** 2 + (SPEED * tn) ** 2)
    cpi = WAVELENGTH * rho * (plat / dist) / (2.0 * case["ds"]) / SPEED
    k0 = torch.floor((tn - 0.5 * cpi - in_grid.sensing_start) * PRF).clamp(min=0)
    k1 = torch.ceil((tn + 0.5 * cpi - in_grid.sensing_start) * PRF).clamp(max=case["na"])
    atm = torch.zeros_like(h)
    if case["tropo"] == "tsx":
        cos_inc = (up - s * sin_lat) / rho
        atm = 2.0 * 2.3 * torch.exp(-h / 6000.0) / (C * cos_inc)
    return k0.int(), k1.int(), atm, h


def _delay(r, s):
    """Two-way delay to a point at closest range r from s metres past it."""
    tau = torch.addcmul(r * r, s, s).sqrt_().mul_(C)
    return tau.add_(SPEED * s).mul_(2.0 / (C * C - SPEED * SPEED))


def _exact_pixels(case, raw, in_grid, t, r, k0, k1, atm):
    """Backprojection of [pixels] points (t, r), tap by tap."""
    na, nr, w = case["na"], case["nr"], case["width"]
    table = _knab_table(w)
    view = raw.as_strided((na * nr - w + 1, w), (1, 1))
    acc = torch.zeros(len(r), dtype=torch.complex128, device=DEV)
    a, b = int(k0.min()), int(k1.max())
    step = max(1, (1 << 22) // len(r))
    for ka in range(a, b, step):
        k = torch.arange(ka, min(b, ka + step), device=DEV)
        s = SPEED * ((in_grid.sensing_start + k.double() / PRF)[None, :] - t[:, None])
        tau = _delay(r[:, None], s).add_(atm[:, None])
        u = (tau - 2.0 * R0 / C) * (C / (2.0 * DR))
        low = (torch.ceil(u) if w % 2 == 0 else torch.round(u)) - w // 2
        on = (k[None, :] >= k0[:, None]) & (k[None, :] < k1[:, None])
        at = (low.long() + k[None, :] * nr).clamp_(0, len(view) - 1)
        wt = _tap_weights(w, table, low - u)
        x = (torch.view_as_real(view[at]) * wt[..., None]).sum(2)
        ph = torch.frac(FC * tau).mul_(2.0 * math.pi)
        acc += (torch.view_as_complex(x) * torch.polar(on.double(), ph)).sum(1)
    return acc


def _exact_block(case, raw, in_grid, t, r, k0, k1, atm):
    """Backprojection of a large block [lines, samples], pulse by pulse: the
    taps are summed at 2048 offsets per bin and interpolated between them."""
    nr, w, q = case["nr"], case["width"], 2048
    table = _knab_table(w)
    # a sample at j + f, 0 <= f < 1, is the sum over bins j - w // 2 + m
    # (one bin to spare on either side) of weight(m - w // 2 - f)
    f = torch.arange(q, dtype=torch.float64, device=DEV) / q
    m = torch.arange(w + 2, dtype=torch.float64, device=DEV) - (w + 2) // 2
    x = (m[:, None] - f[None, :]).abs()
    a = x * ((TABLE - 1.0) / (w / 2.0))
    i = a.floor().clamp(max=TABLE - 2).long()
    wts = torch.where(x <= w / 2.0, table[i] + (a - i) * (table[i + 1] - table[i]),
                      torch.zeros_like(a)).to(torch.complex128)
    acc = torch.zeros(atm.shape, dtype=torch.complex128, device=DEV)
    first, last = k0.amin(1).tolist(), k1.amax(1).tolist()
    c0 = max(0, int((r[0] - R0) / DR) - w - 8)
    c1 = min(nr, int((r[-1] - R0) / DR) + w + 700)
    for k in range(min(first), max(last)):
        lines = [n for n in range(len(first)) if first[n] <= k < last[n]]
        lo, hi = lines[0], lines[-1] + 1
        line = raw[k, c0:c1].to(torch.complex128).unfold(0, w + 2, 1) @ wts
        line = line.view(-1)
        s = SPEED * (in_grid.sensing_start + k / PRF - t[lo:hi, None])
        tau = _delay(r[None, :], s).add_(atm[lo:hi])
        # position in the fine line: bin c0 + (w + 2) // 2 is its start
        g = tau.mul(q * C / (2.0 * DR)).sub_(q * (2.0 * R0 / (2.0 * DR) + c0 + (w + 2) // 2))
        n = g.long()
        g -= n
        ph = tau.mul_(FC).frac_().mul_(2.0 * math.pi)
        on = ((k0[lo:hi] <= k) & (k1[lo:hi] > k)).double()
        y0, y1 = line[n], line[n + 1]
        y0 += (y1 - y0) * g
        acc[lo:hi] += y0 * torch.polar(on, ph)
    return acc


def _exact_image(case, seed, raw, in_grid, t, r):
    """One output block in 64 bits (taps, phases and sums), and its heights."""
    win = [_exact_windows(case, seed, in_grid, t[i:i + 256], r) for i in range(0, len(t), 256)]
    k0, k1, atm, height = (torch.cat(x) for x in zip(*win))
    if height.numel() >= 1 << 19:
        return _exact_block(case, raw, in_grid, t, r, k0, k1, atm), height
    tt, rr = (x.reshape(-1) for x in torch.broadcast_tensors(t[:, None], r[None, :]))
    k0, k1, atm = k0.reshape(-1), k1.reshape(-1), atm.reshape(-1)
    z = torch.cat([_exact_pixels(case, raw, in_grid, *(x[i:i + (1 << 16)]
                                                       for x in (tt, rr, k0, k1, atm)))
                   for i in range(0, len(rr), 1 << 16)])
    return z.view(height.shape), height


def _exact_presum(case, seed):
    t, sw, xs, ys, fdl = _presum_inputs(case, seed)
    nt, nr = case["na"], case["nr"]
    raw = _complex_normal((nt, nr), _generator(seed, 4))
    scale = case["length"] / SPEED

    def acorr(d):
        x = np.abs(2.0 * d / scale)
        return np.where(x > 2, 0.0, np.where(x < 1, x * x * (0.75 * x - 1.5) + 1,
                                             x * (x * (1.5 - 0.25 * x) - 3) + 2))

    out = torch.zeros((nt, nr), dtype=torch.complex128, device=DEV)
    r = R0 + DR * torch.arange(nr, dtype=torch.float64, device=DEV)
    sx = (fdl[0, 1] - fdl[0, 0]) / (xs[1] - xs[0])
    sy = (fdl[1, 0] - fdl[0, 0]) / (ys[1] - ys[0])
    tout = t[0] + np.arange(nt) / PRF
    first = np.searchsorted(t, tout - scale, side="left")
    last = np.searchsorted(t, tout + scale, side="right")
    # each output pulse's runs of range bins with one pattern of valid pulses
    runs, jobs = [], {}
    for i in range(nt):
        a, b = int(first[i]), int(last[i])
        cuts = np.unique(np.concatenate([[0, nr], sw[:, a:b].ravel()]))
        runs.append([])
        for c0, c1 in zip(cuts[:-1], cuts[1:]):
            ok = ((sw[:, a:b, 0] <= c0) & (c0 < sw[:, a:b, 1])).any(0)
            idx = np.nonzero(ok)[0]
            runs[i].append([c1 - c0, np.zeros(b - a)])
            jobs.setdefault(len(idx), []).append((i, runs[i][-1][1], idx))
    for m, todo in jobs.items():
        if m == 0:
            continue
        x = np.stack([t[first[i] + idx] for i, _, idx in todo])
        to = np.array([tout[i] for i, _, _ in todo])
        g = acorr(x[:, :, None] - x[:, None, :])
        v = np.linalg.solve(g, acorr(to[:, None] - x)[..., None])[..., 0]
        for (_, w, idx), wv in zip(todo, v):
            w[idx] = wv
    for i in range(nt):
        a, b = int(first[i]), int(last[i])
        if b == a:
            continue
        lens = torch.tensor([n for n, _ in runs[i]], device=DEV)
        tab = torch.from_numpy(np.stack([w for _, w in runs[i]], axis=1)).to(DEV)
        wt = torch.repeat_interleave(tab, lens, dim=1, output_size=nr)
        fd = fdl[0, 0] + sy * (tout[i] - ys[0]) + sx * (r - xs[0])
        trel = torch.from_numpy(t[a:b] - tout[i]).to(DEV)
        ph = torch.frac(-trel[:, None] * fd[None, :]).mul_(2 * math.pi)
        out[i] = (torch.polar(torch.ones_like(ph), ph) * wt * raw[a:b]).sum(0)
    return out


def exact(case, seed):
    op = case["op"]
    if op in ("backproject", "scene", "blocks"):
        in_grid, out_grid = _grids(case)
        raw = _pulses(case, seed, in_grid, out_grid)
        outs = []
        for r0, c0, nl, nw in _tiles(case, seed):
            t = out_grid.sensing_start + (r0 + torch.arange(nl, dtype=torch.float64, device=DEV)) / PRF
            r = out_grid.starting_range + (c0 + torch.arange(nw, dtype=torch.float64, device=DEV)) * DR
            z, h = _exact_image(case, seed, raw, in_grid, t, r)
            outs.append(z)
            if case.get("height"):
                outs.append(h)
        return outs
    if op == "rangecomp":
        x = _complex_normal((case["batch"], case["n"]), _generator(seed, 2))
        h = np.conj(_chirp(case)[::-1]).astype(np.complex128)
        m, n = case["chirp"], case["n"]
        size = 1 << (n + m - 2).bit_length()
        hf = torch.fft.fft(torch.from_numpy(h).to(DEV), size)
        off, length = {"Full": (0, n + m - 1), "Valid": (min(m, n) - 1, abs(n - m) + 1),
                       "Same": (m // 2, n)}[case["mode"]]
        out = torch.empty((case["batch"], length), dtype=torch.complex128, device=DEV)
        for k in range(0, case["batch"], 1024):
            f = torch.fft.fft(x[k:k + 1024].to(torch.complex128), size)
            out[k:k + 1024] = torch.fft.ifft(f.mul_(hf))[:, off:off + length]
        return out
    if op == "presum":
        return _exact_presum(case, seed)
    z, rc, prior = _rslc_inputs(case, seed)
    y = z.to(torch.complex128)
    if rc is not None:
        y *= rc.to(torch.complex128)
    if prior is not None:
        y += prior
    figures = []
    for v in (y.real, y.imag):
        v = v[~torch.isnan(v)]
        figures += [v.min(), v.max(), v.mean(), v.std()]
    # truncated mantissas and encoded bytes have no value in 64 bits
    out = dict(z=None if case["encoding"] == "complex64_zero_mantissa" else y, n_valid=None,
               stats=torch.stack(figures))
    if case["encoding"] == "complex32":
        out["encoded"] = None
    return out
