"""The line-interpolated split sum (strips of output lines focused from a few
of them) against the all-FP64 oracle, on random pulses and a full synthetic
aperture (about 4,000 pulses): strip heights and widths at their edges, both
kernel widths it takes, straight and curved orbits over rough terrain, and
blocks where it takes none or only some of the strips.

Tolerances, from the method's own bounds: the tap weights are within 1e-5 of
the tabulated kernel at any position (2e-6 at width 9), which white pulses turn
into at most sqrt(8) x 1e-5 = 2.8e-5 relative; the node interpolation leaves at
most 1.5e-4 at a chunk's end, a tenth of that on average; FP32 phases of 16
cycles 6e-6 rad: 6e-5 together.  Over rough terrain from a curved orbit a strip
may stray 1e-4 rad from its nodes at a chunk's ends, 6e-5 RMS over the chunk:
1e-4 with the other terms.  The pixel-by-pixel sum's weight table is good to
1.5e-4 on white pulses: 2e-4 where it takes part."""
import numpy as np
import pytest

import oracle
from helpers import complex_rel_error

pytestmark = pytest.mark.gpu

NA, NR = 4600, 192


def _scene(width=8, orbit="straight", relief=0.0, doppler=0.0, na=NA, bandwidth=0.8,
           dr=None):
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import KnabKernel, LUT2d, Orbit, TabulatedKernelF32
    from isce3_amd.geometry import DEMInterpolator
    if orbit == "straight":
        orb = sim.straight_orbit()
    else:
        t = -50.0 + 10.0 * np.arange(11)
        r = sim.WGS84_A + sim.ALTITUDE
        a = sim.SPEED / r * t
        orb = Orbit.from_arrays(
            sim.EPOCH, -50.0, 10.0,
            np.stack([r * np.cos(a), 0 * a, r * np.sin(a)], axis=1),
            sim.SPEED * np.stack([-np.sin(a), 0 * a, np.cos(a)], axis=1))
    in_grid = sim._grid(-0.5 * na / sim.PRF, sim.PRF, sim.R0, dr or sim.DR, na, NR)
    dem = DEMInterpolator(50.0)
    if relief:
        dem = sim._dem_around(orb, in_grid, 256, 30.0, 0.8, relief, 3)
    xs = sim.R0 + sim.DR * np.array([-20.0, NR + 20.0])
    ys = np.array([-45.0, 45.0])
    lut = LUT2d(xs, ys, np.full((2, 2), doppler)) if doppler else LUT2d()
    rng = np.random.default_rng(5)
    raw = (rng.standard_normal((na, NR)) + 1j * rng.standard_normal((na, NR))).astype(np.complex64)
    kernel = TabulatedKernelF32(KnabKernel(float(width), bandwidth), 2048)
    return orb, RadarGeometry(in_grid, orb, lut), dem, raw, kernel


def _run(scene, rows, cols, c0=40, dr=None, prf=None, tropo="nodelay", options=None, ds=6.0,
         bandwidth=0.8):
    """(GPU split result, FP64 oracle) of a block of rows x cols pixels."""
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import LUT2d
    from isce3_amd.focus import backproject
    orb, in_geom, dem, raw, kernel = scene
    prf = prf or sim.PRF
    grid = sim._grid(-0.5 * rows / prf + 0.3 / prf, prf, sim.R0 + (c0 + 0.37) * sim.DR,
                     dr or sim.DR, rows, cols)
    og = RadarGeometry(grid, orb, LUT2d())
    out = np.empty(grid.shape, np.complex64)
    err = backproject(out, og, raw, in_geom, dem, sim.FC, ds, kernel, tropo, precision="split",
                      options=options)
    ref, _, _, rc = oracle.backproject(og, raw, in_geom, dem, sim.FC, ds, kernel, tropo, mode=1,
                                       kernel_bandwidth=bandwidth)
    assert err == (rc == 6)
    rel = complex_rel_error(out, ref)
    print(f"[lines] {rows}x{cols} rel={rel:.2e}", flush=True)
    assert (np.isnan(out) == np.isnan(ref)).all()
    return rel


@pytest.mark.parametrize("width", [8, 9])
@pytest.mark.parametrize("rows,cols", [(1, 64), (5, 3), (16, 65), (33, 64), (64, 20), (65, 63),
                                       (130, 40)])
def test_strip_edges_match_fp64_oracle(torch_gpu, width, rows, cols):
    assert _run(_scene(width), rows, cols) <= 6e-5


@pytest.mark.parametrize("orbit,relief,tropo", [("straight", 100.0, "tsx"),
                                                ("circular", 0.0, "nodelay"),
                                                ("circular", 100.0, "tsx")])
def test_orbits_and_terrain_match_fp64_oracle(torch_gpu, orbit, relief, tropo):
    assert _run(_scene(8, orbit, relief), 96, 70, tropo=tropo) <= 1e-4


@pytest.mark.parametrize("ds,na,dr,c0", [(5.0, NA + 800, None, 40), (3.0, 8200, None, 60),
                                         (4.0, 6400, 3.0, 40)])
@pytest.mark.parametrize("rows,cols,tropo", [(16, 40, "nodelay"), (33, 20, "tsx"), (70, 33, "nodelay")])
def test_finer_resolutions(torch_gpu, ds, na, dr, c0, rows, cols, tropo):
    """Strips of 32 lines with 64 pulses per chunk (5 m) and with 32 (3 m), and of 16
    lines (4 m with a range spacing of 3 m), over whole apertures of 4,600, 7,700 and
    5,700 pulses that stay inside the range line."""
    assert _run(_scene(8, na=na, dr=dr), rows, cols, c0=c0, ds=ds, dr=dr, tropo=tropo) <= 6e-5


@pytest.mark.parametrize("width,bandwidth", [(8, 0.6), (9, 0.9)])
def test_other_kernels(torch_gpu, width, bandwidth):
    assert _run(_scene(width, bandwidth=bandwidth), 50, 64, bandwidth=bandwidth) <= 6e-5


@pytest.mark.parametrize("kw", [dict(dr=9.0), dict(prf=400.0), dict(c0=-30), dict(c0=150)])
def test_strips_left_to_the_pixel_sum(torch_gpu, kw):
    """Output range spacing off the input's, lines too far apart, and blocks
    whose first or last columns' taps leave the range line (a strip of 64
    columns beside one that qualifies)."""
    assert _run(_scene(8), 40, 100 if "c0" in kw else 40, **kw) <= 2e-4


def test_native_doppler(torch_gpu):
    """A squinted aperture, whose lines lie further apart at its far end."""
    assert _run(_scene(8, doppler=400.0), 48, 64) <= 2e-4


@pytest.mark.parametrize("doppler", [150.0, 400.0])
@pytest.mark.parametrize("rows,cols", [(32, 64), (33, 20), (100, 70)])
def test_squinted_strips(torch_gpu, doppler, rows, cols):
    """The plan takes strips of 32 lines (and 32 pulses per chunk) for it, which
    qualify: the line-interpolated sum's tolerance."""
    assert _run(_scene(8, doppler=doppler), rows, cols) <= 6e-5


def test_grids_without_strips(torch_gpu):
    """Grids off the input's range spacing, or with lines too far apart, beside
    one of strips in a batch: each as alone, to the bit, and alone they take no
    strip workspace."""
    import ctypes as C
    from isce3_amd import _native, sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import LUT2d
    from isce3_amd.focus import backproject, backproject_blocks
    orb, in_geom, dem, raw, kernel = _scene(8)
    d_raw = torch_gpu.from_numpy(raw).to("cuda:0")

    def grid(rows, cols, dr=1.0, prf=1.0):
        return sim._grid(-0.5 * rows / sim.PRF, sim.PRF / prf, sim.R0 + 40 * sim.DR, dr * sim.DR,
                         rows, cols)

    grids = [grid(64, 70, dr=0.75), grid(65, 70), grid(48, 70, prf=5.0), grid(33, 64),
             grid(20, 40, dr=1.25)]
    geoms = [RadarGeometry(g, orb, LUT2d()) for g in grids]

    def empty(g):
        return torch_gpu.empty(tuple(g.shape), dtype=torch_gpu.complex64, device="cuda:0")

    alone = [empty(g) for g in grids]
    for o, g in zip(alone, geoms):
        backproject(o, g, d_raw, in_geom, dem, sim.FC, 6.0, kernel, "nodelay", precision="split")
    batch = [empty(g) for g in grids]
    backproject_blocks(batch, geoms, d_raw, in_geom, dem, sim.FC, 6.0, kernel, "nodelay",
                       precision="split")
    for a, b in zip(alone, batch):
        np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())

    def taken(g):
        from isce3_amd.focus import geometry_struct, parse_geo2rdr_params, parse_rdr2geo_params
        ctx, st, failed = C.c_void_p(), _native.Stats_t(), C.c_int(0)
        lib = _native.lib()
        _native.check(lib.bp_context_create(0, C.byref(ctx)))
        out, geom = empty(g), RadarGeometry(g, orb, LUT2d())
        og, ig = geometry_struct(geom), geometry_struct(in_geom)
        dm, kr, opt = dem._struct(), kernel._struct(), _native.Options_t()
        r2g, g2r = parse_rdr2geo_params({}), parse_geo2rdr_params({})
        torch_gpu.cuda.synchronize()
        free = torch_gpu.cuda.mem_get_info(0)[0]
        rc = lib.bp_backproject(ctx, C.byref(og), C.byref(ig), C.byref(dm), sim.FC, 6.0, C.byref(kr),
                                0, C.byref(r2g), C.byref(g2r), C.c_void_p(d_raw.data_ptr()),
                                C.c_void_p(out.data_ptr()), None, _native.PRECISION_SPLIT,
                                C.byref(opt), None, C.byref(failed), C.byref(st))
        n = free - torch_gpu.cuda.mem_get_info(0)[0]
        _native.check(rc)
        lib.bp_context_destroy(ctx)
        return n

    # 4096 pixels of 112 bytes a strip, against 0.3 MB of workspace as well
    assert taken(grid(640, 640, dr=0.75)) <= 640 * 640 * 112 + (8 << 20)
    assert taken(grid(640, 640)) >= 640 * 640 * 112 + (24 << 20)


@pytest.mark.parametrize("width,ds,na,c0,cols", [(9, 6.0, NA, 40, 70), (8, 3.0, 8200, 60, 40),
                                                 (8, 6.0, NA, -30, 130)])
def test_whole_and_band_by_band_agree(torch_gpu, width, ds, na, c0, cols):
    """Pulses in host memory under a budget below a strip's window: the strip's
    pulses go through the device in parts, with the same result to the bit; with
    chunks of 64 and of 32 pulses, and with strips beside them that are left to the
    pixel-by-pixel sum (a block that begins before the swath)."""
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import LUT2d
    from isce3_amd.focus import backproject
    orb, in_geom, dem, raw, kernel = _scene(width, na=na)
    grid = sim._grid(-0.5 * 150 / sim.PRF, sim.PRF, sim.R0 + c0 * sim.DR, sim.DR, 150, cols)
    og = RadarGeometry(grid, orb, LUT2d())
    lines = 64 if ds >= 6 else 32
    outs = []
    # whole; bands of one strip row each (its lines' window); parts of a strip's window
    windows = [0]
    for windows_of in (0, 1, 2):
        budget = windows[windows_of] * NR * 8
        out = np.empty(grid.shape, np.complex64)
        st = {}
        backproject(out, og, raw, in_geom, dem, sim.FC, ds, kernel, "nodelay",
                    precision="split", max_window_bytes=budget, stats=st)
        print(f"[lines] budget {budget}: {st['bands']} bands, {st['window_pulses']} pulses",
              flush=True)
        outs.append(out)
        if not windows_of:
            strip = st["window_pulses"] - 150 + lines
            windows += [strip + lines // 2, strip - lines // 2]
        else:
            assert st["bands"] >= 2
    np.testing.assert_array_equal(outs[1], outs[0])
    np.testing.assert_array_equal(outs[2], outs[0])


def test_groups_of_one_strip_agree(torch_gpu):
    """A context whose workspace is limited to one strip runs a block of 18 strips
    in as many groups, with the same result to the bit."""
    import ctypes as C
    from isce3_amd import _native, sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import LUT2d
    from isce3_amd.focus import geometry_struct, parse_geo2rdr_params, parse_rdr2geo_params
    orb, in_geom, dem, raw, kernel = _scene(8)
    d_raw = torch_gpu.from_numpy(raw).to("cuda:0")
    geom = RadarGeometry(sim._grid(-0.2, sim.PRF, sim.R0 + 40 * sim.DR, sim.DR, 64 * 6, 130), orb,
                         LUT2d())
    og, ig, dm, kr = geometry_struct(geom), geometry_struct(in_geom), dem._struct(), kernel._struct()
    r2g, g2r = parse_rdr2geo_params({}), parse_geo2rdr_params({})
    lib, outs = _native.lib(), []
    for limit in (-1, 0):
        ctx, failed, opt, st = C.c_void_p(), C.c_int(0), _native.Options_t(), _native.Stats_t()
        _native.check(lib.bp_context_create(0, C.byref(ctx)))
        _native.check(lib.bp_context_limit_workspace(ctx, limit))
        out = torch_gpu.empty((64 * 6, 130), dtype=torch_gpu.complex64, device="cuda:0")
        torch_gpu.cuda.synchronize()
        rc = lib.bp_backproject(ctx, C.byref(og), C.byref(ig), C.byref(dm), sim.FC, 6.0, C.byref(kr),
                                0, C.byref(r2g), C.byref(g2r), C.c_void_p(d_raw.data_ptr()),
                                C.c_void_p(out.data_ptr()), None, _native.PRECISION_SPLIT,
                                C.byref(opt), None, C.byref(failed), C.byref(st))
        lib.bp_context_destroy(ctx)
        _native.check(rc)
        outs.append(out.cpu().numpy())
    np.testing.assert_array_equal(outs[1], outs[0])
    assert np.isfinite(outs[0]).all()


@pytest.mark.parametrize("width,tropo", [(8, "nodelay"), (9, "tsx")])
def test_few_and_many_strips_agree(torch_gpu, width, tropo):
    """The lines kernel of a few strips (four wavefronts per segment) and that of
    many, on the same strip: a block of 18 strips and its first one alone, the
    same to the bit."""
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import LUT2d
    from isce3_amd.focus import backproject
    orb, in_geom, dem, raw, kernel = _scene(width, relief=100.0 if tropo == "tsx" else 0.0)
    outs = []
    for cols, rows in ((64, 64 * 18), (64, 64)):
        grid = sim._grid(-0.2, sim.PRF, sim.R0 + 40 * sim.DR, sim.DR,
                         rows, cols)
        out = np.empty(grid.shape, np.complex64)
        backproject(out, RadarGeometry(grid, orb, LUT2d()), raw, in_geom, dem, sim.FC, 6.0, kernel,
                    tropo, precision="split")
        outs.append(out)
    np.testing.assert_array_equal(outs[0][:64], outs[1])


def test_budget_below_any_strip_window(torch_gpu):
    """Windows of about 45 pulses under a budget of 63: no strip qualifies with
    fewer than 64, so host pulses in bands of tile rows still give the resident
    call's result to the bit."""
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import LUT2d
    from isce3_amd.focus import backproject
    orb, in_geom, dem, raw, kernel = _scene(8)
    og = RadarGeometry(sim._grid(-0.5 * 130 / sim.PRF, sim.PRF, sim.R0 + 40 * sim.DR, sim.DR, 130, 70),
                       orb, LUT2d())
    outs = []
    for pulses in (NA, 63):
        out = np.empty((130, 70), np.complex64)
        backproject(out, og, raw, in_geom, dem, sim.FC, 500.0, kernel, "nodelay",
                    precision="split", max_window_bytes=pulses * NR * 8)
        outs.append(out)
    np.testing.assert_array_equal(outs[1], outs[0])
    assert np.isfinite(outs[0]).all()
