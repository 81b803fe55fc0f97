"""The C-ABI library: it loads without a GPU, exports every function its
headers declare, and its host-side primitives (the same FP64 code the kernels
run) agree with the oracle bit for bit or to the stated ULP-level tolerance."""
import ctypes as C
import math
import os
import re

import numpy as np
import pytest

import oracle
from isce3_amd import _native, core, geometry
from isce3_amd.sim import straight_orbit

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
REF = np.load(os.path.join(ROOT, "tests", "golden", "ref_blocks.npz"))
D3 = C.c_double * 3


def declared_functions(header):
    src = open(os.path.join(ROOT, "include", header)).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"^\s*(?:const\s+)?[a-z_0-9]+\s*\*?\s*(bp_\w+|sim_\w+)\s*\(",
                                 src, flags=re.M)))


@pytest.mark.parametrize("header,lib", [("isce3_amd_backproject.h", "libisce3_amd.so"),
                                        ("isce3_amd_rangecomp.h", "libisce3_amd.so"),
                                        ("isce3_amd_rslc.h", "libisce3_amd.so"),
                                        ("isce3_amd_presum.h", "libisce3_amd.so"),
                                        ("isce3_amd_sim.h", "libisce3_amd_sim.so")])
def test_library_exports_every_declared_symbol(header, lib):
    names = declared_functions(header)
    assert len(names) >= {"isce3_amd_sim.h": 2, "isce3_amd_rangecomp.h": 4, "isce3_amd_rslc.h": 3,
                          "isce3_amd_presum.h": 5}.get(header, 15)
    h = C.CDLL(os.path.join(ROOT, "isce3_amd", "lib", lib))
    missing = [n for n in names if not hasattr(h, n)]
    assert not missing, missing


def declared_arities(header):
    src = open(os.path.join(ROOT, "include", header)).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    src = re.sub(r"//[^\n]*", "", src)
    out = {}
    for m in re.finditer(r"^\s*(?:const\s+)?[a-z_0-9]+\s*\*?\s*(bp_\w+)\s*\(([^;{]*?)\)\s*;",
                         src, flags=re.M):
        params = m.group(2).strip()
        out[m.group(1)] = 0 if params in ("", "void") else params.count(",") + 1
    return out


@pytest.mark.parametrize("header", ["isce3_amd_backproject.h", "isce3_amd_rangecomp.h",
                                    "isce3_amd_rslc.h", "isce3_amd_presum.h"])
def test_every_declared_function_has_a_binding_of_its_arity(header):
    """ctypes converts Python floats and ints only for functions whose argument
    types are declared: every function of the headers has a binding in the
    package, with as many arguments as the declaration."""
    arity = declared_arities(header)
    assert set(arity) == set(declared_functions(header))
    unbound = [n for n in arity if n not in _native._SIGNATURES]
    assert not unbound, unbound
    wrong = {n: (a, len(_native._SIGNATURES[n][1])) for n, a in arity.items()
             if len(_native._SIGNATURES[n][1]) != a}
    assert not wrong, wrong


def test_context_create_without_gpu_fails_cleanly():
    """No GPU: context creation reports a HIP error instead of crashing."""
    try:
        import torch
        if torch.cuda.is_available():
            pytest.skip("a GPU is visible")
    except ImportError:
        pass
    h = C.c_void_p()
    rc = _native.lib().bp_context_create(0, C.byref(h))
    assert rc == _native.BP_ERR_HIP
    assert "device" in _native.last_error().lower()


def test_knab_table_matches_reference_bits():
    for w in (8.0, 9.0):
        k = core.TabulatedKernelF32(core.KnabKernel(w, 0.8), 2048)
        np.testing.assert_array_equal(k.table, REF[f"table_f32_w{w:g}_bw0.8"])


def test_tabulated_kernel_call_matches_reference():
    k = core.TabulatedKernelF32(core.KnabKernel(8.0, 0.8), 2048)
    got = np.array([k(x) for x in REF["tab_eval_x"][:800]], dtype=np.float32)
    np.testing.assert_array_equal(got, REF["tab_eval_w8"][:800])


def test_knab_kernel_call():
    k = core.KnabKernel(8.0, 0.8)
    np.testing.assert_allclose([k(x) for x in REF["knab_x"]], REF["knab_w8"], rtol=0, atol=1e-15)


def test_orbit_interpolation_matches_oracle():
    orb = straight_orbit()
    # perturb into a curved trajectory so all Hermite terms matter
    t = np.array(orb.time)
    pos = orb.position + 4.0 * np.column_stack([t ** 2, -0.5 * t ** 2, 0.1 * t ** 3 / 50])
    vel = orb.velocity + 4.0 * np.column_stack([2 * t, -t, 0.3 * t ** 2 / 50])
    o2 = core.Orbit.from_arrays(orb.reference_epoch, t[0], orb.spacing, pos, vel)
    os_ = oracle.orbit_struct(o2)
    rng = np.random.Generator(np.random.PCG64(3))
    for tt in rng.uniform(t[0], t[-1], 200):
        p, v = o2.interpolate(tt)
        po, vo = D3(), D3()
        assert oracle.lib().orc_orbit_interpolate(C.byref(os_), tt, 0, po, vo) == 0
        np.testing.assert_allclose(p, list(po), rtol=0, atol=1e-9)
        np.testing.assert_allclose(v, list(vo), rtol=0, atol=1e-12)
    with pytest.raises(IndexError):
        o2.interpolate(t[-1] + 1.0)


def test_ellipsoid_matches_oracle():
    e = core.Ellipsoid()
    rng = np.random.Generator(np.random.PCG64(4))
    for _ in range(100):
        llh = np.array([rng.uniform(-3, 3), rng.uniform(-1.4, 1.4), rng.uniform(-400, 8000)])
        xyz = e.lon_lat_to_xyz(llh)
        xo = D3()
        oracle.lib().orc_lonlat_to_xyz(e.a, e.e2, D3(*llh), xo)
        np.testing.assert_allclose(xyz, list(xo), rtol=0, atol=1e-8)
        back = e.xyz_to_lon_lat(xyz)
        lo = D3()
        oracle.lib().orc_xyz_to_lonlat(e.a, e.e2, D3(*xyz), lo)
        # the product code takes a cube root where the reference (and the
        # oracle) call pow(x, 1/3): heights agree to ~1e-9 m
        np.testing.assert_allclose(back[:2], list(lo)[:2], rtol=0, atol=1e-12)
        assert abs(back[2] - lo[2]) < 1e-8


def test_dem_and_lut_match_oracle():
    rng = np.random.Generator(np.random.PCG64(6))
    z = rng.normal(0, 100, (64, 80)).astype(np.float32)
    dem = geometry.DEMInterpolator(12.5).load_dem_array(z, 7.0, -0.2, 0.001, 0.0012)
    do = oracle.dem_struct(dem)
    for _ in range(300):
        x, y = rng.uniform(6.99, 7.09), rng.uniform(-0.21, -0.12)
        assert dem.interpolate_xy(x, y) == oracle.lib().orc_dem_interpolate_xy(C.byref(do), x, y)
        lon, lat = math.radians(x), math.radians(y)
        assert dem.interpolate_lonlat(lon, lat) == oracle.lib().orc_dem_interpolate_lonlat(
            C.byref(do), lon, lat)
    data = rng.normal(0, 50, (5, 7))
    lut = core.LUT2d(800e3, -3.0, 100.0, 0.5, data)
    lo = oracle.lut_struct(lut)
    for _ in range(200):
        y, x = rng.uniform(-4, 1), rng.uniform(790e3, 801e3)
        assert lut.eval(y, x) == oracle.lib().orc_lut2d_eval(C.byref(lo), y, x)
    assert core.LUT2d().eval(1.0, 2.0) == 0.0


def test_bracket_solvers_match_oracle():
    from isce3_amd.sim import make_scene
    sc = make_scene("tiny")
    o = oracle.orbit_struct(sc.orbit)
    d = oracle.dem_struct(sc.dem)
    p = oracle.R2G_t(1e-5, 0.0, math.pi / 2)
    g = oracle.G2R_t(1e-7, 0, 0, 0.0, 0.0)
    lut = oracle.lut_struct(sc.doppler)
    for t, r in sc.target_radar:
        x = geometry.rdr2geo_bracket(t, r, sc.orbit, "right", 0.0, sc.out_grid.wavelength, sc.dem)
        xo = D3()
        assert oracle.lib().orc_rdr2geo_bracket(t, r, 0.0, C.byref(o), C.byref(d),
                                                sc.out_grid.wavelength, -1, C.byref(p), xo) == 0
        np.testing.assert_allclose(x, list(xo), rtol=0, atol=1e-6)
        ta, ra = geometry.geo2rdr_bracket(x, sc.orbit, sc.doppler, sc.out_grid.wavelength, "right")
        to, ro = C.c_double(), C.c_double()
        assert oracle.lib().orc_geo2rdr_bracket(D3(*x), C.byref(o), C.byref(lut),
                                                sc.out_grid.wavelength, -1, C.byref(g),
                                                C.byref(to), C.byref(ro)) == 0
        assert abs(ta - to.value) < 1e-9 and abs(ra - ro.value) < 1e-6
        # round trip: zero-Doppler time and range of the located target
        assert abs(ta - t) < 1e-6 and abs(ra - r) < 1e-4


def test_datetime_and_geometry_epochs():
    e = core.DateTime("2025-01-01T00:00:00")
    assert (core.DateTime("2025-01-01T00:00:10.25") - e).total_seconds() == 10.25
    assert core.DateTime(2025, 1, 1, 0, 0, 10.25) == core.DateTime("2025-01-01T00:00:10.250")
    orb = straight_orbit(epoch=e)
    from isce3_amd.container import RadarGeometry
    from isce3_amd.product import RadarGridParameters
    grid = RadarGridParameters(1.5, 0.24, 1000.0, 8e5, 5.0, "right", 10, 20,
                               core.DateTime("2025-01-01T00:00:02"))
    g = RadarGeometry(grid, orb, core.LUT2d())
    assert g.radar_grid.sensing_start == 3.5 and g.reference_epoch == e
    assert g.sensing_time[0] == 3.5 and g.slant_range[19] == 8e5 + 19 * 5.0
    assert g.look_side == core.LookSide.Right
    orb2 = orb.copy()
    orb2.update_reference_epoch(core.DateTime("2025-01-01T00:00:05"))
    assert orb2.start_time == orb.start_time - 5.0


def test_orbit_rejects_nonuniform_state_vectors():
    e = core.DateTime("2025-01-01T00:00:00")
    svs = [core.StateVector(e + core.TimeDelta(t), [7e6, 0, t], [0, 0, 1]) for t in (0, 10, 21, 30)]
    with pytest.raises(ValueError):
        core.Orbit(svs)


def test_scratch_bytes_match_the_server_accounting():
    """The tile server charges each worker the library's per-pixel scratch."""
    from isce3_amd import serve
    lib = _native.lib()
    assert lib.bp_scratch_bytes_per_pixel(_native.PRECISION_PLAIN) == \
        serve.RECORD_BYTES_PER_PIXEL["plain"]
    assert lib.bp_scratch_bytes_per_pixel(_native.PRECISION_SPLIT) == \
        serve.RECORD_BYTES_PER_PIXEL["split"]


@pytest.mark.parametrize("precision,width,max_pixels,least,most", [
    ("split", 8, 1 << 24, 1 << 30, (3 << 29) + (1 << 24)), ("split", 9, 1 << 16, 1 << 20, 156 * 700000),
    ("split", 6, 1 << 24, 0, 0), ("plain", 8, 1 << 24, 128 << 20, 256 << 20),
    ("plain", 8, 4096, 1, 16 << 20)])
def test_workspace_bytes(precision, width, max_pixels, least, most):
    """What a scene's sums hold beside its records, without and with a limit
    (2^16 pixels in 64 blocks: workspace for 156 strips)."""
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.focus import _PRECISION, geometry_struct
    grid = sim._grid(-2.5, sim.PRF, sim.R0, sim.DR, 8192, 16384)
    geometry = RadarGeometry(grid, sim.straight_orbit(), core.LUT2d())
    kernel = core.TabulatedKernelF32(core.KnabKernel(float(width), 0.8), 2048)
    ig, kr = geometry_struct(geometry), kernel._struct()

    def held(limit, scene=1):
        return _native.lib().bp_workspace_bytes(C.byref(ig), sim.FC, 6.0, C.byref(kr), 1,
                                                _PRECISION[precision], max_pixels, 64, scene, limit)

    assert least <= held(-1) <= most
    assert held(-1) <= held(-1, 0) <= (3 << 29) + (9 << 20)   # a context's calls of any shape
    assert held(10 << 20) <= max(10 << 20, (9 << 20) + (1 << 20))
    ig.doppler.have_data, ig.doppler.width = 1, 1      # refused as the calls refuse it
    assert held(-1) == _native.BP_ERR_INVALID_ARGUMENT
    ig.doppler.have_data = 0
    assert held(0) <= (9 << 20) + (1 << 20)     # 32 bytes a strip, and one strip


def _windowed_sinc(x, width, window):
    h = width / 2.0
    w = {"hann": 0.5 + 0.5 * np.cos(np.pi * x / h),
         "kaiser": np.i0(6.0 * np.sqrt(np.maximum(1 - (x / h) ** 2, 0))) / np.i0(6.0)}[window]
    return np.sinc(x) * w


@pytest.mark.parametrize("width", [8, 9])
@pytest.mark.parametrize("kind,taken", [
    (0.3, True), (0.6, True), (0.95, True), ("hann", True), ("kaiser", True),
    ("box", False), ("steps", False), ("noise", False), ("nan", False), ("triangle", False)])
def test_kernels_the_line_sum_takes(width, kind, taken):
    """Knab and windowed-sinc tables of 2048 entries are smooth enough for the
    weight polynomials (1e-4 of the peak, in the cell and past its ends); tables
    with steps, kinks in a tap's cell, noise or NaN keep the pixel-by-pixel sum."""
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.focus import geometry_struct
    geometry = RadarGeometry(sim._grid(-2.5, sim.PRF, sim.R0, sim.DR, 8192, 16384),
                             sim.straight_orbit(), core.LUT2d())
    n, h = 2048, width / 2.0
    x = h / (n - 1) * np.arange(n)
    if isinstance(kind, float):
        table = core.TabulatedKernelF32(core.KnabKernel(float(width), kind), n).table
    elif kind in ("hann", "kaiser"):
        table = _windowed_sinc(x, width, kind)
    else:
        table = {"box": np.ones(n), "steps": np.round(np.sinc(x) * 64) / 64,
                 "triangle": np.maximum(1 - np.abs(x - 0.1), 0),
                 "noise": np.random.default_rng(1).standard_normal(n),
                 "nan": np.where(np.arange(n) == 700, np.nan, np.sinc(x))}[kind]
        table[-1] = 0.0
    table = np.ascontiguousarray(table, np.float32)
    kr = _native.Kernel_t(h, n, 0, table.ctypes.data)
    ig = geometry_struct(geometry)
    held = _native.lib().bp_workspace_bytes(C.byref(ig), sim.FC, 6.0, C.byref(kr), 1,
                                            _native.PRECISION_SPLIT, 1 << 20, 64, 1, -1)
    assert (held > 0) == taken, held


@pytest.mark.parametrize("width", [8, 9])
def test_line_plan_host_time(width):
    """The plan of the line-interpolated sum, which every split call makes
    before its first launch (the kernel's weight polynomials above all), takes
    some 25 us; the least of 50 calls keeps below 100."""
    import time
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.focus import geometry_struct
    geometry = RadarGeometry(sim._grid(-2.5, sim.PRF, sim.R0, sim.DR, 8192, 16384),
                             sim.straight_orbit(), core.LUT2d())
    kernel = core.TabulatedKernelF32(core.KnabKernel(float(width), 0.8), 2048)
    ig, kr = geometry_struct(geometry), kernel._struct()
    times = []
    for _ in range(50):
        t0 = time.perf_counter()
        n = _native.lib().bp_workspace_bytes(C.byref(ig), sim.FC, 6.0, C.byref(kr), 1,
                                             _native.PRECISION_SPLIT, 1 << 20, 64, 1, -1)
        times.append(time.perf_counter() - t0)
    assert n > 0 and min(times) < 100e-6, min(times)


def test_sincos_turns_against_long_double():
    """The plain sum's FP64 phase rotation: sin/cos of 2 pi t for t in turns
    agree with an extended-precision evaluation to a few ulp, over the
    magnitudes fc * tau takes (about 7e6 turns at 850 km and L band) and
    across the quadrant boundaries of the reduction."""
    rng = np.random.Generator(np.random.PCG64(5))
    # the reduction rounds 4t to an integer with one FMA against 1.5 * 2^52,
    # valid for |t| < 2^49: up to that bound, including ties at odd eighths
    big = rng.uniform(2.0 ** 40, 2.0 ** 48, 400) * rng.choice([-1.0, 1.0], 400)
    ties = np.concatenate([2.0 ** 47 + np.arange(-16, 17) / 8.0, -(2.0 ** 46) + np.arange(9) / 8.0])
    t = np.concatenate([rng.uniform(-1, 1, 4000), rng.uniform(7.0e6, 7.3e6, 4000),
                        np.arange(-8, 9) / 8.0, np.arange(-8, 9) / 8.0 + 1e-12, big, ties,
                        np.array([0.0, 0.125, 0.375, 1e-300, -0.25 + 2 ** -40])])
    s = C.c_double()
    c = C.c_double()
    err = 0.0
    for ti in t:
        _native.lib().bp_sincos_turns(float(ti), C.byref(s), C.byref(c))
        # reference: reduce the exact double t in extended precision
        tl = np.longdouble(ti)
        frac = tl - np.rint(tl)
        ang = np.longdouble(2) * np.longdouble("3.14159265358979323846264338327950288") * frac
        err = max(err, abs(float(np.sin(ang)) - s.value), abs(float(np.cos(ang)) - c.value))
    assert err <= 4e-16
    # exact quadrant values
    for q, (es, ec) in enumerate([(0, 1), (1, 0), (0, -1), (-1, 0)]):
        _native.lib().bp_sincos_turns(q / 4.0, C.byref(s), C.byref(c))
        assert (s.value, c.value) == (es, ec) or (abs(s.value - es) < 1e-16 and abs(c.value - ec) < 1e-16)
