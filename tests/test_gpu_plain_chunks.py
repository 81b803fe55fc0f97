"""The plain sum's chunks of 64 pulses (delay by a cubic, phasor by recurrence)
against the oracle: raw sets shorter than a chunk, at its multiples and
off them, windows that begin and end inside chunks, and low short-range
tracks where the cubic fits all, none or some of the pixels.

Tolerance: weights and products in FP32, up to 9 taps of 6e-8 each in weight, product
and sum, add as random errors to at most 3e-7 of a pixel; a cubic within 1e-9
cycles (6e-9 rad) or 8 ulp of the phase (4e-8 rad at 850 km) and a phasor within
2e-8 are below that: 5e-7."""
import numpy as np
import pytest

import oracle
from helpers import complex_rel_error

pytestmark = pytest.mark.gpu


def _check(na, ds, rows=21, cols=35, altitude=None, speed=None, prf=None, r0=None, width=8):
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import KnabKernel, LUT2d, Orbit, TabulatedKernelF32
    from isce3_amd.focus import backproject
    from isce3_amd.geometry import DEMInterpolator
    prf, r0, nr = prf or sim.PRF, r0 or sim.R0, 96
    orb = sim.straight_orbit()
    if altitude:
        t = -50.0 + 10.0 * np.arange(11)
        pos = np.stack([0 * t + sim.WGS84_A + altitude, 0 * t, speed * t], axis=1)
        orb = Orbit.from_arrays(sim.EPOCH, -50.0, 10.0, pos,
                                np.repeat([[0.0, 0.0, speed]], len(t), axis=0))
    in_grid = sim._grid(-0.5 * na / prf, prf, r0, sim.DR, na, nr)
    in_geom = RadarGeometry(in_grid, orb, LUT2d())
    grid = sim._grid(-0.5 * rows / prf, prf, r0 + 12.3 * sim.DR, sim.DR, rows, cols)
    og = RadarGeometry(grid, orb, LUT2d())
    rng = np.random.default_rng(na)
    raw = (rng.standard_normal((na, nr)) + 1j * rng.standard_normal((na, nr))).astype(np.complex64)
    kernel = TabulatedKernelF32(KnabKernel(float(width), 0.8), 2048)
    dem = DEMInterpolator(50.0)
    out = np.empty(grid.shape, np.complex64)
    backproject(out, og, raw, in_geom, dem, sim.FC, ds, kernel, "nodelay", precision="plain")
    ref, _, _, _ = oracle.backproject(og, raw, in_geom, dem, sim.FC, ds, kernel, "nodelay", mode=0)
    assert (np.isnan(out) == np.isnan(ref)).all()
    rel = complex_rel_error(out, ref)
    print(f"[plain chunks] na={na} ds={ds} rel={rel:.2e}", flush=True)
    assert rel <= 5e-7


@pytest.mark.parametrize("width", [8, 9])
@pytest.mark.parametrize("na", [1, 63, 64, 65, 200, 256])
def test_every_pulse(torch_gpu, na, width):
    _check(na, 6.0, width=width)


@pytest.mark.parametrize("na", [300, 321])
def test_windows_inside_chunks(torch_gpu, na):
    _check(na, 200.0)


@pytest.mark.parametrize("prf", [100.0, 700.0, 3000.0])
def test_short_ranges(torch_gpu, prf):
    _check(330, 6.0, altitude=3000.0, speed=120.0, prf=prf, r0=5000.0)


def test_segments_and_whole_windows_agree(torch_gpu):
    """A grid of more wavefronts than get segments of their own, and its first
    rows alone, which are summed by segments: the same to the bit."""
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import KnabKernel, LUT2d, TabulatedKernelF32
    from isce3_amd.focus import backproject
    from isce3_amd.geometry import DEMInterpolator
    na, nr, rows, cols = 1500, 1060, 1040, 1030
    orb = sim.straight_orbit()
    in_grid = sim._grid(-0.5 * na / sim.PRF, sim.PRF, sim.R0, sim.DR, na, nr)
    rng = np.random.default_rng(1)
    raw = (rng.standard_normal((na, nr)) + 1j * rng.standard_normal((na, nr))).astype(np.complex64)
    kernel = TabulatedKernelF32(KnabKernel(8.0, 0.8), 2048)
    outs = []
    for n in (rows, 33):
        grid = sim._grid(-0.5 * rows / sim.PRF, sim.PRF, sim.R0 + 12 * sim.DR, sim.DR, n, cols)
        out = np.empty(grid.shape, np.complex64)
        backproject(out, RadarGeometry(grid, orb, LUT2d()), raw, RadarGeometry(in_grid, orb, LUT2d()),
                    DEMInterpolator(50.0), sim.FC, 40.0, kernel, "nodelay", precision="plain")
        outs.append(out)
    np.testing.assert_array_equal(outs[0][:33], outs[1])


def test_chunk_phase_against_single_delays(torch_gpu):
    """63 pulses as the first of a whole chunk (delays by the cubic, the pulses
    behind them zero) and as a chunk that the data's end cuts off (a delay per
    pulse), at a wavelength of 2.4 mm: 7e8 cycles, so that FP64 rounding shows.
    What is left between the two is the rounding of a delay per pulse, five
    roundings of half an ulp of 7e8 cycles (7.5e-7 rad each at most, 2.2e-7 RMS):
    4.8e-7; the cubic of delays in two words adds less than 2e-7 to it, rounded
    delays at its nodes would add as much again (6.6e-7 was measured)."""
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import KnabKernel, LUT2d, TabulatedKernelF32
    from isce3_amd.focus import backproject
    from isce3_amd.geometry import DEMInterpolator
    nr, rows, cols = 96, 40, 40
    orb = sim.straight_orbit()
    og = RadarGeometry(sim._grid(-0.5 * rows / sim.PRF, sim.PRF, sim.R0 + 12.3 * sim.DR, sim.DR,
                                 rows, cols), orb, LUT2d())
    rng = np.random.default_rng(2)
    raw = np.zeros((127, nr), np.complex64)
    raw[:63] = rng.standard_normal((63, nr)) + 1j * rng.standard_normal((63, nr))
    outs = []
    for na in (127, 63):
        ig = RadarGeometry(sim._grid(-32 / sim.PRF, sim.PRF, sim.R0, sim.DR, na, nr), orb, LUT2d())
        out = np.empty((rows, cols), np.complex64)
        backproject(out, og, raw[:na], ig, DEMInterpolator(50.0), 100 * sim.FC, 0.01,
                    TabulatedKernelF32(KnabKernel(8.0, 0.8), 2048), "nodelay", precision="plain")
        outs.append(out.astype(complex))
    rel = np.linalg.norm(outs[0] - outs[1]) / np.linalg.norm(outs[1])
    print(f"[plain chunks] cubic and single delays differ by {rel:.2e}", flush=True)
    assert rel <= 5.2e-7


def test_short_range_low_prf_costs_no_more_than_delays(torch_gpu):
    """Where no chunk keeps the cubic's tolerance, updates take the time of an
    evaluated delay each, 1.19 of one by the cubic (measured at 1200 x 1200 pixels;
    1.48 when every chunk tries its nodes first), alone and in a scene's graph."""
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import KnabKernel, LUT2d, Orbit, TabulatedKernelF32
    from isce3_amd.focus import Scene, backproject
    from isce3_amd.geometry import DEMInterpolator
    t = -50.0 + 10.0 * np.arange(11)
    pos = np.stack([0 * t + sim.WGS84_A + 3000.0, 0 * t, 120.0 * t], axis=1)
    orb = Orbit.from_arrays(sim.EPOCH, -50.0, 10.0, pos, np.repeat([[0.0, 0.0, 120.0]], 11, axis=0))
    na, n = 1000, 1100
    raw = torch_gpu.ones((na, n + 100), dtype=torch_gpu.complex64, device="cuda:0")
    out = torch_gpu.empty((n, n), dtype=torch_gpu.complex64, device="cuda:0")
    kernel, rate = TabulatedKernelF32(KnabKernel(8.0, 0.8), 2048), []
    for prf in (200.0, 3000.0):
        ig = RadarGeometry(sim._grid(-0.5 * na / prf, prf, 5000.0, sim.DR, na, n + 100), orb, LUT2d())
        og = RadarGeometry(sim._grid(-0.5 * n / prf, prf, 5300.0, sim.DR, n, n), orb, LUT2d())
        best, st = np.inf, {}
        for _ in range(4):
            backproject(out, og, raw, ig, DEMInterpolator(50.0), sim.FC, 0.1, kernel, "nodelay",
                        precision="plain", stats=st)
            best = min(best, st["sum_ms"] / st["updates"])
        rate.append(best)
        part = og.radar_grid.offset_and_resize(100, 200, 33, 65)
        tile = torch_gpu.empty((33, 65), dtype=torch_gpu.complex64, device="cuda:0")
        want = torch_gpu.empty_like(tile)
        backproject(want, RadarGeometry(part, orb, LUT2d()), raw, ig, DEMInterpolator(50.0), sim.FC,
                    0.1, kernel, "nodelay", precision="plain")
        with Scene(raw, ig, orb, LUT2d(), DEMInterpolator(50.0), sim.FC, 0.1, kernel, "nodelay",
                   precision="plain", max_pixels=1 << 12, max_blocks=1) as scene:
            for _ in range(2):
                scene.focus([tile], [part])
                np.testing.assert_array_equal(tile.cpu().numpy(), want.cpu().numpy())
    print(f"[plain chunks] time per update, single delays over cubic: {rate[0] / rate[1]:.2f}",
          flush=True)
    assert rate[0] <= 1.33 * rate[1]
