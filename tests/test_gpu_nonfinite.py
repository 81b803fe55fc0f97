"""Samples that are not finite among the pulses of a line-interpolated strip.

A NaN or an infinity reaches the pixels whose taps hold it and, as lines 2i
and 2i + 1 share one gather of a bin more than the taps in the pixel-by-pixel
sum, their partners and the pixels whose last tap lies one bin below it; no
other pixel of the strip, whose lines otherwise share sums.  Which pixels hold a
sample is the oracle's answer; the rest keep the pixel-by-pixel sum's
accuracy (2e-4, its weight table on white pulses)."""
import numpy as np
import pytest

import oracle
from helpers import complex_rel_error

pytestmark = pytest.mark.gpu

NA, NR, ROWS, COLS, C0 = 4600, 192, 128, 24, 60


def _scene():
    from isce3_amd import sim
    from isce3_amd.container import RadarGeometry
    from isce3_amd.core import KnabKernel, LUT2d, TabulatedKernelF32
    from isce3_amd.geometry import DEMInterpolator
    orb = sim.straight_orbit()
    in_grid = sim._grid(-0.5 * NA / sim.PRF, sim.PRF, sim.R0, sim.DR, NA, NR)
    grid = sim._grid(-0.5 * ROWS / sim.PRF + 0.3 / sim.PRF, sim.PRF, sim.R0 + (C0 + 0.37) * sim.DR,
                     sim.DR, ROWS, COLS)
    rng = np.random.default_rng(5)
    raw = (rng.standard_normal((NA, NR)) + 1j * rng.standard_normal((NA, NR))).astype(np.complex64)
    return (RadarGeometry(grid, orb, LUT2d()), RadarGeometry(in_grid, orb, LUT2d()),
            DEMInterpolator(50.0), raw, TabulatedKernelF32(KnabKernel(8.0, 0.8), 2048))


def _focus(sc, raw, window=0, stats=None):
    from isce3_amd import sim
    from isce3_amd.focus import backproject
    og, ig, dem, _, kernel = sc
    out = np.empty((ROWS, COLS), np.complex64)
    backproject(out, og, raw, ig, dem, sim.FC, 6.0, kernel, "nodelay", precision="split",
                max_window_bytes=window, stats=stats)
    return out


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("k", [700, 1100, 3500, 3900])
def test_reaches_the_pixels_that_hold_it(torch_gpu, k, value):
    from isce3_amd import sim
    sc = _scene()
    og, ig, dem, raw, kernel = sc
    held = []
    for b in (79, 80):
        z = raw.copy()
        z[k, b] = value
        ref = oracle.backproject(og, z, ig, dem, sim.FC, 6.0, kernel, "nodelay", mode=1,
                                 kernel_bandwidth=0.8)[0]
        held.append(~np.isfinite(ref))
    below, held = held
    # the sample has entered some lines' taps and not others' of a column
    assert any(0 < held[r:r + 64, c].sum() < 64 for r in (0, 64) for c in range(COLS))
    partner = held.reshape(ROWS // 2, 2, COLS)[:, ::-1].reshape(ROWS, COLS)
    allowed = held | partner | below
    out = _focus(sc, z)
    bad = ~np.isfinite(out)
    print(f"[nonfinite] pulse {k} {value}: held {held.sum()}, out {bad.sum()}", flush=True)
    assert (bad | ~held).all() and (allowed | ~bad).all()
    assert complex_rel_error(out[~allowed], ref[~allowed]) <= 2e-4


def test_host_pulses_in_parts(torch_gpu):
    """Under a budget below a strip's window the sample's strip is done again
    from bands of tile rows, as with the pulses on the device."""
    sc = _scene()
    raw = sc[3].copy()
    st = {}
    whole = _focus(sc, raw, stats=st)
    raw[1100, 80] = np.nan
    budget = (st["window_pulses"] - ROWS + 64 - 40) * NR * 8
    part_st = {}
    got = _focus(sc, raw, budget, part_st)
    assert part_st["bands"] > 2
    np.testing.assert_array_equal(got, _focus(sc, raw))
    assert np.isnan(got).any() and np.isfinite(whole).all()


def test_scene_replays(torch_gpu):
    """In a scene's graph and in batches, as in a call of its own."""
    from isce3_amd import sim
    from isce3_amd.focus import Scene, backproject_blocks
    sc = _scene()
    og, ig, dem, raw, kernel = sc
    raw = raw.copy()
    raw[700, 80] = np.inf
    d_raw = torch_gpu.from_numpy(raw).to("cuda:0")
    want = _focus(sc, raw)
    outs = [torch_gpu.empty((ROWS, COLS), dtype=torch_gpu.complex64, device="cuda:0")
            for _ in range(2)]
    backproject_blocks(outs, [og, og], d_raw, ig, dem, sim.FC, 6.0, kernel, "nodelay",
                       precision="split")
    for o in outs:
        np.testing.assert_array_equal(o.cpu().numpy(), want)
    with Scene(d_raw, ig, og.orbit, og.doppler, dem, sim.FC, 6.0, kernel, "nodelay",
               precision="split", max_pixels=ROWS * COLS, max_blocks=1) as scene:
        for _ in range(3):
            outs[0].zero_()
            scene.focus(outs[:1], [og.radar_grid])
            np.testing.assert_array_equal(outs[0].cpu().numpy(), want)
