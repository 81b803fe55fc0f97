"""Resident scenes (bp_scene_*): the step replayed from a captured HIP graph
gives every block the result of bp_backproject_blocks bit for bit, on every
replay, with eager work and synchronisations between the replays, for
batches of different sizes and launch options, and rejects requests beyond
its reserved scratch."""
import numpy as np
import pytest

from helpers import scene_and_raw
from test_gpu_blocks import uneven_blocks

pytestmark = pytest.mark.gpu


def eager(sc, raw_dev, grids, precision, opts):
    import torch
    from isce3_amd.focus import backproject_blocks
    outs = [torch.full(tuple(b.shape), 5 + 5j, dtype=torch.complex64, device="cuda:0")
            for b in grids]
    hs = [torch.zeros(tuple(b.shape), dtype=torch.float32, device="cuda:0") for b in grids]
    st = {}
    flags = backproject_blocks(outs, [sc.out_geometry(b) for b in grids], raw_dev,
                               sc.in_geometry(), sc.dem, sc.fc, sc.ds, sc.kernel,
                               sc.dry_tropo_model, heights=hs, precision=precision,
                               options=opts, stats=st)
    return [o.cpu().numpy() for o in outs], [h.cpu().numpy() for h in hs], flags, st


def replay(scene, grids, opts, heights=True):
    import torch
    outs = [torch.full(tuple(b.shape), -1 - 1j, dtype=torch.complex64, device="cuda:0")
            for b in grids]
    hs = [torch.zeros(tuple(b.shape), dtype=torch.float32, device="cuda:0") for b in grids] \
        if heights else None
    st = {}
    flags = scene.focus(outs, grids, hs, options=opts, stats=st)
    return ([o.cpu().numpy() for o in outs], [h.cpu().numpy() for h in hs] if heights else None,
            flags, st)


@pytest.mark.parametrize("precision", ["plain", "split"])
def test_graph_replays_equal_eager_calls(torch_gpu, precision):
    from isce3_amd.focus import Scene
    torch = torch_gpu
    sc, raw = scene_and_raw("small")
    raw_dev = torch.from_numpy(raw.copy()).cuda()
    grids = uneven_blocks(sc)
    opts = {"tile_rows": 2}
    ref = eager(sc, raw_dev, grids, precision, opts)
    with Scene(raw_dev, sc.in_geometry(), sc.orbit, sc.doppler, sc.dem, sc.fc, sc.ds,
               sc.kernel, sc.dry_tropo_model, precision=precision, max_pixels=1 << 16,
               max_blocks=16) as scene:
        for rep in range(3):
            print(f"[scene] precision={precision} replay={rep}", flush=True)
            outs, hs, flags, st = replay(scene, grids, opts)
            for z, z0, h, h0 in zip(outs, ref[0], hs, ref[1]):
                np.testing.assert_array_equal(z, z0)
                np.testing.assert_array_equal(h, h0)
            assert flags == ref[2]
            assert st["updates"] == ref[3]["updates"]
            # eager work and a synchronisation between replays
            eager(sc, raw_dev, grids[:2], precision, opts)
            torch.cuda.synchronize()
        # a smaller batch replays the same graph with new counts
        sub = [grids[3], grids[0]]
        ref_sub = eager(sc, raw_dev, sub, precision, opts)
        outs, _, flags, _ = replay(scene, sub, opts, heights=False)
        for z, z0 in zip(outs, ref_sub[0]):
            np.testing.assert_array_equal(z, z0)


def test_new_launch_options_capture_a_new_graph(torch_gpu):
    from isce3_amd.focus import Scene
    torch = torch_gpu
    sc, raw = scene_and_raw("tiny")
    raw_dev = torch.from_numpy(raw.copy()).cuda()
    grids = [sc.out_grid]
    with Scene(raw_dev, sc.in_geometry(), sc.orbit, sc.doppler, sc.dem, sc.fc, sc.ds,
               sc.kernel, sc.dry_tropo_model, precision="split", max_pixels=1 << 14,
               max_blocks=4) as scene:
        for opts in ({"tile_rows": 1}, {"tile_rows": 8, "chunk": 16, "staged": 1},
                     {"tile_rows": 4, "blocks_per_cu": 1}, {"tile_rows": 2, "lane_rows": 2},
                     {"tile_rows": 1}):
            print(f"[scene] options={opts}", flush=True)
            ref = eager(sc, raw_dev, grids, "split", opts)
            outs, _, _, _ = replay(scene, grids, opts, heights=False)
            np.testing.assert_array_equal(outs[0], ref[0][0])


def test_scene_limits(torch_gpu):
    from isce3_amd import errors
    from isce3_amd.focus import Scene
    torch = torch_gpu
    sc, raw = scene_and_raw("tiny")
    raw_dev = torch.from_numpy(raw.copy()).cuda()
    g = sc.out_grid
    with Scene(raw_dev, sc.in_geometry(), sc.orbit, sc.doppler, sc.dem, sc.fc, sc.ds,
               sc.kernel, sc.dry_tropo_model, precision="split", max_pixels=g.length * g.width - 1,
               max_blocks=1) as scene:
        out = torch.empty(tuple(g.shape), dtype=torch.complex64, device="cuda:0")
        with pytest.raises(errors.InvalidArgument):
            scene.focus([out], [g])
        small = g.offset_and_resize(0, 0, 4, 4)
        o1 = torch.empty((4, 4), dtype=torch.complex64, device="cuda:0")
        o2 = torch.empty((4, 4), dtype=torch.complex64, device="cuda:0")
        with pytest.raises(errors.InvalidArgument):
            scene.focus([o1, o2], [small, small])  # two blocks, one reserved
        assert scene.focus([o1], [small]) == [False]


def test_strip_counts_without_allocation(torch_gpu):
    """Replays of 40 strips, of one, of 640 narrow ones (more than the scene has
    workspace for at a time: several groups in the graph) and of 40 again: the
    eager results, and no device memory beyond a graph's own."""
    from isce3_amd import sim
    from isce3_amd.focus import Scene
    torch = torch_gpu
    sc = sim.make_scene("tiny")
    na, nr = 1600, 2700
    sc.in_grid = sim._grid(-0.5 * na / sim.PRF, sim.PRF, sim.R0, sim.DR, na, nr)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(4)
    raw_dev = torch.randn((na, nr), dtype=torch.complex64, device="cuda:0", generator=gen)

    def block(rows, cols, c0):
        return sim._grid(-0.5 * rows / sim.PRF, sim.PRF, sim.R0 + c0 * sim.DR, sim.DR, rows, cols)

    batches = [[block(64, 40 * 64, 40)], [block(20, 33, 40)],
               [block(1024, 1, 40 + 9 * i) for i in range(40)], [block(64, 40 * 64, 40)]]
    with Scene(raw_dev, sc.in_geometry(), sc.orbit, sc.doppler, sc.dem, sc.fc, sc.ds, sc.kernel,
               sc.dry_tropo_model, precision="split", max_pixels=40 * 4096, max_blocks=64) as scene:
        refs = [eager(sc, raw_dev, b, "split", {}) for b in batches]
        replay(scene, batches[1], {})
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info(0)[0]
        for b, ref in zip(batches, refs):
            print(f"[scene] {len(b)} blocks of {b[0].length} x {b[0].width}", flush=True)
            outs, _, _, st = replay(scene, b, {}, heights=False)
            for z, z0 in zip(outs, ref[0]):
                np.testing.assert_array_equal(z, z0)
            assert st["updates"] == ref[3]["updates"]
        taken = free - torch.cuda.mem_get_info(0)[0]
        print(f"[scene] {taken / 2 ** 20:.1f} MiB taken", flush=True)
        assert taken <= 16 << 20


def test_strips_left_beside_others(torch_gpu):
    """Blocks at the swath's edge, where some strips are left to the pixel-by-pixel
    sum: replayed, and launched beside the others once the scene has met such strips;
    then blocks without any, all as eager."""
    from isce3_amd import sim
    from isce3_amd.focus import Scene
    torch = torch_gpu
    sc = sim.make_scene("tiny")
    na, nr = 1600, 400
    sc.in_grid = sim._grid(-0.5 * na / sim.PRF, sim.PRF, sim.R0, sim.DR, na, nr)
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(6)
    raw_dev = torch.randn((na, nr), dtype=torch.complex64, device="cuda:0", generator=gen)

    def block(rows, cols, c0, dr=1.0):
        return sim._grid(-0.5 * rows / sim.PRF, sim.PRF, sim.R0 + c0 * sim.DR, dr * sim.DR, rows, cols)

    edge = [block(100, 170, -20), block(33, 64, 100), block(40, 50, 150, 0.7)]
    inside = [block(70, 100, 100)]
    with Scene(raw_dev, sc.in_geometry(), sc.orbit, sc.doppler, sc.dem, sc.fc, sc.ds, sc.kernel,
               sc.dry_tropo_model, precision="split", max_pixels=1 << 15, max_blocks=4) as scene:
        for b in (edge, edge, edge, inside, inside, edge):
            ref = eager(sc, raw_dev, b, "split", {})
            outs, _, _, st = replay(scene, b, {}, heights=False)
            for z, z0 in zip(outs, ref[0]):
                np.testing.assert_array_equal(z, z0)
            assert st["updates"] == ref[3]["updates"]


@pytest.mark.parametrize("precision,limit", [("split", -1), ("split", 20 << 20), ("plain", -1)])
def test_memory_held_as_stated(torch_gpu, precision, limit):
    """A scene takes at most its per-pixel scratch and bp_workspace_bytes (and
    some MiB of tables and allocation granules), and a limit does not change
    results."""
    import ctypes as C
    from isce3_amd import _native
    from isce3_amd.focus import _PRECISION, Scene, geometry_struct
    torch = torch_gpu
    sc, raw = scene_and_raw("small")
    raw_dev = torch.from_numpy(raw.copy()).cuda()
    grids = uneven_blocks(sc)
    ref = eager(sc, raw_dev, grids, precision, {})
    ctx = C.c_void_p()
    lib = _native.lib()
    _native.check(lib.bp_context_create(0, C.byref(ctx)))
    _native.check(lib.bp_context_limit_workspace(ctx, limit))
    max_pixels = 1 << 20
    geometry = sc.in_geometry()
    ig, kr = geometry_struct(geometry), sc.kernel._struct()
    said = max_pixels * lib.bp_scratch_bytes_per_pixel(_PRECISION[precision]) + \
        lib.bp_workspace_bytes(C.byref(ig), sc.fc, sc.ds, C.byref(kr), 1, _PRECISION[precision],
                               max_pixels, 16, 1, limit)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info(0)[0]
    with Scene(raw_dev, sc.in_geometry(), sc.orbit, sc.doppler, sc.dem, sc.fc, sc.ds, sc.kernel,
               sc.dry_tropo_model, precision=precision, max_pixels=max_pixels, max_blocks=16,
               _context=ctx) as scene:
        taken = free - torch.cuda.mem_get_info(0)[0]
        print(f"[scene] {precision} limit {limit}: {taken / 2 ** 20:.1f} MiB, stated "
              f"{said / 2 ** 20:.1f}", flush=True)
        assert taken <= said + (24 << 20)
        outs = replay(scene, grids, {}, heights=False)[0]
        for z, z0 in zip(outs, ref[0]):
            np.testing.assert_array_equal(z, z0)
    lib.bp_context_destroy(ctx)
