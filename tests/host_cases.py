"""Cases of tests/test_host_runtime.py, each run in a process of its own as
``python host_cases.py CASE``: the library's host code without a GPU."""
import ctypes
import sys

import hip_host
import numpy as np
import synth
from habitat_sim_amd import RendererConfiguration, RendererStandalone
from habitat_sim_amd import _native as N
from habitat_sim_amd import math3d as m3


def _triangle():
    pos = np.array([(-1, -1, -3), (1, -1, -3), (0, 1, -3)], np.float32)
    return synth.mesh_file([(pos, np.arange(3, dtype=np.uint32), None, None, 0)], [synth.flat((1, 1, 1, 1))])


def _scenes(tile, grid, nodes):
    r = RendererStandalone(RendererConfiguration().set_tile_size_count(tile, grid))
    assert r.add_file_data(_triangle())
    for s in range(grid[0] * grid[1]):
        for k in range(nodes):
            r.add_node_hierarchy(s, "m0", None, k + 1)
    return r


def _bins(function):
    """Calls function(list of RasterItem) at each launch of the lane rasteriser."""
    def launched(_, grid, args):
        items = ctypes.cast(args[1], ctypes.POINTER(ctypes.POINTER(hip_host.RasterItem))).contents
        function(items[:ctypes.cast(args[2], ctypes.POINTER(ctypes.c_uint32)).contents.value])
    hip_host.on_launch("k_raster_lane", None, launched)


def _soup(n):
    """n triangles, three vertices each."""
    pos = np.random.default_rng(n).uniform(-1.0, 1.0, (3 * n, 3)).astype(np.float32)
    return synth.mesh_file([(pos, np.arange(3 * n, dtype=np.uint32), None, None, 0)], [synth.flat((1, 1, 1, 1))])


def moved_nodes_of_a_failed_frame():
    """A frame that ends at an allocation leaves nothing of its moved nodes to
    the next one, whose scenes may have lost them: that one sends everything."""
    moved = []
    hip_host.on_launch("k_inputs", hip_host.InputArgs, lambda a, grid, args: moved.append(
        {a.nodes[i]: list(a.transforms[16 * i:16 * i + 16]) for i in range(a.n_nodes)}))
    r = _scenes((32, 32), (3, 1), 3000)
    r.draw()
    assert moved.pop() == {}
    # more moved nodes than the pinned block has room for: it is allocated again
    for s in range(3):
        r.transformations(s)._a[:] = m3.translation((0.0, 0.0, -1.0 - s))
    hip_host.fail("hipHostMalloc")
    try:
        r.draw()
        raise AssertionError("the frame did not fail")
    except N.GbrError as e:
        assert e.status == N.ERR_OOM, e
    assert not moved
    r.clear(1)
    r.clear(2)
    r.draw()
    assert moved.pop() == {}, "nodes of the failed frame were sent again"
    # and later frames send what moves in them
    t = m3.translation((1.0, 2.0, 3.0))
    r.transformations(0)[5] = t
    r.draw()
    sent = moved.pop()
    assert list(sent) == [5] and np.array_equal(np.float32(sent[5]), np.asarray(t, np.float32).reshape(-1)), sent
    r.close()


def redwood_stays_inside_wide_images():
    """The last row and column that k_redwood clamps to lie inside the image at
    every size: as floats, sides beyond 2^24 pixels may round up."""
    seen = []
    hip_host.on_launch("k_redwood", hip_host.RedwoodArgs,
                       lambda a, grid, args: seen.append((a.npx, a.W, int(a.xmax), int(a.ymax))))
    h = ctypes.c_void_p()
    table = np.ones(N.REDWOOD_MODEL_FLOATS, np.float32)
    N.call("gbr_redwood_create", table.ctypes.data, 0, 1.0, 1, ctypes.byref(h))
    image = ctypes.c_void_p(1 << 20)  # never read: kernels do not run
    sides = [2, 3, 640, (1 << 23) - 1, 1 << 23, (1 << 23) + 2, (1 << 24) - 1, 1 << 24, (1 << 24) + 1, (1 << 24) + 2,
             16777220, 33554437, (1 << 29) - 3]
    for side in sides:
        for rows, cols in ((3, side), (side, 3)):
            N.call("gbr_redwood_simulate", h, image, 1, rows, cols, image, None)
            npx, w, xmax, ymax = seen.pop()
            assert (npx, w) == (rows * cols, cols)
            for last, n in ((xmax, cols), (ymax, rows)):
                f = np.float32(n - 1)
                assert last <= n - 1, f"{rows} x {cols}: clamped to {last}"
                assert last == int(f if int(f) <= n - 1 else np.nextafter(f, np.float32(0))), (last, n)
    N.call("gbr_redwood_destroy", h)


def bin_capacity_follows_the_factor():
    """Below 2 a bin holds the factor's share of its scene's triangles and no
    more; from 2 (the default) on it holds more, and more with each factor."""
    bins = []
    _bins(bins.append)
    n = 40000  # 16 bins of 2500 triangles on average
    r = RendererStandalone(RendererConfiguration().set_tile_size_count((128, 128), (1, 1)))
    assert r.add_file_data(_soup(n))
    r.add_node_hierarchy(0, "m0", None, 1)
    assert r.tuning().bin_capacity_factor == 2.0
    caps = {}
    for factor in (0.25, 0.5, 1.0, 1.25, 1.5, 1.9, 2.0, 2.5, 3.0, 6.0):
        r.set_tuning(bin_capacity_factor=factor, graph=0)
        r.draw()
        (cap,) = {b.bin_cap for b in bins[-1]}
        assert len(bins[-1]) == 16 and all(b.entries == i * cap for i, b in enumerate(bins[-1]))
        caps[factor] = cap
        if factor < 2.0:
            share = int(n / 16 * np.float32(factor))
            assert share <= cap < share + 64, (factor, cap)
    assert sorted(set(caps.values())) == list(caps.values()), caps
    r.close()


def closed_objects_free_their_memory():
    """Device and pinned memory is all given back by close()."""
    def renderer(tuning, lights):
        cfg = RendererConfiguration().set_tile_size_count((64, 48), (2, 1)).set_max_light_count(lights)
        r = RendererStandalone(cfg)
        assert r.add_file_data(_triangle())
        for s in range(2):
            r.add_node_hierarchy(s, "m0", None, 1)
        if lights:
            r.add_light(0, 0, N.LIGHT_POINT)
        r.vis_init(1)
        r.set_tuning(**tuning)
        for _ in range(2):
            r.draw()
        r.vis_collect()
        r.color_image()
        r.depth_image()
        r.color_image_into((0, 0, 8, 8), np.zeros((8, 8, 3), np.uint8))
        r.vis_loss_grad(np.zeros((32, N.VIS_FEATURES), np.float32), np.zeros(32, np.uint8))
        r.close()

    for tuning in (dict(), dict(cull_mode=N.CULL_HIZ), dict(cull_mode=N.CULL_LEARNED, raster_mode=1),
                   dict(timing=1, graph=0)):
        for lights in (0, 2):
            renderer(tuning, lights)
            assert hip_host.memory_blocks() == 0, (tuning, lights, hip_host.memory_blocks())
    h = ctypes.c_void_p()
    table = np.ones(N.REDWOOD_MODEL_FLOATS, np.float32)
    N.call("gbr_redwood_create", table.ctypes.data, 0, 1.0, 1, ctypes.byref(h))
    depth = np.ones((4, 6), np.float32)
    N.call("gbr_redwood_simulate_host", h, depth.ctypes.data, 4, 6, depth.ctypes.data)
    N.call("gbr_redwood_destroy", h)
    assert hip_host.memory_blocks() == 0


def wide_bins_give_way_to_memory():
    """Where the wide entry list does not fit a quarter of the free memory, bins
    get the factor's share: a scene that fits with that is drawn."""
    bins = []
    _bins(bins.append)

    def draw():
        r = RendererStandalone(RendererConfiguration().set_tile_size_count((128, 128), (4, 2)))
        assert r.add_file_data(_soup(40000))
        for s in range(8):
            r.add_node_hierarchy(s, "m0", None, 1)
        r.draw()
        used = hip_host.device_memory_used()
        (cap,) = {b.bin_cap for b in bins[-1]}
        assert all(b.entries == i * cap for i, b in enumerate(bins[-1]))
        r.draw()
        r.close()
        return cap, used

    wide, used = draw()
    assert wide == 10048
    # 128 bins of 10048 or 5056 entries of 4 bytes, with half as much room again
    hip_host.device_memory(used - (2 << 20))
    cap, less = draw()
    assert cap == 5056 and less == used - 6 * 128 * (10048 - 5056), (cap, used - less)


def _pinned(shape):
    p = ctypes.c_void_p()
    hip_host.runtime().hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(int(np.prod(shape))), ctypes.c_uint(0))
    return np.frombuffer((ctypes.c_uint8 * int(np.prod(shape))).from_address(p.value), np.uint8).reshape(shape)


def readback_by_destination():
    """An image read into memory that HIP knows (pinned, managed) is one 2D copy
    by the device, without a second copy by the host, unless it is small;
    pageable memory gets its rows from the renderer's pinned staging."""
    r = _scenes((512, 512), (2, 1), 1)
    r.draw()
    page, pin = np.zeros((512, 1024, 4), np.uint8), _pinned((512, 1024, 4))
    rgb, pin_rgb = np.zeros((512, 1024, 3), np.uint8), _pinned((512, 1024, 3))
    for image, w, h, copies in ((page, 1024, 512, 0), (rgb, 1024, 512, 0), (pin, 1024, 512, 1), (pin, 700, 511, 1),
                                (pin_rgb, 1024, 512, 1), (pin, 128, 128, 0), (pin_rgb, 64, 64, 0), (pin_rgb, 128, 128, 1)):
        before = hip_host.calls("hipMemcpy2DAsync")
        r.color_image_into((0, 0, w, h), image[:h, :w])
        assert hip_host.calls("hipMemcpy2DAsync") - before == copies, (image.shape, w, h)
    # (kernels do not run: the copied rows are those of fresh, zeroed device memory)
    pin[:] = 7
    r.color_image_into((0, 0, 700, 511), pin[:511, 300:1000])
    assert not pin[:511, 300:1000].any() and (pin[:511, :300] == 7).all() and (pin[511:] == 7).all()
    assert (pin[:, 1000:] == 7).all()
    r.close()


def more_moved_nodes_every_frame():
    """A program that moves a few more nodes each frame makes the pinned blocks
    grow now and then, not every frame; every moved node is sent."""
    moved = []
    hip_host.on_launch("k_inputs", hip_host.InputArgs, lambda a, grid, args: moved.append(
        [(a.nodes[i], a.transforms[16 * i + 12]) for i in range(a.n_nodes)]))
    r = _scenes((32, 32), (3, 1), 3000)  # 6000 nodes each
    r.draw()
    blocks = []
    for frame, n in enumerate(list(range(4000, 4400)) + list(range(17700, 18000, 50)) + [18000]):
        left = n
        for s in range(3):
            m = min(left, 6000)
            r.transformations(s)._a[:m, 3, 0] = frame + 1.0
            left -= m
        before = hip_host.calls("hipHostMalloc")
        r.draw()
        if hip_host.calls("hipHostMalloc") != before:
            blocks.append(n)
        sent = moved.pop()
        assert sent == [(k, frame + 1.0) for k in range(n)], (frame, n)
    assert len(blocks) <= 5, blocks
    r.close()


def input_blocks_are_waited_for():
    """Draws alternate between three pinned input blocks, and one is written
    again only after the event behind the kernel that last read it."""
    pending = {}  # block -> its event, recorded and not yet waited for
    used = []     # the block of each launch
    early = []    # launches whose block was still in use

    def call(name, grid, args):
        if "k_inputs" in name:
            src = hip_host.InputArgs.from_address(args[0]).src
            if src in pending:  # (an exception would end here, in the runtime's call)
                early.append(len(used))
            used.append(src)
            pending[src] = None
        elif name == "hipEventRecord" and used and pending.get(used[-1], 0) is None:
            pending[used[-1]] = args[0]
        elif name == "hipEventSynchronize":
            for src in [s for s, e in pending.items() if e == args[0]]:
                del pending[src]

    r = _scenes((32, 32), (2, 1), 40)
    hip_host.on_call(call)
    for frame in range(10):
        r.transformations(frame % 2)._a[frame, 3, 0] = frame + 1.0
        r.draw()
    assert not early, f"frames {early} wrote blocks that were not waited for"
    assert len(used) == 10 and len(set(used)) == 3 and all(a == b for a, b in zip(used, used[3:]))
    assert len(pending) == 3 and None not in pending.values()
    r.close()


if __name__ == "__main__":
    globals()[sys.argv[1]]()
    print("case passed:", sys.argv[1])
