"""The rasteriser, clipper, texture sampler, frame inputs and readback at the
sizes where their work is split, bit for bit against the oracle: triangles from
a fraction of a pixel to beyond the guard band, workgroups' and waves' worth of
them and one more, tiles that end inside a bin and inside an 8x8 block, more
textures than fit in LDS, every filter and wrap mode at sizes that are no power
of two, any subset of the planes."""
import ctypes
import os

import numpy as np
import pytest

import synth
from habitat_sim_amd import RendererConfiguration, RendererStandalone
from habitat_sim_amd import _native as N
from habitat_sim_amd import hip, scenes
from habitat_sim_amd import math3d as m3
from habitat_sim_amd.assets import (GL_CLAMP_TO_EDGE, GL_LINEAR, GL_LINEAR_MIPMAP_LINEAR,
                                    GL_LINEAR_MIPMAP_NEAREST, GL_MIRRORED_REPEAT, GL_NEAREST,
                                    GL_NEAREST_MIPMAP_LINEAR, GL_NEAREST_MIPMAP_NEAREST, GL_REPEAT)
from oracle.oracle import OracleRenderer

pytestmark = pytest.mark.gpu

NTHREADS = min(16, os.cpu_count() or 1)
BITS = {"color": N.PLANE_COLOR, "depth": N.PLANE_DEPTH, "linear_depth": N.PLANE_LINEAR_DEPTH,
        "semantic": N.PLANE_SEMANTIC}


def _soup(rng, n, size):
    """n triangles around the camera at the origin, which looks along -z; edge
    lengths from a hundredth of `size` to `size`, some across the near plane."""
    c = rng.uniform((-6.0, -6.0, -12.0), (6.0, 6.0, 1.0), (n, 1, 3))
    s = size * 10.0 ** rng.uniform(-2.0, 0.0, (n, 1, 1))
    return (c + s * rng.uniform(-1.0, 1.0, (n, 3, 3))).reshape(-1, 3).astype(np.float32)


def _pair(tile, grid, planes=N.PLANE_ALL, **tuning):
    r = RendererStandalone(RendererConfiguration().set_tile_size_count(tile, grid), planes=planes)
    if tuning:
        r.set_tuning(**tuning)
    return r, OracleRenderer(tile, grid)


def _draw(r, o):
    r.draw()
    o.draw(NTHREADS)


def _same(r, o, names=tuple(BITS), tag=""):
    for name in names:
        a, b = getattr(r, f"{name}_image")(), getattr(o, f"{name}_image")()
        diff = a != b
        if diff.ndim == 3:
            diff = diff.any(-1)
        assert not diff.any(), f"{tag} {name}: {int(diff.sum())} pixels differ from the oracle"


def _camera(x, scene, tile, pose=None):
    P = m3.perspective_projection(1.4, tile[0] / tile[1], 0.05, 50.0)
    x.update_camera(scene, P, m3.inverted_rigid(m3.identity() if pose is None else pose))


@pytest.mark.parametrize("tile,tuning", [((64, 64), {}), ((131, 77), {}), ((131, 77), dict(bin_size=8)),
                                         ((33, 129), dict(bin_size=16)), ((8, 8), {}), ((1, 1), {}),
                                         ((131, 77), dict(raster_mode=1)),
                                         ((131, 77), dict(raster_mode=1, bin_size=8, cull_mode=N.CULL_HIZ)),
                                         ((200, 9), dict(cull_mode=N.CULL_FRUSTUM)),
                                         ((97, 97), dict(cull_mode=N.CULL_HIZ, lane_pixels=16))])
def test_triangles_of_every_size(tile, tuning):
    """Seven scenes of 0 to 1500 triangles each; two frames, so that a culled
    one has a previous frame's visible set too."""
    rng = np.random.default_rng(tile[0] * 1000 + tile[1])
    counts = (1, 0, 63, 64, 65, 257, 1500)
    meshes = [(_soup(rng, max(n, 1), size), np.arange(3 * max(n, 1), dtype=np.uint32), None, None, k % 2)
              for k, (n, size) in enumerate(zip(counts, (300.0, 1.0, 3.0, 40.0, 2.0, 1.0, 1.0)))]
    fd = synth.mesh_file(meshes, [synth.flat((0.9, 0.5, 0.2, 1)), synth.flat((0.3, 0.6, 1.0, 1))])
    r, o = _pair(tile, (4, 2), **tuning)
    for x in (r, o):
        assert x.add_file_data(fd)
        for s, n in enumerate(counts):
            if n:
                x.add_node_hierarchy(s, f"m{s}", None, s + 1)
            # (outside the frustum behind the camera: every vertex beyond a plane)
            x.add_node_hierarchy(s, "m2", m3.translation((0.0, 0.0, 60.0)), 90)
            _camera(x, s, tile)
    _draw(r, o)
    _same(r, o, tag="first")
    if min(tile) > 1:
        assert len(np.unique(r.semantic_image())) > 4
    for x in (r, o):
        for s in range(len(counts)):
            _camera(x, s, tile, m3.rotation_y(0.4))
    _draw(r, o)
    _same(r, o, tag="second")
    r.close()


@pytest.mark.parametrize("tuning", [{}, dict(cull_mode=N.CULL_HIZ), dict(bin_size=8)])
def test_a_whole_scene_in_one_bin(tuning):
    """9000 small triangles inside 16x16 pixels: a bin's list many times longer
    than the mean."""
    rng = np.random.default_rng(5)
    p = rng.uniform((-0.1, -0.1, -3.0), (0.1, 0.1, -1.0), (9000, 1, 3)) + rng.uniform(-0.02, 0.02, (9000, 3, 3))
    mesh = (p.reshape(-1, 3).astype(np.float32), np.arange(27000, dtype=np.uint32), None, None, 0)
    r, o = _pair((128, 128), (2, 1), **tuning)
    for x in (r, o):
        assert x.add_file_data(synth.mesh_file([mesh], [synth.flat((1, 1, 1, 1))]))
        x.add_node_hierarchy(1, "m0", None, 7)
        for s in range(2):
            _camera(x, s, (128, 128))
    for _ in range(2):
        _draw(r, o)
        _same(r, o)
    r.close()


def _levels(rng, w, h):
    out = []
    while True:
        out.append(rng.integers(0, 256, (h, w, 4), dtype=np.uint8))
        if w == h == 1:
            return out
        w, h = max(w // 2, 1), max(h // 2, 1)


MINS = (GL_NEAREST, GL_LINEAR, GL_NEAREST_MIPMAP_NEAREST, GL_LINEAR_MIPMAP_NEAREST,
        GL_NEAREST_MIPMAP_LINEAR, GL_LINEAR_MIPMAP_LINEAR)
WRAPS = (GL_REPEAT, GL_CLAMP_TO_EDGE, GL_MIRRORED_REPEAT)


@pytest.mark.parametrize("count", [1, 7, 8, 9, 18])
def test_textures_filters_and_wraps(count):
    """`count` textures (8 descriptors fit in LDS), their sizes from 1x1 to
    37x64, each filter with each wrap mode, seen under perspective with
    coordinates well outside [0, 1]; the last texel of the last one is read."""
    rng = np.random.default_rng(count)
    sizes = ((4, 4), (1, 1), (37, 64), (2, 1), (5, 3), (16, 16), (1, 9), (33, 17), (64, 8))
    textures, meshes = [], []
    for k in range(count):
        w, h = sizes[k % len(sizes)]
        t = synth.texture(_levels(rng, w, h), min_filter=MINS[k % 6], mag_filter=(GL_NEAREST, GL_LINEAR)[k // 3 % 2],
                          wrap=WRAPS[(k + k // 6) % 3])
        t.wrap_t = WRAPS[(k // 2) % 3]
        textures.append(t)
        tilt = rng.uniform(-1.5, 1.5, 2)
        pos = np.array([[x, y, -4.0 + tilt[0] * x + tilt[1] * y] for x, y in ((-1, -1), (1, -1), (1, 1), (-1, 1))])
        pos += (rng.uniform(-1.5, 1.5), rng.uniform(-1.5, 1.5), 0.0)
        scale = 10.0 ** rng.uniform(-1.0, 1.3)
        uv = np.array([(0, 0), (1, 0), (1, 1), (0, 1)]) * scale + rng.uniform(-2.0, 2.0, 2)
        meshes.append((pos.astype(np.float32), np.array([0, 1, 2, 0, 2, 3], np.uint32), uv.astype(np.float32), None, k))
    fd = synth.mesh_file(meshes, [synth.flat((1, 1, 1, 1), texture=k) for k in range(count)], textures)
    tile = (150, 101)
    r, o = _pair(tile, (3, 1))
    for x in (r, o):
        assert x.add_file_data(fd)
        for s in range(3):
            for k in range(count):
                if s == 0 or (k + s) % 2 == 0:
                    x.add_node_hierarchy(s, f"m{k}", None, k + 1)
            _camera(x, s, tile, m3.translation((0.0, 0.0, -1.2 * s)))
    _draw(r, o)
    _same(r, o)
    r.close()


@pytest.mark.parametrize("names", [("color",), ("depth",), ("semantic",), ("linear_depth",),
                                   ("linear_depth", "semantic"), ("color", "depth"), ("color", "semantic")])
def test_any_subset_of_the_planes(names):
    rng = np.random.default_rng(11)
    tile = (70, 41)
    planes = sum(BITS[n] for n in names)
    r, o = _pair(tile, (2, 2), planes=planes)
    mesh = (_soup(rng, 200, 2.0), np.arange(600, dtype=np.uint32), rng.uniform(-1, 2, (600, 2)), None, 0)
    fd = synth.mesh_file([mesh], [synth.flat((1, 1, 1, 1), texture=0)],
                         [synth.texture(_levels(rng, 13, 7), min_filter=GL_LINEAR_MIPMAP_LINEAR, mag_filter=GL_LINEAR)])
    for x in (r, o):
        assert x.add_file_data(fd)
        for s in range(4):
            x.add_node_hierarchy(s, "m0", m3.rotation_y(0.5 * s), s + 1)
            _camera(x, s, tile)
    _draw(r, o)
    _same(r, o, names)
    r.close()


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("envs", [1, 5])
def test_moved_nodes_lights_and_cameras_over_frames(envs, graph):
    """Frames that move nothing, one node, every node, only cameras, only
    lights, nodes and lights of some scenes: the image is always the one of the
    present state."""
    rng = np.random.default_rng(envs)
    tile = (48, 48)
    n = 150
    nodes = 40
    pos = _soup(rng, n, 1.0)
    mesh = (pos, np.arange(3 * n, dtype=np.uint32), None, None, 0)
    fd = synth.mesh_file([mesh], [synth.flat((0.8, 0.8, 0.8, 1))])
    fd.materials[0].flat = False
    normal = rng.standard_normal(pos.shape)
    fd.meshes[0].normals = (normal / np.linalg.norm(normal, axis=1, keepdims=True)).astype(np.float32)
    grid = (envs, 1)
    r = RendererStandalone(RendererConfiguration().set_tile_size_count(tile, grid).set_max_light_count(2))
    r.set_tuning(graph=graph)
    o = OracleRenderer(tile, grid, max_light_count=2)
    ids = {}
    for x in (r, o):
        assert x.add_file_data(fd)
        for s in range(envs):
            ids[s] = [x.add_node_hierarchy(s, "m0", m3.scaling((0.3, 0.3, 0.3)), k + 1) for k in range(nodes)]
            light = x.add_empty_node(s)
            ids[s].append(light)
            x.add_light(s, light, N.LIGHT_POINT)
            _camera(x, s, tile)
    frames = [(), ("all",), (), ("one",), ("camera",), ("light",), ("one", "camera", "light"), ("some",), ("all", "light")]
    for f, what in enumerate(frames):
        for s in range(envs):
            move = []
            if "all" in what:
                move = list(range(nodes + 1))
            elif "one" in what and s == envs - 1:
                move = [int(rng.integers(nodes))]
            elif "some" in what and s % 2 == 0:
                move = sorted(rng.choice(nodes + 1, 7, replace=False))
            poses = [m3.mul(m3.translation(tuple(rng.uniform(-2, 2, 3) - (0, 0, 3))), m3.rotation_y(rng.uniform(0, 6)))
                     for _ in move]
            colour = rng.uniform(0.0, 2.0, 3).astype(np.float32)
            yaw = rng.uniform(-0.3, 0.3)
            for x in (r, o):
                t = x.transformations(s)
                for k, p in zip(move, poses):
                    t[ids[s][k]] = p
                if "light" in what:
                    x.light_colors(s)[0] = colour
                    x.light_ranges(s)[0] = np.float32(5.0 + f)
                if "camera" in what:
                    _camera(x, s, tile, m3.rotation_y(yaw))
        _draw(r, o)
        _same(r, o, tag=f"frame {f} {what}")
    r.close()


@pytest.mark.parametrize("scale", [1.0, 1e-12, 1e-25, 1e-40, 1e12, 1e20, 0.0])
def test_light_operands_of_every_magnitude(scale):
    """Normals of every length with zero and nearly zero components, lights of
    no, tiny, huge and infinite range, far away and on the surface."""
    tile = (64, 48)
    quads = [((-2, -2), (0, 0, 1)), ((0, -2), (0, 1, 0)), ((-2, 0), (1e-20, 0.6, 0.8)), ((0, 0), (0.3, -1e-30, 0.9))]
    meshes, normals = [], []
    for (x, y), n in quads:
        pos = np.array([(x, y, -3), (x + 2, y, -3), (x + 2, y + 2, -3), (x, y + 2, -3)], np.float32)
        meshes.append((pos, np.array([0, 1, 2, 0, 2, 3], np.uint32), None, None, 0))
        normals.append(np.tile(np.array(n, np.float64) * scale, (4, 1)).astype(np.float32))
    fd = synth.mesh_file(meshes, [synth.flat((0.9, 0.7, 0.8, 1))])
    fd.materials[0].flat = False
    for mesh, n in zip(fd.meshes, normals):
        mesh.normals = n
    lights = [((0.5, 0.5, -2.0), np.inf), ((-0.5, 0.5, -2.5), 3.0), ((0.0, 0.0, -3.0), 1e-35), ((1e12, 0.0, 0.0), 1e30),
              ((1e-25, 1e-25, -3.0), 5.0), ((0.0, 1e30, 0.0), np.inf), None, ((0.3, -0.4, -1.0), 0.0)]
    r = RendererStandalone(RendererConfiguration().set_tile_size_count(tile, (2, 1)).set_max_light_count(8))
    o = OracleRenderer(tile, (2, 1), max_light_count=8)
    for x in (r, o):
        assert x.add_file_data(fd)
        for s in range(2):
            for k in range(4):
                x.add_node_hierarchy(s, f"m{k}", None, k + 1)
            for i, light in enumerate(lights):
                node = x.add_empty_node(s)
                if light is None:
                    x.transformations(s)[node] = m3.look_at((0, 0, 0), (0.2, -1.0, -0.5), (0.0, 0.0, 1.0))
                    x.add_light(s, node, N.LIGHT_DIRECTIONAL)
                else:
                    x.transformations(s)[node] = m3.translation(light[0])
                    x.add_light(s, node, N.LIGHT_POINT)
                    x.light_ranges(s)[i] = np.float32(light[1])
                x.light_colors(s)[i] = np.array((0.2, 0.3, 0.1), np.float32)
            _camera(x, s, tile, m3.rotation_y(0.1 * s))
    _draw(r, o)
    _same(r, o)
    r.close()


def test_readback_rectangles_strides_and_large_images():
    """A framebuffer beyond 8 MB a plane, whole, in rectangles of odd offsets
    and sizes, into padded rows and as three channels."""
    rng = np.random.default_rng(2)
    tile = (523, 701)
    r, o = _pair(tile, (4, 2))
    mesh = (_soup(rng, 60, 4.0), np.arange(180, dtype=np.uint32), None, None, 0)
    for x in (r, o):
        assert x.add_file_data(synth.mesh_file([mesh], [synth.flat((0.2, 0.7, 0.4, 1))]))
        for s in range(8):
            x.add_node_hierarchy(s, "m0", m3.rotation_y(0.3 * s), s + 1)
            _camera(x, s, tile)
    _draw(r, o)
    _same(r, o)
    w, h = 4 * tile[0], 2 * tile[1]
    color, sem, lin = o.color_image(), o.semantic_image(), o.linear_depth_image()
    for x0, y0, x1, y1 in ((0, 0, w, h), (1, 3, 2, 4), (5, 0, 5 + 131, h), (0, h - 1, w, h), (w - 7, 11, w, 500)):
        pad = rng.integers(0, 256, (y1 - y0, x1 - x0 + 3, 4), dtype=np.uint8)
        keep = pad.copy()
        r.color_image_into((x0, y0, x1, y1), pad[:, :x1 - x0])
        np.testing.assert_array_equal(pad[:, :x1 - x0], color[y0:y1, x0:x1])
        np.testing.assert_array_equal(pad[:, x1 - x0:], keep[:, x1 - x0:])
        rgb = np.zeros((y1 - y0, x1 - x0, 3), np.uint8)
        r.color_image_into((x0, y0, x1, y1), rgb)
        np.testing.assert_array_equal(rgb, color[y0:y1, x0:x1, :3])
        ids = np.zeros((y1 - y0, x1 - x0 + 5), np.uint32)
        r.semantic_image_into((x0, y0, x1, y1), ids[:, :x1 - x0])
        np.testing.assert_array_equal(ids[:, :x1 - x0], sem[y0:y1, x0:x1])
        assert not ids[:, x1 - x0:].any()
        z = np.zeros((y1 - y0, x1 - x0), np.float32)
        r.linear_depth_image_into((x0, y0, x1, y1), z)
        np.testing.assert_array_equal(z, lin[y0:y1, x0:x1])
    r.close()


def test_a_bin_forced_to_the_rescan_more_often_than_a_word_holds():
    """More clipped primitives than record slots (2^20; every triangle here is
    a work item too wide for the vertex cache, which the clip pass takes), all
    in the tile's one bin: each one past the slots forces the bin's exact
    rescan.  Their number is the first for which adding the capacity and one
    each time would take the 32-bit count past 2^32 to below the capacity."""
    slots = 1 << 20
    extra = next(k for k in range(4000, 5000)
                 if (slots + k * (((slots + k + 63) & ~63) + 1)) % (1 << 32) <= ((slots + k + 63) & ~63))
    n = slots + extra
    rng = np.random.default_rng(17)
    tile = (32, 32)
    # right triangles of three pixels a side (each holds a pixel centre), facing the camera
    corner = rng.uniform(0.0, 29.0, (n, 1, 2)) + np.array([(0, 0), (3, 0), (0, 3)])
    pos = np.concatenate([corner / 16.0 - 1.0, rng.uniform(-0.9, 0.9, (n, 3, 1))], -1).reshape(-1, 3)
    where = rng.permutation(3 * n).astype(np.uint32)  # vertex k of the list lies at where[k]
    verts = np.empty((3 * n, 3), np.float32)
    verts[where] = pos
    mesh = (verts, where, None, rng.uniform(0, 1, (3 * n, 4)), 0)
    fd = synth.mesh_file([mesh], [synth.flat((1, 1, 1, 1))])
    r, o = _pair(tile, (1, 1), planes=N.PLANE_COLOR | N.PLANE_DEPTH | N.PLANE_SEMANTIC)
    for x in (r, o):
        assert x.add_file_data(fd)
        x.add_node_hierarchy(0, "m0", None, 3)
        x.update_camera(0, m3.identity(), m3.identity())
    for _ in range(2):
        _draw(r, o)
        _same(r, o, ("color", "depth", "semantic"))
        st = r.frame_stats()
        assert st["triangles_clipped"] > slots and st["overflowed_bins"] == 1, st
    r.close()


@pytest.mark.parametrize("wrap", [GL_CLAMP_TO_EDGE, GL_MIRRORED_REPEAT, GL_REPEAT])
@pytest.mark.parametrize("size", [(5, 3), (8, 4)])
def test_wrap_modes_that_are_none(wrap, size):
    """A file may carry any number as a wrap mode; one that is none of GL's
    repeats, also where its low 16 bits are another mode's."""
    rng = np.random.default_rng(3)
    t = synth.texture(_levels(rng, *size), min_filter=GL_LINEAR, mag_filter=GL_LINEAR, wrap=wrap + (1 << 16))
    t.wrap_t = wrap + (5 << 16)
    pos = np.array([(-1, -1, -2), (1, -1, -2), (1, 1, -2), (-1, 1, -2)], np.float32)
    uv = np.array([(-1.6, -1.3), (2.7, -1.3), (2.7, 2.2), (-1.6, 2.2)], np.float32)
    fd = synth.mesh_file([(pos, np.array([0, 1, 2, 0, 2, 3], np.uint32), uv, None, 0)],
                         [synth.flat((1, 1, 1, 1), texture=0)], [t])
    tile = (61, 47)
    r, o = _pair(tile, (1, 1))
    for x in (r, o):
        assert x.add_file_data(fd)
        x.add_node_hierarchy(0, "m0", None, 1)
        _camera(x, 0, tile)
    _draw(r, o)
    _same(r, o)
    r.close()


def test_readback_into_pinned_memory():
    """Images on both sides of the line above which the device copies into
    pinned memory itself, whole and in padded rows, four bytes and packed RGB8."""
    tile = (401, 263)
    runtime, pin = hip.hip(), ctypes.c_void_p()
    assert runtime.hipHostMalloc(ctypes.byref(pin), ctypes.c_size_t(1 << 20), ctypes.c_uint(0)) == 0
    pinned = np.frombuffer((ctypes.c_uint8 * (1 << 20)).from_address(pin.value), np.uint8)

    def nines(dtype, *shape):
        image = pinned[:int(np.prod(shape)) * np.dtype(dtype).itemsize].view(dtype).reshape(shape)
        image[...] = 9
        return image

    r, o = _pair(tile, (2, 1))
    mesh = (_soup(np.random.default_rng(4), 60, 4.0), np.arange(180, dtype=np.uint32), None, None, 0)
    for x in (r, o):
        assert x.add_file_data(synth.mesh_file([mesh], [synth.flat((0.2, 0.7, 0.4, 1))]))
        for s in range(2):
            x.add_node_hierarchy(s, "m0", m3.rotation_y(0.3 * s), s + 1)
            _camera(x, s, tile)
    _draw(r, o)
    color, lin = o.color_image(), o.linear_depth_image()
    for x0, y0, x1, y1 in ((0, 0, 802, 263), (1, 3, 2, 4), (10, 0, 138, 256), (10, 0, 139, 256), (300, 7, 428, 92),
                           (300, 7, 428, 93), (3, 1, 802, 40)):
        w, h = x1 - x0, y1 - y0
        for pad in (0, 5):
            for c in (4, 3):
                image = nines(np.uint8, h, w + pad, c)
                r.color_image_into((x0, y0, x1, y1), image[:, :w])
                np.testing.assert_array_equal(image[:, :w], color[y0:y1, x0:x1, :c])
                assert (image[:, w:] == 9).all()
            depth = nines(np.float32, h, w + pad)
            r.linear_depth_image_into((x0, y0, x1, y1), depth[:, :w])
            np.testing.assert_array_equal(depth[:, :w], lin[y0:y1, x0:x1])
            assert (depth[:, w:] == 9).all()
    r.close()
    assert runtime.hipHostFree(pin) == 0


def test_frames_submitted_ahead_of_the_gpu():
    """Ten frames with their own cameras and moved nodes, submitted without a
    wait between them (a frame takes longer on the GPU than its submission on
    the host), their planes copied in stream order: each is the frame that the
    same inputs give when every draw is waited for."""
    spec = scenes.apartments(256, tile=64)
    cfg = RendererConfiguration().set_tile_size_count(spec.tile, spec.grid)
    rng = np.random.default_rng(8)
    names = ("color", "linear_depth", "semantic")
    r = RendererStandalone(cfg, planes=sum(BITS[n] for n in names))
    scenes.populate(r, spec)
    n = len(spec.envs)
    proj = np.stack([e.projection for e in spec.envs]).astype(np.float32)
    views = np.stack([[m3.inverted_rigid(scenes.random_pose_in_box(rng, (2.0, 2.0), (10.0, 10.0))) for _ in range(n)]
                      for _ in range(10)]).astype(np.float32)
    tops = len(r.transformations(0)) // 2
    moves = [[(int(rng.integers(n)), 2 * int(rng.integers(1, tops)), m3.translation(tuple(rng.uniform(-1, 1, 3))))
              for _ in range(40)] for _ in range(10)]
    start = [np.array(r.transformations(s)._a) for s in range(n)]
    runtime, size = hip.hip(), 4 * n * spec.tile[0] * spec.tile[1]

    def frames(wait):
        for s in range(n):
            r.transformations(s)._a[:] = start[s]
        r.draw()
        r.synchronize()
        kept = [[hip.DeviceBuffer(size) for _ in names] for _ in range(10)]
        for k in range(10):
            r.update_cameras(0, proj, views[k])
            for s, node, t in moves[k]:
                r.transformations(s)[node] = t
            r.draw()
            for name, buf in zip(names, kept[k]):
                assert runtime.hipMemcpyAsync(buf.ptr, ctypes.c_void_p(r.plane_device_pointer(BITS[name])),
                                              ctypes.c_size_t(size), hip.D2D, ctypes.c_void_p(r.stream())) == 0
            if wait:
                r.synchronize()
        r.synchronize()
        out = np.zeros((10, len(names), size // 4), np.uint32)
        for k in range(10):
            for i in range(len(names)):
                kept[k][i].to_host(out[k, i])
                kept[k][i].close()
        return out

    ref = frames(True)
    got = frames(False)
    for k in range(10):
        np.testing.assert_array_equal(got[k], ref[k], err_msg=f"frame {k}")
        assert k == 0 or (ref[k] != ref[k - 1]).any()
    r.close()


@pytest.mark.parametrize("tile,tuning", [((1100, 1000), {}), ((1100, 1000), dict(cull_mode=N.CULL_HIZ)),
                                         ((270, 262), dict(bin_size=8)),
                                         ((270, 262), dict(bin_size=8, cull_mode=N.CULL_HIZ)),
                                         ((270, 262), dict(bin_size=8, raster_mode=1, cull_mode=N.CULL_HIZ)),
                                         ((530, 517), dict(bin_size=16, chunk_triangles=64))])
def test_more_bins_than_the_lds_counts(tile, tuning):
    """Scenes of more than 1024 bins, whose (bin, triangle) pairs go straight to
    the bins, beside one with a small viewport, whose pairs are counted in LDS."""
    rng = np.random.default_rng(29)
    r, o = _pair(tile, (3, 1), **tuning)
    meshes = [(_soup(rng, n, size), np.arange(3 * n, dtype=np.uint32), None, rng.uniform(0, 1, (3 * n, 4)), 0)
              for n, size in ((4000, 1.0), (2500, 3.0))]
    fd = synth.mesh_file(meshes, [synth.flat((1, 1, 1, 1))])
    for x in (r, o):
        assert x.add_file_data(fd)
        x.set_scene_viewport(1, (70, 50))
        for s in range(3):
            x.add_node_hierarchy(s, "m0", None, 1 + s)
            x.add_node_hierarchy(s, "m1", m3.rotation_y(0.5), 7)
    for f in range(3):
        for x in (r, o):
            for s in range(3):
                _camera(x, s, tile, m3.rotation_y(0.3 * f + s))
        _draw(r, o)
        _same(r, o, tag=f"frame {f}")
    r.close()
