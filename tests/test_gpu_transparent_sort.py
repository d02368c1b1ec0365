"""The transparent pass's sort and tile lists at the sizes where they change: meshes around a sort chunk of
1024 triangles and around the 32768 of the chunked sort, more meshes than one sort launch takes, one mesh
drawn twice, tiles of each size, and tile counts around the change from 256 to 2048 segments.  Frames equal
the oracle's, and those of another tiling where the oracle would take long; the sorted order is the stable
descending one."""
import numpy as np
import pytest

from draw_amd import workloads
from draw_amd.scene import Camera, Scene, Texture
from parity import assert_same, oracle

pytestmark = pytest.mark.gpu


def _scene(ns, width, height, half=0.8):
    """Overlapping windows of 2 n^2 triangles each, one object a window."""
    rng = np.random.default_rng(sum(ns) + width)
    objs = []
    for k, n in enumerate(ns):
        tex = Texture(ka=(0.2, 0.2, 0.2), kd=(0.8, 0.6, 0.4), ks=(0.3, 0.3, 0.3), alpha=0.5,
                      map_kd=workloads.checker_texture(64, 8, rng))
        objs.append(workloads.window_object(n, half, 0.05 * (k % 20), tex, x0=0.07 * (k % 5) - 0.1, y0=0.05 * (k % 7)))
    return Scene(width, height, Camera(position=(0.1, 0.2, 3.0), fov_x=60.0, near=-0.1, far=-100.0), (0.0, 6.0, 6.0), objs)


def _order(obj, cam):
    t, v = obj.meshes[0].triangles, obj.vertices.astype(np.float32)
    ctr = ((v[t[:, 0]] + v[t[:, 1]]) + v[t[:, 2]]) / np.float32(3.0)
    d = ctr - np.array(cam, np.float32)
    return t[np.argsort(-np.sqrt((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]), kind="stable")]


@pytest.mark.parametrize("ns,W,H,tile,waves", [
    ([1], 64, 48, 16, 4),
    ([22, 23], 160, 120, 8, 1),                    # 968 and 1058 triangles
    ([32, 1, 45], 160, 120, 16, 4),                # 2048, 2 and 4050
    ([100], 8, 8, 8, 1),                           # 20,000 in one tile
    ([3] * 35 + [40], 160, 120, 32, 4),            # three launches of sixteen meshes at most
    ([128], 200, 150, 16, 4),                      # 32,768: the chunked sort's largest mesh
    ([129, 10], 200, 150, 16, 4),                  # 33,282: the radix sort, a chunked one after it
    ([181], 200, 150, 16, 4),                      # 65,522: the tile lists by the pair kernels
    ([182, 10], 200, 150, 16, 4),                  # 66,448: by the radix sort
])
def test_sizes(renderer, ns, W, H, tile, waves):
    s = _scene(ns, W, H)
    want = [_order(o, s.camera.position) for o in s.objects]
    ref = oracle(s)
    renderer.set_tiling(tile, waves)
    try:
        c, w = renderer.render(s)
    finally:
        renderer.set_tiling(16, 4)
    assert_same(c.frame, c.depth, w, ref, label=f"windows {ns}")
    renderer.sync_transparent_order(s)
    for o, t in zip(s.objects, want):
        assert np.array_equal(o.meshes[0].triangles, t)


def test_mesh_drawn_twice(renderer):
    s = _scene([20, 12], 160, 120)
    s.objects = [s.objects[0], s.objects[1], s.objects[0]]
    ref = oracle(s)
    c, w = renderer.render(s)
    assert_same(c.frame, c.depth, w, ref, label="a window drawn twice")


def test_many_tiles(renderer):
    """2048 segments (4104x2048 in tiles of 8) against 256 (tiles of 16)."""
    s = _scene([60, 50], 4104, 2048, half=1.4)
    got = []
    try:
        for tile in (8, 16):
            renderer.set_tiling(tile, 1 if tile == 8 else 4)
            c, _ = renderer.render(s)
            got.append(c.frame.copy())
    finally:
        renderer.set_tiling(16, 4)
    assert np.array_equal(got[0], got[1])
