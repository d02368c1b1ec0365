"""Triangles of large tile boxes, whose 8x8-tile blocks the waves of a workgroup share out: fewer blocks than waves,
as many, one more, and more than every lane of every wave takes at once, in rows, columns and squares.  The near-first
frame and its bin entries equal those of the other bin orders, and the oracle's."""
import numpy as np
import pytest

from draw_amd import workloads
from draw_amd.scene import Camera, Scene
from parity import assert_same, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("general", [False, True])
@pytest.mark.parametrize("W,H", [
    (320, 56),      # 40x7 tiles: 5 blocks
    (1024, 64),     # 128x8: 16
    (64, 1032),     # 8x129: 17
    (16384, 16),    # 2048x2: 256 (one workgroup takes at most 2048 tiles: general)
    (2600, 2600),   # 325x325: 1681, over 16 waves of 64 lanes
])
def test_large_boxes(renderer, W, H, general):
    rng = np.random.default_rng(W)
    tex = workloads._phong(workloads.noise_texture(32, rng))
    big = workloads.soup_object(24, W, H, 60.0, 0.1, 100.0, 3.0, tex, rng, cross_frac=0.2, median_px=0.4 * W * H,
                                sigma=0.3)
    objs = [big]
    if general:  # past the one-workgroup kernels' triangles
        objs.append(workloads.soup_object(3000, W, H, 60.0, 0.1, 100.0, 3.0, tex, rng, median_px=10.0))
    s = Scene(W, H, Camera(position=(0.0, 0.0, 3.0), fov_x=60.0, near=-0.1, far=-100.0), (0.0, 6.0, 6.0), objs)
    ref = oracle(s)
    entries = set()
    renderer.set_tiling(8, 1)
    try:
        for mode in (0, 1, 2):
            renderer.set_bin_order(mode)
            c, w = renderer.render(s)
            assert_same(c.frame, c.depth, w, ref, label=f"bin order {mode}")
            entries.add(renderer.stats()["bin_entries"])
    finally:
        renderer.set_bin_order(2)
        renderer.set_tiling(16, 4)
    assert len(entries) == 1
