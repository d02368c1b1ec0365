"""The binning's rules at their edges: 2560 and 2561 input triangles and 2048 and 2049 tiles (one workgroup
or the general kernels), and triangles of more than 256 tiles, few and more than a block's waves share
out, with the 8x8-tile blocks of their boxes cut by the canvas.  Frame, depth and winner ids equal the
oracle's in every bin order, and the numbers of bin entries are the same in all of them."""
import numpy as np
import pytest

from draw_amd import workloads
from draw_amd.scene import Camera, Scene
from parity import assert_same, oracle

pytestmark = pytest.mark.gpu


def _soup(seed, n, W, H, median_px, cross):
    rng = np.random.default_rng(seed)
    tex = workloads._phong(workloads.noise_texture(64, rng))
    o = workloads.soup_object(n, W, H, 60.0, 0.1, 100.0, 3.0, tex, rng, cross_frac=cross, median_px=median_px, sigma=0.8)
    return Scene(W, H, Camera(position=(0.0, 0.0, 3.0), fov_x=60.0, near=-0.1, far=-100.0), (0.0, 6.0, 6.0), [o])


@pytest.mark.parametrize("W,H,tile,waves,n,median,cross", [
    (320, 240, 16, 4, 2560, 60.0, 0.2),
    (320, 240, 16, 4, 2561, 60.0, 0.2),
    (512, 256, 8, 1, 2500, 60.0, 0.2),       # 2048 tiles
    (16392, 8, 8, 1, 2500, 20.0, 0.2),       # 2049 tiles in one row
    (333, 197, 8, 1, 40, 20_000.0, 0.5),     # 42x25 tiles: a few triangles of large boxes, one workgroup
    (333, 197, 8, 1, 2500, 20_000.0, 0.5),   # more than 64 of them there
    (333, 197, 8, 1, 30_000, 20_000.0, 0.5), # and in a block of the general kernels
])
def test_binning_edges(renderer, W, H, tile, waves, n, median, cross):
    s = _soup(W + n, n, W, H, median, cross)
    ref = oracle(s)
    entries = set()
    renderer.set_tiling(tile, waves)
    try:
        for mode in (0, 1, 2):
            renderer.set_bin_order(mode)
            c, w = renderer.render(s)
            assert_same(c.frame, c.depth, w, ref, label=f"{n} triangles, bin order {mode}")
            entries.add(renderer.stats()["bin_entries"])
    finally:
        renderer.set_bin_order(2)
        renderer.set_tiling(16, 4)
    assert len(entries) == 1
