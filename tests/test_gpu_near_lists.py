"""The near-first tile lists (k_pair_*) at the sizes where their segments, digits and buffers end:
one tile with more triangles than a sort block keeps in registers, tile counts around one segment
each, the change from 256 to 2048 segments, more wide triangles than an emit block's LDS buffer, and
geometry block counts around a scan round.  The frame, depth and winner ids and the number of bin
entries equal those of the submission-ordered lists, and the oracle's where it is quick."""
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


@pytest.mark.parametrize("W,H,tile,waves,n,median,cross,check", [
    (8, 8, 8, 1, 20_000, 20.0, 0.2, True),              # one segment of some 10,000 pairs
    (40, 24, 8, 1, 17_000, 30.0, 0.2, True),
    (2040, 8, 8, 1, 17_000, 30.0, 0.2, True),           # 255, 256 and 257 tiles
    (2048, 8, 8, 1, 17_000, 30.0, 0.2, True),
    (2056, 8, 8, 1, 17_000, 30.0, 0.2, True),
    (333, 197, 16, 4, 60_000, 900.0, 0.1, False),       # mostly wide triangles
    (333, 197, 32, 4, 17_000, 20.0, 1.0, True),         # every triangle crosses the near plane
    (4096, 2048, 8, 1, 50_000, 400.0, 0.1, False),      # 131072 tiles: 256 segments
    (4104, 2048, 8, 1, 50_000, 400.0, 0.1, False),      # 131328 tiles: 2048 segments
    (320, 240, 8, 1, 1_300_000, 1200.0, 0.0, False),    # over 512 wide triangles per emit block
    (64, 48, 16, 4, 2_097_153, 2.0, 0.0, False),        # 8193 blocks of 256: a scan round and one
])
def test_near_lists_equal_submission_order(renderer, W, H, tile, waves, n, median, cross, check):
    s = _soup(W + n, n, W, H, median, cross)
    got = {}
    renderer.set_tiling(tile, waves)
    try:
        for mode in (1, 2):
            renderer.set_bin_order(mode)
            c, w = renderer.render(s)
            got[mode] = (c.frame.copy(), c.depth.copy(), w.copy(), renderer.stats())
    finally:
        renderer.set_bin_order(2)
        renderer.set_tiling(16, 4)
    a, b = got[1], got[2]
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[2], b[2])
    assert np.array_equal(a[1].view(np.uint32), b[1].view(np.uint32))
    assert a[3]["bin_entries"] == b[3]["bin_entries"] > 0
    if check:
        assert_same(b[0], b[1], b[2], oracle(s), label="near first")
