"""The quadrant raster's staged records: tiles whose lists are mostly small triangles (rasterized a
record to a few lanes), lists around a chunk of 128 records, rectangles around 8 pixels, records that
are not exact because their texture coordinates lie above 1 (still inside the texture) or their edges
are long, under every tiling.  Byte for byte against the oracle."""
import numpy as np
import pytest

from draw_amd import workloads
from draw_amd.scene import Camera, Scene
from parity import assert_same, oracle

pytestmark = pytest.mark.gpu

TILINGS = [(8, 1), (16, 1), (16, 2), (16, 4), (32, 1), (32, 2), (32, 4), (32, 8), (32, 16)]


def _scene(seed, n, W, H, median_px, sigma, uv_over):
    rng = np.random.default_rng(seed)
    tex = workloads._phong(workloads.noise_texture(64, rng))
    o = workloads.soup_object(n, W, H, 60.0, 0.1, 100.0, 3.0, tex, rng, cross_frac=0.05, median_px=median_px,
                              sigma=sigma)
    if uv_over:  # floor(u * 63) stays at most 63
        o.texture_vertices = (o.texture_vertices * np.float32(1.0003)).astype(np.float32)
    return Scene(W, H, Camera(position=(0.0, 0.0, 3.0), fov_x=60.0, near=-0.1, far=-100.0), (0.0, 6.0, 6.0), [o])


@pytest.mark.parametrize("n,W,H,median,sigma,uv_over", [
    (3, 16, 16, 20.0, 0.5, False), (250, 8, 8, 4.0, 0.3, False), (257, 31, 33, 4.0, 0.3, False),
    (2_000, 64, 48, 1.5, 0.4, False), (20_000, 64, 48, 3.0, 0.6, False), (3_000, 70, 41, 30.0, 0.4, False),
    (2_000, 64, 48, 4.0, 0.6, True), (400, 3000, 40, 40_000.0, 0.5, False)])
def test_small_records_bit_exact(renderer, n, W, H, median, sigma, uv_over):
    s = _scene(n + W, n, W, H, median, sigma, uv_over)
    ref = oracle(s)
    try:
        for tile, waves in TILINGS:
            renderer.set_tiling(tile, waves)
            c, w = renderer.render(s)
            assert_same(c.frame, c.depth, w, ref, label=f"{tile}x{waves}")
    finally:
        renderer.set_tiling(16, 4)


@pytest.mark.parametrize("kind,tile,waves", [(0, 16, 4), (0, 32, 4), (1, 16, 4), (1, 32, 8)])
def test_shard_visibility_of_both_rasters(renderer, kind, tile, waves):
    """The packed visibility that the quadrant raster writes itself, and k_vis_pack's of the other kind:
    one shard of one, merged with nothing and shaded, is the frame."""
    s = _scene(9, 4_000, 75, 53, 12.0, 0.8, False)
    ref = oracle(s)
    r = renderer
    r.set_raster(kind, tile, waves)
    try:
        from draw_amd.render import frame_uniforms
        fr, cv = frame_uniforms(s), r.canvas(s.width, s.height)
        vis = r.device_alloc(8 * s.width * s.height)
        r.render_shard(fr, r.mesh_handles(s), 0, cv, vis)
        r.shade_shard(vis, 0)
        f, d, w = r.read(cv, s.width, s.height)
        r.device_free(vis)
        assert_same(f, d, w, ref, label=f"shard {kind}:{tile}x{waves}")
    finally:
        r.set_raster(0, 16, 4)
