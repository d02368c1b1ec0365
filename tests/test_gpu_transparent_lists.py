"""The submission-ordered tile lists of a transparent pass where the canvas leaves their segments few counters per
tile: by 256 segments, by 2048 and by the stable sort, triangles spread out and piled up in a few tiles.  The frame
equals that of the canvas in larger tiles."""
import numpy as np
import pytest

from draw_amd import workloads
from draw_amd.scene import Camera, Scene, Texture

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,half", [([90, 13], 1.2), ([91, 13], 1.2), ([91, 13], 0.01), ([128, 2], 0.02)])
@pytest.mark.parametrize("W,H", [(3840, 2160), (7680, 4320)])
def test_few_counters(renderer, ns, half, W, H):
    rng = np.random.default_rng(sum(ns))
    objs = []
    for k, n in enumerate(ns):
        tex = Texture(ka=(0.2, 0.2, 0.2), kd=(0.8, 0.6, 0.4), ks=(0.3, 0.3, 0.3), alpha=0.5,
                      map_kd=workloads.checker_texture(64, 8, rng))
        objs.append(workloads.window_object(n, half, 0.1 * k, tex, x0=0.03, y0=0.02))
    # every second triangle of the first window once more, near the others: ids far apart share tiles
    m = objs[0].meshes[0]
    m.triangles = np.concatenate([m.triangles, m.triangles[::2]])
    s = Scene(W, H, Camera(position=(0.1, 0.2, 3.0), fov_x=60.0, near=-0.1, far=-100.0), (0.0, 6.0, 6.0), objs)
    got = []
    try:
        for tile, waves in ((8, 1), (32, 4)):
            renderer.set_tiling(tile, waves)
            c, _ = renderer.render(s)
            got.append(c.frame.copy())
    finally:
        renderer.set_tiling(16, 4)
    assert np.array_equal(got[0], got[1])
    assert (got[0] != got[0][0, 0]).any()
