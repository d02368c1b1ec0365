"""The GUI overlay's raster at the sizes where its waves and rounds end: canvases that are no
multiple of its 8x8 pixels, lists around its rounds of 64 and 256 triangles and around an odd
number of hits, clip rectangles that miss their triangles (collapsed to row or column 0), zero-area
triangles, coordinates beyond exact edge arithmetic, and a three-component font.  Byte for byte
against the oracle."""
import numpy as np
import pytest

from draw_amd import gui, workloads
from draw_amd.scene import TextureMap
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _list(seed, W, H, n_tri, far):
    """n_tri triangles under 7 clip rectangles: ordinary, off-canvas, at the border, empty and huge."""
    rng = np.random.default_rng(seed)
    v = np.zeros(3 * n_tri, gui.GUI_VERTEX)
    c = rng.uniform([-8, -8], [W + 8, H + 8], (n_tri, 1, 2)) + rng.normal(0, max(2.0, W / 12), (n_tri, 3, 2))
    flat = rng.random(n_tri) < 0.1
    c[flat, 2] = c[flat, 0]                      # zero area
    if far:
        c[::3] *= rng.choice([1e3, 1e5, 1e7], (len(c[::3]), 1, 1))   # edges beyond 2^24
    v["pos"] = c.reshape(-1, 2)
    v["uv"] = rng.uniform(0.02, 0.95, (3 * n_tri, 2))
    v["col"] = rng.integers(0, 256, (3 * n_tri, 4))
    v["col"][rng.random(3 * n_tri) < 0.5, 3] = 255
    clips = [(0, 0, W, H), (-20, -20, -5, -5), (W + 3, 2, W + 9, H), (0, 0, 1, 1), (W / 3, H / 3, W / 2, H),
             (5, 5, 2, 2), (-1e9, -1e9, 1e9, 1e9)]
    cuts = np.linspace(0, n_tri, len(clips) + 1).astype(int)
    cmds = np.zeros(len(clips), gui.GUI_CMD)
    for k, r in enumerate(clips):
        cmds[k] = (r, 3 * cuts[k], 3 * (cuts[k + 1] - cuts[k]), 0, 0)
    return v, np.arange(3 * n_tri, dtype=np.uint32), cmds


@pytest.mark.parametrize("W,H,n_tri,far,comp", [
    (1, 1, 7, False, 4), (7, 5, 63, False, 4), (8, 8, 64, False, 4), (9, 17, 65, True, 4), (16, 16, 255, False, 4),
    (33, 15, 257, True, 4), (130, 71, 513, False, 4), (130, 71, 300, True, 3), (801, 599, 1200, False, 4)])
def test_gui_edges_bit_exact(renderer, W, H, n_tri, far, comp):
    s = workloads.torus_scene(5, width=W, height=H)
    font = gui.font_atlas(4)
    if comp == 3:
        font = TextureMap(font.img[..., 1:])
    v, i, c = _list(n_tri, W, H, n_tri, far)
    ref = O.render(s)
    assert O.gui_draw(ref.frame, ref.depth, v, i, c, font) == 0
    cv = renderer.render_device(s)
    renderer.draw_gui(cv, v, i, c, font)
    f, d, _ = renderer.read(cv, W, H)
    assert np.array_equal(f, ref.frame)
    assert np.array_equal(d.view(np.uint32), ref.depth.view(np.uint32))
