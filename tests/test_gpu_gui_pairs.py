"""The GUI raster takes triangles two at a time: waves that only the first of a pair covers, only the second, both or
neither (large panels in halves, strips and glyphs, in odd and even numbers), and a font sample outside the atlas under
one of them.  Byte for byte against the oracle."""
import numpy as np
import pytest

from draw_amd import gui, workloads
from draw_amd._lib import DrawHipError
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _panels(W, H, n, rng, bad=None):
    v = np.zeros(4 * n, gui.GUI_VERTEX)
    for k in range(n):
        w, h = [(W, H), (W / 2, H), (W, 3.0), (9.0, 12.0)][k % 4]
        x, y = rng.uniform(0, W - w + 0.5), rng.uniform(0, H - h + 0.5)
        v["pos"][4 * k:4 * k + 4] = [(x, y), (x + w, y), (x + w, y + h), (x, y + h)]
        v["uv"][4 * k:4 * k + 4] = rng.uniform(0.02, 0.9, (4, 2))
        v["col"][4 * k:4 * k + 4] = rng.integers(0, 256, 4)
    if bad is not None:
        v["uv"][4 * bad:4 * bad + 4] = 3.0
    i = (4 * np.arange(n)[:, None] + np.array([0, 1, 2, 0, 2, 3])).ravel().astype(np.uint32)
    return v, i


@pytest.mark.parametrize("W,H,n", [(64, 64, 1), (65, 63, 4), (203, 117, 9), (640, 480, 40)])
@pytest.mark.parametrize("cut", [0, 3])  # the last triangle left out: an odd number
def test_gui_pairs(renderer, W, H, n, cut):
    rng = np.random.default_rng(W)
    s = workloads.torus_scene(5, width=W, height=H)
    font = gui.font_atlas(4)
    v, i = _panels(W, H, n, rng)
    i = i[:len(i) - cut]
    c = np.zeros(1, gui.GUI_CMD)
    c[0] = ((0, 0, W, H), 0, len(i), 0, 0)
    ref = O.render(s)
    assert O.gui_draw(ref.frame, ref.depth, v, i, c, font) == 0
    cv = renderer.render_device(s)
    renderer.draw_gui(cv, v, i, c, font)
    f, d, _ = renderer.read(cv, W, H)
    assert np.array_equal(f, ref.frame)
    assert np.array_equal(d.view(np.uint32), ref.depth.view(np.uint32))


@pytest.mark.parametrize("bad", [0, 1, 2, 3])
def test_a_sample_outside_the_atlas(renderer, bad):
    W, H = 96, 80
    s = workloads.torus_scene(5, width=W, height=H)
    v, i = _panels(W, H, 4, np.random.default_rng(3), bad)
    c = np.zeros(1, gui.GUI_CMD)
    c[0] = ((0, 0, W, H), 0, len(i), 0, 0)
    ref = O.render(s)
    assert O.gui_draw(ref.frame, ref.depth, v, i, c, gui.font_atlas(4)) != 0
    cv = renderer.render_device(s)
    with pytest.raises(DrawHipError, match="DH_E_TEXCOORD"):
        renderer.draw_gui(cv, v, i, c, gui.font_atlas(4))
