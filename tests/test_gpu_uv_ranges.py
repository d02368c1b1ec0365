"""Texture coordinates outside [0, 1]: negative ones (sampled as 0), ones above 1 that stay in their row or run on
into the rows below it, ones that just stay in the map without the emit being able to tell, NaN, and ones that
leave it; maps of one texel to long rows, with and without an ambient map.  Frames equal the oracle's byte for byte,
and fail where it does."""
import numpy as np
import pytest

from draw_amd import workloads
from draw_amd._lib import DrawHipError
from draw_amd.scene import TextureMap
from oracle import oracle as O
from parity import assert_same

pytestmark = pytest.mark.gpu

F = np.float32


def _uv(kind, uv, w, h):
    u, v = uv[:, 0].astype(np.float64), uv[:, 1].astype(np.float64)
    mu, mv = max(w - 1, 1), max(h - 1, 1)
    if kind == "negative":
        u, v = u - 0.5, v - 0.5
    elif kind == "far negative":
        u, v = u * 41 - 40, v * 3000 - 2999
    elif kind == "in the last texel":  # up to a quarter of a texel beyond
        u, v = u * (1 + 0.25 / mu), v * (1 + 0.25 / mv)
    elif kind == "undecided":  # inside by a few ten-thousandths of a texel
        u, v = np.full_like(u, 1 + 0.9996 / mu), np.full_like(v, 1 + 0.9996 / mv)
    elif kind == "rows below":
        u, v = u * 3, 0.9 * v + 0.1
    elif kind == "just rows enough":
        u, v = u * 2, v * 0.9 + 2.5 / mv
    elif kind == "nan":
        u = np.where(np.arange(len(u)) % 5 == 0, np.nan, u)
    elif kind == "outside u":
        u, v = u * 3, v * (0.5 / mv)
    elif kind == "outside v":
        v = v * 2
    return np.stack([u, v], 1).astype(F)


@pytest.mark.parametrize("w,h,comp,ambient", [(64, 64, 4, False), (17, 5, 3, True), (2, 3, 4, False), (1, 1, 3, False),
                                              (1, 40, 4, True), (20000, 2, 4, False)])
def test_uv_ranges(renderer, w, h, comp, ambient):
    rng = np.random.default_rng(w)
    done = {}
    for kind in ("negative", "far negative", "in the last texel", "undecided", "rows below", "just rows enough", "nan",
                 "outside u", "outside v"):
        s = workloads.soup_scene(5, 700, 80, 60, 8)
        o = s.objects[0]
        t = o.textures[0]
        t.map_kd = TextureMap(rng.integers(0, 256, (h, w, comp), np.uint8))
        if ambient:
            t.map_ka = TextureMap(rng.integers(0, 256, (7, 33, 3), np.uint8))
        o.texture_vertices = _uv(kind, o.texture_vertices, w, h)
        ref = O.render(s)
        done[kind] = ref.rc
        for kind_r, tile, waves in ((0, 16, 4), (0, 32, 4), (0, 8, 1), (1, 16, 4)):
            renderer.set_raster(kind_r, tile, waves)
            try:
                if ref.rc == 0:
                    c, win = renderer.render(s)
                    assert_same(c.frame, c.depth, win, ref, label=f"{kind} {kind_r}:{tile}x{waves}")
                else:
                    with pytest.raises(DrawHipError, match="DH_E_TEXCOORD"):
                        renderer.render(s)
            finally:
                renderer.set_raster(0, 16, 4)
    # the coordinates are what their names say
    assert done["negative"] == done["far negative"] == done["nan"] == 0
    if not ambient:
        assert done["in the last texel"] == done["undecided"] == 0
    if h > 4 and not ambient:
        assert done["outside v"] != 0
