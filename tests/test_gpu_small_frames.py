"""The one-workgroup kernels of small frames, at the sizes where their rounds of 1024 triangles end and at their limit of
2560: soups and triangles that clip into several, against the general binning and the oracle; and frames of a fresh
context that outgrow its first capacities there, in clipped triangles (k_geom_small) and in bin entries
(k_bin_small)."""
import numpy as np
import pytest

from draw_amd import workloads
from draw_amd.render import Renderer
from draw_amd.scene import IndexedMesh
from parity import assert_same, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1023, 1024, 1025, 2049, 2560, 2561])
@pytest.mark.parametrize("slivers", [False, True])
def test_limits(renderer, n, slivers):
    s = workloads.sliver_scene(31 + n, n, 96, 64) if slivers else workloads.soup_scene(n, n, 200, 120, 32)
    ref = oracle(s)
    got = {}
    try:
        for mode in (1, 2):  # submission order: general binning
            renderer.set_bin_order(mode)
            c, w = renderer.render(s)
            assert_same(c.frame, c.depth, w, ref, label=f"bin order {mode}")
            st = renderer.stats()
            assert st["tris_out"] == ref.stats["tris_emitted"]
            got[mode] = st["bin_entries"]
    finally:
        renderer.set_bin_order(2)
    assert got[1] == got[2]


@pytest.mark.parametrize("n", [0, 1, 31, 32, 33])
@pytest.mark.parametrize("W,H", [(16384, 8), (16392, 8), (512, 512), (520, 512)])  # 2048, 2049, 4096, 4160 tiles
def test_few_triangles_on_many_tiles(renderer, n, W, H):
    s = workloads.soup_scene(17 + n, max(n, 1), W, H, 32, cross_frac=0.3)
    if n == 0:
        s.objects = []
    else:  # half of them across many tiles
        big = workloads.soup_object((n + 1) // 2, W, H, 60.0, 0.1, 100.0, 3.0, s.objects[0].textures[0],
                                    np.random.default_rng(n), cross_frac=0.0, median_px=0.2 * W * H, sigma=0.5)
        s.objects[0].meshes[0].triangles = s.objects[0].meshes[0].triangles[:n // 2]
        s.objects.append(big)
    ref = oracle(s)
    entries = set()
    renderer.set_tiling(8, 1)
    try:
        for mode in (1, 2):
            renderer.set_bin_order(mode)
            c, w = renderer.render(s)
            assert_same(c.frame, c.depth, w, ref, label=f"bin order {mode}")
            entries.add(renderer.stats()["bin_entries"])
    finally:
        renderer.set_bin_order(2)
        renderer.set_tiling(16, 4)
    assert len(entries) == 1


def _front_slivers(n):
    """sliver_scene's triangles that face the camera, the first n of them."""
    s = workloads.sliver_scene(37, 3 * n, 160, 120)
    o = s.objects[0]
    t = o.meshes[0].triangles
    a, b, c = (o.vertices[t[:, k]].astype(np.float64) for k in range(3))
    to_camera = np.array([0.0, 0.0, 3.0]) - (a + b + c) / 3.0
    front = np.einsum("ij,ij->i", np.cross(b - a, c - b), to_camera) > 0
    o.meshes = [IndexedMesh(np.ascontiguousarray(t[front][:n]), 0, "front slivers")]
    assert o.meshes[0].triangles.shape[0] == n
    return s


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("n", [1024, 2560])
def test_clipped_triangles_outgrow_a_fresh_context(n, mode):
    s = _front_slivers(n)
    ref = oracle(s)
    assert ref.stats["tris_emitted"] > n + n // 4 + 1024
    r = Renderer(0)
    try:
        r.set_bin_order(mode)
        c, w = r.render(s)
        assert_same(c.frame, c.depth, w, ref, label=f"bin order {mode}")
        assert r.stats()["retries"] >= 1
        assert r.stats()["tris_out"] == ref.stats["tris_emitted"]
    finally:
        r.close()


def test_bin_entries_outgrow_a_fresh_context():
    W, H, n = 512, 256, 40  # 2048 tiles of 8x8
    s = workloads.soup_scene(41, n, W, H, 32, cross_frac=0.0)
    o = workloads.soup_object(n, W, H, 60.0, 0.1, 100.0, 3.0, s.objects[0].textures[0], np.random.default_rng(41),
                              cross_frac=0.0, median_px=0.4 * W * H, sigma=0.2)
    s.objects = [o]
    ref = oracle(s)
    r = Renderer(0, 8, 1)
    try:
        c, w = r.render(s)
        assert_same(c.frame, c.depth, w, ref)
        st = r.stats()
        assert st["bin_entries"] > 4 * (n + n // 4 + 1024) + 2048 and st["retries"] >= 1, st
    finally:
        r.close()
