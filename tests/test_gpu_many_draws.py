"""Frames of many small meshes: waves of one draw, of two and of up to 32 in the geometry kernels, with a mesh cut
inside a wave, on the boundary and empty, in the one-workgroup and the general geometry and in a batch.  Byte for
byte against the oracle."""
import numpy as np
import pytest

from draw_amd import workloads
from draw_amd.render import frame_uniforms
from draw_amd.scene import IndexedMesh
from parity import assert_same, oracle

pytestmark = pytest.mark.gpu


def _scene(seed, sizes, W=90, H=70):
    s = workloads.soup_scene(seed, sum(sizes), W, H, 16)
    o = s.objects[0]
    t, cuts = o.meshes[0].triangles, np.cumsum([0] + list(sizes))
    o.textures.append(workloads._phong(workloads.noise_texture(8, np.random.default_rng(seed)), 5))
    o.meshes = [IndexedMesh(np.ascontiguousarray(t[a:b]), k % 2) for k, (a, b) in enumerate(zip(cuts, cuts[1:]))]
    return s


SIZES = {"pairs": [2] * 300, "one each": [1] * 130, "pairs, general": [2] * 1400, "cuts": [64, 63, 1, 65, 0, 191, 256, 2],
         "cuts, general": [1000, 24, 0, 1500, 3, 61, 7], "twelve": [12] * 260}


@pytest.mark.parametrize("name", SIZES)
def test_many_draws(renderer, name):
    s = _scene(len(name), SIZES[name])
    c, w = renderer.render(s)
    assert_same(c.frame, c.depth, w, oracle(s), label=name)


def test_many_draws_in_a_batch(renderer):
    scenes = [_scene(k, n) for k, n in enumerate(SIZES.values())]
    for s, cv in zip(scenes, renderer.render_batch([(s, frame_uniforms(s)) for s in scenes])):
        f, d, w = renderer.read(cv, s.width, s.height)
        assert_same(f, d, w, oracle(s), label=f"{len(s.objects[0].meshes)} meshes")
