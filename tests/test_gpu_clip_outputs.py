"""The emits' clipped list, two lanes a triangle, at the sizes where its 32-triangle units end and where
the geometry lists change from one workgroup to the general kernels (16384 triangles): slivers across both
the near and the far plane, three outputs each, so that one lane goes round twice; in every bin order.
Frame, depth, winner ids and the number of clipped triangles equal the oracle's."""
import pytest

from draw_amd import workloads
from parity import assert_same, oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 65, 16_384, 16_385])
def test_clipped_outputs(renderer, n):
    s = workloads.sliver_scene(seed=29 + n, n_tri=n, width=96, height=64)
    ref = oracle(s)
    try:
        for mode in (0, 1, 2):
            renderer.set_bin_order(mode)
            c, w = renderer.render(s)
            assert_same(c.frame, c.depth, w, ref, label=f"{n} slivers, bin order {mode}")
            assert renderer.stats()["tris_out"] == ref.stats["tris_emitted"]
    finally:
        renderer.set_bin_order(2)
