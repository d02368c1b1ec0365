"""Large canvas reads through the staging ring (from the second one of a context on): totals around the
1 MB where it starts, pixel counts that are no multiple of four, fewer and more chunks than the ring holds,
one, two and three buffers, changing from read to read.  The arrays equal the device buffers copied directly."""
import ctypes as C
import threading

import numpy as np
import pytest

from draw_amd import workloads
from draw_amd.render import Renderer, frame_uniforms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(300, 291), (363, 361), (512, 513), (1021, 1027), (1920, 1080), (2500, 1501)])
def test_staged_reads(W, H):
    r = Renderer(0)
    try:
        cv = r.canvas(W, H)
        p = [C.c_void_p() for _ in range(3)]
        r._check(r.L.dh_canvas_device_ptrs(r.ctx, cv, *(C.byref(q) for q in p)), "dh_canvas_device_ptrs")
        for k, (depth, winner) in enumerate([(True, True), (True, False), (True, True), (False, False), (False, True),
                                             (True, False)]):
            s = workloads.torus_scene(k + 1, W, H)
            r.render_device(s, frame_uniforms(s), r.mesh_handles(s))
            want = [r.device_read(q.value, 4 * W * H, t) for q, t in zip(p, (np.uint8, np.float32, np.uint32))]
            f = np.zeros((H, W, 4), np.uint8)
            d = np.full((H, W), -1.0, np.float32) if depth else None
            w = np.full((H, W), 7, np.uint32) if winner else None
            r.read_into(cv, f, d, w)
            assert np.array_equal(f.ravel(), want[0])
            assert d is None or np.array_equal(d.ravel().view(np.uint32), want[1].view(np.uint32))
            assert w is None or np.array_equal(w.ravel(), want[2])
    finally:
        r.close()


def test_threads_reading_one_context():
    W, H = 900, 700
    r = Renderer(0)
    try:
        s = workloads.torus_scene(3, W, H)
        cv = r.render_device(s, frame_uniforms(s), r.mesh_handles(s))
        want, depth = np.zeros((H, W, 4), np.uint8), np.zeros((H, W), np.float32)
        r.read_into(cv, want, depth)
        bad = []

        def reader():
            for _ in range(20):
                f, d = np.zeros_like(want), np.zeros_like(depth)
                r.read_into(cv, f, d)
                if not (np.array_equal(f, want) and np.array_equal(d, depth)):
                    bad.append(1)

        ts = [threading.Thread(target=reader) for _ in range(3)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not bad
    finally:
        r.close()
