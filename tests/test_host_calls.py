"""The library's host code without a device, on a stand-in for the HIP runtime (standin_hip.c): what it hands to
the kernels after an allocation failed, and large canvas reads whose helper threads are late or whose staging cannot
be allocated, and which lists a transparent pass gets."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, {root!r})
S = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)
S.standin_room.argtypes, S.standin_room.restype = [C.c_uint64], C.c_int64
S.standin_fail_alloc.argtypes = S.standin_host_allocs.argtypes = [C.c_long]
S.standin_launches.restype = C.c_long
S.standin_launch_name.argtypes, S.standin_launch_name.restype = [C.c_long], C.c_char_p
S.standin_launch_arg.argtypes, S.standin_launch_arg.restype = [C.c_long, C.c_int], C.c_uint64
S.standin_queries.restype = C.c_uint64
S.standin_hold_array.argtypes, S.standin_hold_array.restype = [C.c_size_t, C.c_double], C.c_void_p
import numpy as np
from draw_amd import workloads
from draw_amd._lib import DrawHipError
from draw_amd.render import Renderer, frame_uniforms
"""


@pytest.fixture(scope="module")
def standin(tmp_path_factory):
    so = tmp_path_factory.mktemp("standin") / "libstandin.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", os.path.join(HERE, "standin_hip.c"), "-o", str(so)], check=True)
    return str(so)


def run(standin, body, timeout=100):
    r = subprocess.run([sys.executable, "-c", PRELUDE.format(root=ROOT, so=standin) + body], capture_output=True,
                       text=True, timeout=timeout, cwd=ROOT)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


# A frame, a larger one one of whose allocations fails (each in turn), then one of a size between: its kernels must
# get no capacity beyond the end of any buffer.
CAPACITIES = """
def lim32(x):
    return x & 0xFFFFFFFF

# kernel -> [(pointer argument, bytes it must have, as a function of the arguments)]
def boxes(cap):
    return ((cap + 15) & ~15) + 8 * cap
CHECKS = {
    "k_geom_emit": [(6, lambda a: 96 * a(8)), (7, lambda a: 144 * a(8)), (11, lambda a: 4 * a(8)),
                    (12, lambda a: boxes(a(8))), (13, lambda a: 4 * a(8))],
    "k_pair_hist": [(0, lambda a: boxes(a(5))), (1, lambda a: 4 * a(5)), (2, lambda a: 96 * a(5))],
    "k_pair_scatter": [(0, lambda a: boxes(a(5))), (10, lambda a: 8 * a(9))],
    "k_pair_sort": [(0, lambda a: 8 * a(2)), (4, lambda a: 4 * a(2)), (5, lambda a: 8 * a(3)), (6, lambda a: 4 * a(2))],
    "k_bin_small": [(0, lambda a: 96 * a(3)), (5, lambda a: boxes(a(3))), (6, lambda a: 4 * a(3)), (9, lambda a: 4 * a(8))],
    "k_bin_emitILb": [(0, lambda a: 96 * a(3)), (6, lambda a: 4 * a(3)), (10, lambda a: 4 * a(9)), (11, lambda a: 4 * a(9))],
    "k_bin_emit_wide": [(9, lambda a: 4 * a(8)), (10, lambda a: 4 * a(8))],
    "k_radix_hist": [(0, lambda a: 4 * a(2))],
    "k_radix_scatter": [(i, lambda a: 4 * a(5)) for i in range(4)],
}
seen = set()
def check(label):
    for i in range(S.standin_launches(0)):
        name = S.standin_launch_name(i).decode()
        for k, rules in CHECKS.items():
            if k not in name:
                continue
            seen.add(k)
            for arg, need in rules:
                p, n = S.standin_launch_arg(i, arg), need(lambda j: lim32(S.standin_launch_arg(i, j)))
                if p:
                    room = S.standin_room(p)
                    assert room >= n, f"{label}: {name} argument {arg} needs {n} bytes, its buffer has {room}"

def render(r, n_tri):
    s = workloads.soup_scene(1, n_tri, 640, 480, 16)
    return r.render_device(s)

for bins in (1, 2):
    failed = 0
    for k in range(64):
        r = Renderer(0)
        r.set_bin_order(bins)
        render(r, 500)
        s = workloads.soup_scene(1, 60_000, 640, 480, 16)  # its resources first: the frame's own allocations are to fail
        fr, hs = frame_uniforms(s), r.mesh_handles(s)
        S.standin_fail_alloc(k)
        try:
            r.render_device(s, fr, hs)
        except DrawHipError:
            failed += 1
        S.standin_fail_alloc(-1)
        S.standin_launches(1)
        render(r, 9_000)
        check(f"bins {bins}, allocation {k} failed")
        n = failed
        r.close()
        if n <= k:
            break
    assert failed >= 10, failed
assert seen == set(CHECKS) - {"k_bin_small"}, seen
"""


def test_capacities_after_a_failed_allocation(standin):
    run(standin, CAPACITIES)


# A helper thread that is not given the processor in the middle of its copy delays the read and does not fail it;
# a device that stops raising flags does.
LATE_HELPER = """
W, H = 1280, 720
r = Renderer(0)
cv = r.canvas(W, H)
p = [C.c_void_p() for _ in range(3)]
r._check(r.L.dh_canvas_device_ptrs(r.ctx, cv, *(C.byref(q) for q in p)), "dh_canvas_device_ptrs")
want = np.random.default_rng(1).integers(0, 256, 4 * W * H, np.uint8)
C.memmove(p[0].value, want.ctypes.data, want.nbytes)
f, d = np.zeros((H, W, 4), np.uint8), np.zeros((H, W), np.float32)
for _ in range(3):
    r.read_into(cv, f, d)
assert np.array_equal(f.ravel(), want)
at = S.standin_hold_array(4 * W * H, 3.0)
r._check(r.L.dh_canvas_read(r.ctx, cv, at, d.ctypes.data, None), "dh_canvas_read")
assert S.standin_holds() > 0
assert C.string_at(at, 4 * W * H) == want.tobytes()
S.standin_no_reads(1)
try:
    r.read_into(cv, f, d)
    raise SystemExit("a read that the device never did")
except DrawHipError:
    pass
S.standin_no_reads(0)
f[...] = 0
r.read_into(cv, f, d)
assert np.array_equal(f.ravel(), want)
r.close()
"""


def test_a_late_helper_does_not_fail_a_read(standin):
    run(standin, LATE_HELPER)


# Reads of a few megabytes go through the staging from a context's first on, with as much of it as there is; without
# any, through the runtime's copy.  Smaller ones make it once they would have gained from it.
STAGING = """
W, H = 1283, 727
rng = np.random.default_rng(2)
for pieces in (0, 1, 2, 3, 4):
    r = Renderer(0)
    cv = r.canvas(W, H)
    p = [C.c_void_p() for _ in range(3)]
    r._check(r.L.dh_canvas_device_ptrs(r.ctx, cv, *(C.byref(q) for q in p)), "dh_canvas_device_ptrs")
    S.standin_host_allocs(pieces)
    for k in range(5):
        want = [rng.integers(0, 256, 4 * W * H, np.uint8) for _ in p]
        for q, v in zip(p, want):
            C.memmove(q.value, v.ctypes.data, v.nbytes)
        out = [np.zeros(4 * W * H, np.uint8) for _ in p]
        dst = [None if (k >> i) & 1 else v.ctypes.data for i, v in enumerate(out)]
        S.standin_launches(1)
        r._check(r.L.dh_canvas_read(r.ctx, cv, *dst), "dh_canvas_read")
        n = sum(b"k_read_out" in S.standin_launch_name(i) for i in range(S.standin_launches(0)))
        assert (n > 0) == (pieces > 0), (pieces, k, n)
        for d, a, b in zip(dst, out, want):
            assert d is None or np.array_equal(a, b), (pieces, k)
    S.standin_host_allocs(-1)
    r.close()
for W, H, first in ((480, 360, 3), (361, 363, None)):  # 1.4 MB; just below 1 MB
    r = Renderer(0)
    cv = r.canvas(W, H)
    f, d = np.zeros((H, W, 4), np.uint8), np.zeros((H, W), np.float32)
    used = []
    for k in range(6):
        S.standin_launches(1)
        r.read_into(cv, f, d)
        used.append(any(b"k_read_out" in S.standin_launch_name(i) for i in range(S.standin_launches(0))))
    assert used == [first is not None and k >= first for k in range(6)], used
    r.close()
"""


def test_reads_with_the_staging_there_is(standin):
    run(standin, STAGING)


# The submission-ordered lists of a transparent pass rank the ids that share a counter against each other.  However its
# triangles lie, at most 1024 of the input's may share one; where the counters do not suffice, the radix sort.
SHARES = """
from draw_amd.scene import Texture
def scene(n, W, H):
    s = workloads.torus_scene(1, W, H)
    o = workloads.soup_object(n, W, H, 60.0, 0.1, 100.0, 3.0, Texture(alpha=0.5), np.random.default_rng(1))
    s.objects = [o]
    return s
got = {}
for W, H, tile in ((640, 480, 16), (3840, 2160, 16), (3840, 2160, 8), (7680, 4320, 8), (30000, 30000, 8)):
    tiles = -(-W // tile) * -(-H // tile)
    r = Renderer(0, tile, 4 if tile == 16 else 1)
    for n in (1, 1000, 2000, 16384, 16385, 32768, 32769, 65536, 65537):
        S.standin_launches(1)
        r.render_device(scene(n, W, H))
        names = [S.standin_launch_name(i).decode() for i in range(S.standin_launches(0))]
        segs = [d for d in (256, 2048) if any(f"k_pair_sortILi{d}ELb1E" in x for x in names)]
        assert len(segs) <= 1
        if segs:
            levels = min(256, 8192 // -(-tiles // segs[0]))
            assert levels and n <= 1024 * levels, (W, H, tile, n, segs, levels)
        else:
            assert any("k_bin_emitILb1E" in x for x in names)
        got[W, tile, n] = segs[0] if segs else 0
    r.close()
assert [got[640, 16, n] for n in (1, 65536, 65537)] == [256, 256, 0]
assert [got[3840, 16, n] for n in (16385, 65536)] == [256, 256]
assert [got[3840, 8, n] for n in (16384, 16385, 65536)] == [256, 2048, 2048]
assert [got[7680, 8, n] for n in (16384, 32768, 32769)] == [2048, 2048, 0]
"""


def test_transparent_lists_by_size(standin):
    run(standin, SHARES)
