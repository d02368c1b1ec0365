"""The work that users of this renderer have it do, as cases that can be measured.

A case is a dict of plain values.  ``listed()`` gives the fixed ones, ``draw(rng)`` another one of the
same ranges, ``prepare(case, seed)`` what a program holds before a frame (renderer, resident meshes,
canvases, uniforms), ``run(state)`` one pass through the public entry points with its whole outputs,
``work(case)`` the bytes and operations the path cannot do without, and ``exact(case, seed)`` the
depth buffers in 64 bits (frames, winner ids and merged visibility words are whole numbers: None).

Every output is a device buffer seen as a tensor, in place (BGRA8 words and winner ids as int32,
visibility words as int64, depth as float32), except a read-back frame, which is two host arrays.
"""
from __future__ import annotations

import ctypes as C
import math
import random

import numpy as np
import torch

from draw_amd import gui, workloads
from draw_amd.render import Renderer, frame_uniforms
from draw_amd.scene import CLEAR_DEPTH, Camera, IndexedMesh, Object, Scene, Texture, TextureMap


# ------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # The smallest call: one object in a window, a frame of some 60 microseconds in which launches
        # and gaps count.  The tiling is what the autotuner picks for it.
        dict(name="torus_640x480", kind="torus", W=640, H=480, n_tri=2304, power=2, tile=32, waves=16, winners=False),
        # The reference application's own frame: 62k triangles of a full-screen scene drawn into its
        # 800x600 canvas at an offset, then the GUI's draw list over it.  Default settings.
        dict(name="app_gui_800x600", kind="app", W=800, H=600, n_tri=60_000, quads=1200, tile=16, waves=4, winners=True),
        # Opaque and transparent meshes of two objects: the back-to-front sort and the blend.
        dict(name="glass_1280x720", kind="glass", W=1280, H=720, n_tri=20_000, tile=16, waves=4, winners=True),
        # A drop-in's whole Scene::render: the frame and the depth end in the caller's host arrays.
        dict(name="readback_1280x720", kind="readback", W=1280, H=720, n_tri=20_000, power=2, tile=16, waves=4,
             winners=False),
        # An ordinary frame at sizes that divide nothing: ragged tiles, an RGB texture (as every JPEG
        # decodes to), a high specular power, default settings.
        dict(name="soup_1237x709_150k", kind="soup", W=1237, H=709, n_tri=150_001, power=32, comp=3, tex=1000, tile=16,
             waves=4, winners=True),
        # The benchmark's frame: 1M triangles at 1080p, the tiling the autotuner picks, a canvas without
        # winner ids (as the reference's).
        dict(name="soup_1080p_1m", kind="soup", W=1920, H=1080, n_tri=1_000_000, power=2, comp=4, tex=2048, tile=32,
             waves=4, winners=False),
        # One large mesh filling a 4K canvas (a serving request's largest resolution): pixels outnumber
        # triangles, the shading and the canvas writes count.
        dict(name="sphere_4k_500k", kind="sphere", W=3840, H=2160, n_tri=500_000, tex=1024, tile=16, waves=4,
             winners=False),
        # Micro-triangles, 2.4 per pixel, on nested shells: geometry and binning bound.
        dict(name="shells_1080p_5m", kind="shells", W=1920, H=1080, n_tri=5_000_000, tex=4096, tile=16, waves=4,
             winners=True),
        # The batched workload: 8 meshes of 1k to 500k triangles, 4 cameras each, four resolutions, one
        # graph-replayed launch.
        dict(name="batch_graph_32", kind="batch", views=32, tri_hi=500_000, tile=32, waves=4, winners=False),
        # What a render server's worker launches: a dozen requests of one moment (mixed meshes and
        # resolutions up to 4K) as one batch without a graph, since no two launches are alike.
        dict(name="batch_serving_12", kind="serving", views=12, tri_hi=500_000, tile=16, waves=4, winners=True),
        # A sort-last frame in two shards: both visibility passes, the merge, both shadings.
        dict(name="shards_1080p_250k", kind="shards", W=1920, H=1080, n_tri=250_000, tile=32, waves=4, winners=True),
    ]


TILINGS = [(8, 1), (16, 2), (16, 4), (32, 4), (32, 8), (32, 16)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["torus", "app", "glass", "readback", "soup", "soup", "sphere", "shells", "batch", "serving",
                       "shards"])
    tile, waves = rng.choice(TILINGS)
    c = dict(kind=kind, tile=tile, waves=waves, winners=rng.random() < 0.5)
    if kind in ("batch", "serving"):
        c.update(views=_log_int(rng, 2, 31 if kind == "batch" else 11), tri_hi=_log_int(rng, 4_000, 500_000))
        c["winners"] = c["winners"] and c["views"] <= 16
        return c
    W = _log_int(rng, 200, 1920)
    c.update(W=W, H=max(96, int(W * rng.uniform(0.4, 0.8))))
    if kind == "torus":
        c.update(n_tri=2304, power=rng.choice([2, 5, 32]))
    elif kind == "app":
        c.update(n_tri=_log_int(rng, 500, 120_000), quads=_log_int(rng, 20, 2000), W=min(W, 1280), H=min(c["H"], 720))
    elif kind == "glass":
        c.update(n_tri=_log_int(rng, 200, 40_000), winners=True)
    elif kind == "readback":
        c.update(n_tri=_log_int(rng, 300, 200_000), power=2)
    elif kind == "soup":
        c.update(n_tri=_log_int(rng, 300, 900_000), power=rng.choice([0, 2, 7, 32]), comp=rng.choice([3, 4]),
                 tex=_log_int(rng, 17, 2048))
    elif kind == "sphere":
        c.update(n_tri=_log_int(rng, 2_000, 500_000), tex=_log_int(rng, 64, 2048), W=2 * W, H=2 * c["H"])
    elif kind == "shells":
        c.update(n_tri=_log_int(rng, 50_000, 4_500_000), tex=_log_int(rng, 64, 4096))
    else:
        c.update(n_tri=_log_int(rng, 2_000, 500_000))
    return c


# ------------------------------------------------------------------------------------------- inputs
def _glass_scene(seed, W, H, n_tri):
    """An object of a torus and a tilted-UV window in front of it, then an object whose window hangs before
    its opaque plate: transparent meshes between and after opaque ones."""
    rng = np.random.default_rng(seed)
    base = workloads.torus_scene(seed, width=W, height=H)

    def material(alpha):
        return Texture(ka=(0.2, 0.2, 0.2), kd=(0.8, 0.6, 0.4), ks=(0.3, 0.3, 0.3), alpha=alpha,
                       map_kd=workloads.checker_texture(256, 8, rng))

    def joined(a, b):
        t = b.meshes[0].triangles.copy()
        t[:, :3] += a.vertices.shape[0]
        t[:, 3:6] += a.texture_vertices.shape[0]
        t[:, 6:] += a.normals_vertices.shape[0]
        return Object(np.concatenate([a.vertices, b.vertices]),
                      np.concatenate([a.normals_vertices, b.normals_vertices]),
                      np.concatenate([a.texture_vertices, b.texture_vertices]),
                      [IndexedMesh(a.meshes[0].triangles, 0), IndexedMesh(t, 1)], [a.textures[0], b.textures[0]])

    n = max(2, int(math.sqrt(n_tri / 4.0)))
    near = workloads.window_object(n, 1.1, 0.8, material(0.5))
    plate = workloads.window_object(2, 0.3, 1.1, Texture(), x0=0.4, y0=0.2)
    front = workloads.window_object(n, 0.6, 1.4, material(0.3), x0=float(rng.uniform(-0.4, 0.0)), y0=-0.1)
    base.objects = [joined(base.objects[0], near), joined(plate, front)]
    return base


def _pool_sizes(case):
    """Triangle counts of the resident meshes: 8, log-spaced from 1000 to tri_hi."""
    return [int(n) for n in np.geomspace(min(1000, case["tri_hi"]), case["tri_hi"], 8)]


def _pool(case, seed):
    """The meshes (tori, spheres and soups by turns), the largest not always of one kind."""
    rng = np.random.default_rng(seed)
    pool = []
    for k, n in enumerate(_pool_sizes(case)):
        tex = Texture(ka=(0.1, 0.1, 0.1), kd=(0.7, 0.7, 0.7), ks=(0.2, 0.2, 0.2),
                      map_kd=workloads.noise_texture(512, rng))
        if (k + case["views"]) % 3 == 0:
            nv = max(3, int(round(math.sqrt(n / 4.0))))
            pool.append(workloads.torus_object(1.0, 0.4, max(3, int(round(n / (2.0 * nv)))), nv, tex,
                                               workloads._rotation(rng)))
        elif (k + case["views"]) % 3 == 1:
            pool.append(workloads.uv_sphere_object(1.2, n, tex, rng))
        else:
            pool.append(workloads._ball_soup(n, 1.2, tex, rng))
    return pool


def _resolution(kind, view):
    """A batch goes through its resolutions by turns; requests come in their shares (8 : 6 : 5 : 1)."""
    if kind == "batch":
        return workloads.RESOLUTIONS[view % 4]
    return workloads.SERVING_RESOLUTIONS[(0, 1, 2, 0, 1, 0, 2, 3, 0, 1, 0, 2, 0, 1, 2, 0, 1, 0, 2, 1)[view % 20]][0]


def _scenes(case, seed):
    """The frames of a case, one Scene a view."""
    kind = case["kind"]
    if kind == "torus":
        return [workloads.torus_scene(seed, case["W"], case["H"], case["power"])]
    if kind == "app":
        W, H = case["W"], case["H"]
        return [workloads.app_scene(seed, screen=(max(1920, W), max(1080, H)), canvas=(W, H), n_tri=case["n_tri"])]
    if kind == "glass":
        return [_glass_scene(seed, case["W"], case["H"], case["n_tri"])]
    if kind == "readback":
        return [workloads.soup_scene(seed, case["n_tri"], case["W"], case["H"], 512, case["power"])]
    if kind == "soup":
        s = workloads.soup_scene(seed, case["n_tri"], case["W"], case["H"], case["tex"], case["power"])
        if case["comp"] == 3:
            m = s.objects[0].textures[0]
            m.map_kd = TextureMap(m.map_kd.img[..., :3])
        return [s]
    if kind == "sphere":
        rng = np.random.default_rng(seed)
        tex = Texture(ka=(0.1, 0.1, 0.1), kd=(0.7, 0.7, 0.7), ks=(0.2, 0.2, 0.2),
                      map_kd=workloads.noise_texture(case["tex"], rng))
        obj = workloads.uv_sphere_object(1.2, case["n_tri"], tex, rng)
        return [Scene(case["W"], case["H"], workloads.random_camera(rng), (0.0, 6.0, 6.0), [obj])]
    if kind == "shells":
        return [workloads.shells_scene(seed, case["n_tri"], case["W"], case["H"], case["tex"])]
    if kind in ("batch", "serving"):
        pool, rng = _pool(case, seed), np.random.default_rng(seed)
        if kind == "batch":  # the views of a mesh follow each other
            objs = [pool[v * len(pool) // case["views"]] for v in range(case["views"])]
        else:
            objs = [pool[(5 * v + 7) % len(pool)] for v in range(case["views"])]  # any mesh, at any resolution
        return [Scene(*_resolution(kind, v), workloads.random_camera(rng), (0.0, 6.0, 6.0), [o])
                for v, o in enumerate(objs)]
    if kind == "shards":
        return [workloads.soup_scene(seed, case["n_tri"], case["W"], case["H"], 1024)]
    raise ValueError(kind)


class _Buffer:
    """Device memory of a renderer as torch sees it (it keeps the renderer alive)."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(int(ptr), False), version=2)


def _tensor(r, ptr, shape, typestr):
    return torch.as_tensor(_Buffer(r, ptr, shape, typestr), device="cuda")


def _canvas_tensors(r, canvas, W, H):
    p = [C.c_void_p() for _ in range(3)]
    r._check(r.L.dh_canvas_device_ptrs(r.ctx, canvas, *(C.byref(q) for q in p)), "dh_canvas_device_ptrs")
    out = [_tensor(r, p[0].value, (H, W), "<i4"), _tensor(r, p[1].value, (H, W), "<f4")]
    return out + [_tensor(r, p[2].value, (H, W), "<i4")] if p[2].value else out


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.kind = case["kind"]
    s.r = Renderer(0, case["tile"], case["waves"])
    s.r.winners = bool(case["winners"])
    scenes = _scenes(case, seed)
    if s.kind in ("batch", "serving"):
        s.items = [(sc, frame_uniforms(sc)) for sc in scenes]
        s.prepared = s.r.batch_views(s.items)
        s.out = [t for (_, fr), cv in zip(s.items, s.prepared[1]) for t in _canvas_tensors(s.r, cv, fr.W, fr.H)]
        return s
    s.scene = scenes[0]
    s.fr = frame_uniforms(s.scene)
    W, H = s.fr.W, s.fr.H
    if s.kind == "shards":
        s.meshes = s.r.mesh_handles(workloads.split_submission(s.scene, 2))
        s.rs = [s.r, s.r.shard_context()]
        s.n = W * H
        vis = [torch.empty(s.n, dtype=torch.int64, device="cuda") for _ in range(2)]
        s.vis = [v.data_ptr() for v in vis]
        s.cv = s.r.canvas(W, H)
        s.out = [vis[0], vis[1]] + _canvas_tensors(s.r, s.cv, W, H)
        return s
    s.meshes = s.r.mesh_handles(s.scene)
    s.cv = s.r.canvas(W, H)
    if s.kind == "readback":
        s.bgra, s.depth = np.empty((H, W, 4), np.uint8), np.empty((H, W), np.float32)
        return s
    if s.kind == "app":
        s.gui = gui.gui_drawlist(seed, W, H, n_quads=case["quads"], n_cmds=8)
        s.font = gui.font_atlas(seed)
    s.out = _canvas_tensors(s.r, s.cv, W, H)
    return s


def run(s):
    if s.kind in ("batch", "serving"):
        s.r.render_batch(s.items, graph=s.kind == "batch", prepared=s.prepared)
        return s.out
    if s.kind == "shards":
        for k in range(2):
            s.rs[k].render_shard(s.fr, s.meshes[k:k + 1], k, s.cv, s.vis[k])
        s.r.vis_merge_min(s.vis[0], s.vis[1], s.n)
        for k in range(2):
            s.rs[k].shade_shard(s.vis[0], k)
        return s.out
    s.r.render_device(s.scene, s.fr, s.meshes)
    if s.kind == "readback":
        s.r.read_into(s.cv, s.bgra, s.depth)
        return [s.bgra, s.depth]
    if s.kind == "app":
        s.r.draw_gui(s.cv, *s.gui, s.font)
    return s.out


# --------------------------------------------------------------------------------------------- work
def _frames(case):
    """(pixels, triangles, bytes of mesh data) over the views of a case, resident data that several views
    read counted for each of them."""
    kind = case["kind"]
    if kind in ("batch", "serving"):
        px = sum(w * h for w, h in (_resolution(kind, v) for v in range(case["views"])))
        tri = case["views"] * sum(_pool_sizes(case)) / 8  # views are spread evenly over the meshes
        return px, tri, tri * (36 + (96 + 16 + 16) / 3)
    px, tri = case["W"] * case["H"], case["n_tri"] + (2304 if kind in ("app", "glass") else 0)
    # index triplets, and vertices (32 bytes each: three a triangle in a soup, half a one in a grid)
    return px, tri, tri * (36 + (96 if kind in ("app", "readback", "soup", "shards") else 16))


def work(case):
    px, tri, mesh = _frames(case)
    per_px = 8 + 4 + (4 if case["winners"] else 0)  # frame and depth written, one texel read
    if case["kind"] == "readback":
        per_px += 16  # the canvas read once more and written to the host
    if case["kind"] == "app":
        per_px += 8  # the GUI's read and write of the frame
    if case["kind"] == "shards":
        per_px += 16  # the merged visibility
    # a triangle: back-face and four side tests, projection, setup, three vertices' light vectors;
    # a pixel: barycentrics, three interpolated vectors, the texel and the lighting
    return {"bytes": int(px * per_px + mesh), "flops": int(tri * 300 + px * 150)}


# ------------------------------------------------------------------------------------ 64-bit depths
def _uniforms64(s):
    """Projection matrix and view planes (near, far, right, left, top, bottom) of a scene in float64."""
    cam, W, H = s.camera, s.width, s.height
    n, f = float(np.float32(cam.near)), float(np.float32(cam.far))
    r = abs(n) * math.tan(math.radians(float(np.float32(cam.fov_x))) / 2.0)
    t = r * H / W
    pos, d = (np.asarray(np.float32(v), np.float64) for v in (cam.position, cam.direction))
    w = -d / np.linalg.norm(d)
    u = np.cross([0.0, 1.0, 0.0], w)
    u /= np.linalg.norm(u)
    v = np.cross(w, u)
    basis = np.stack([u, v, w], 1)
    view = np.eye(4)
    view[:3, :3], view[:3, 3] = basis.T, -basis.T @ pos
    persp = np.array([[n, 0, 0, 0], [0, n, 0, 0], [0, 0, n + f, -n * f], [0, 0, 1, 0]])
    orth = np.diag([1 / r, 1 / t, 2 / (n - f), 1.0])
    orth[2, 3] = -(n + f) / (n - f)
    port = np.array([[W / 2, 0, 0, (W - 1) / 2], [0, H / 2, 0, (H - 1) / 2], [0, 0, 1, 0], [0, 0, 0, 1.0]])

    def world(x, y, z):
        return basis @ np.array([x, y, z]) + pos

    urn, uln, lrn, lln = world(r, t, n), world(-r, t, n), world(r, -t, n), world(-r, -t, n)
    ucf, lcf, rcf, lfc = world(0, f * t / n, f), world(0, -f * t / n, f), world(f * r / n, 0, f), world(-f * r / n, 0, f)
    inside = (urn + lcf) / 2

    def plane(a, b, c):
        q = np.cross(b - a, c - b)
        k = -q @ a
        return np.append(q, k) if q @ inside + k >= 0 else np.append(-q, -k)

    planes = [plane(urn, lrn, lln), plane(lfc, rcf, ucf), plane(rcf, urn, lrn), plane(lfc, lln, uln),
              plane(ucf, uln, urn), plane(lcf, lln, lrn)]
    return port @ orth @ persp @ view, np.stack(planes), pos


def _clip64(v, pl):
    """Triangles (T, 3, 4: xyz and depth) against one plane, as the reference splits them."""
    f = v[..., :3] @ pl[:3] + pl[3]
    whole = (f > 0).all(1)
    cut = ~whole & (f > 0).any(1)
    w, g = v[cut], f[cut]
    r1 = g[:, 0] * g[:, 2] >= 0
    r2 = ~r1 & (g[:, 1] * g[:, 2] >= 0)
    order = torch.tensor([[0, 1, 2], [2, 0, 1], [1, 2, 0]], device=v.device)[r1.long() + 2 * r2.long()]
    w = torch.gather(w, 1, order[..., None].expand(-1, -1, 4))
    a, b, c = w[:, 0], w[:, 1], w[:, 2]

    def at(p):
        q = (p[:, :3] @ pl[:3] + pl[3]) / ((p[:, :3] - c[:, :3]) @ pl[:3]) - 1e-7
        return p + (c - p) * q[:, None]

    na, nb = at(a), at(b)
    two = (c[:, :3] @ pl[:3] + pl[3]) <= 0
    first = torch.where(two[:, None], a, c)
    return torch.cat([v[whole], torch.stack([first, na, nb], 1), torch.stack([a, b, nb], 1)[two]])


def _depth64(s):
    """The depth buffer of a scene's opaque meshes, (H, W) float64, rows bottom-up."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    M, planes, cam = (torch.from_numpy(np.ascontiguousarray(x)).to(dev) for x in _uniforms64(s))
    W, H = s.canvas_size
    depth = torch.full((W * H,), float(CLEAR_DEPTH), dtype=torch.float64, device=dev)
    for o in s.objects:
        pos = torch.from_numpy(o.vertices).to(dev).double()
        vert = torch.cat([pos, (pos - cam).norm(dim=1, keepdim=True)], 1)
        for m in o.opaque_meshes():
            v = vert[torch.from_numpy(m.triangles[:, :3].astype(np.int64)).to(dev)]
            p = v[..., :3]
            q = torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 1])
            keep = ((cam - p.mean(1)) * q).sum(1) > 0
            for k in range(2, 6):
                keep &= ((p @ planes[k, :3] + planes[k, 3]) > 0).any(1)
            v = _clip64(_clip64(v[keep], planes[0]), planes[1])
            h = v[..., :3] @ M[:, :3].T + M[:, 3]
            X = torch.floor(h[..., 0] / h[..., 3] - s.canvas_offset[0] + 0.5)
            Y = torch.floor(h[..., 1] / h[..., 3] - s.canvas_offset[1] + 0.5)
            x0, y0 = X.amin(1).clamp(min=0), Y.amin(1).clamp(min=0)
            w = (X.amax(1).clamp(max=W - 1) - x0 + 1).clamp(min=0)
            n = (w * (Y.amax(1).clamp(max=H - 1) - y0 + 1).clamp(min=0)).long()
            keep = n > 0
            X, Y, D, x0, y0, w, n = X[keep], Y[keep], v[keep][..., 3], x0[keep], y0[keep], w[keep].long(), n[keep]
            ends = n.cumsum(0)
            start = 0
            while start < len(n):  # some ten million box pixels at a time
                base = ends[start] - n[start]
                stop = max(start + 1, int(torch.searchsorted(ends, base + 10_000_000)))
                i = torch.arange(start, min(stop, len(n)), device=dev).repeat_interleave(n[start:stop])
                k = torch.arange(len(i), device=dev) + base - (ends[i] - n[i])
                x, y = x0[i] + k % w[i], y0[i] + k // w[i]
                inside, z = torch.ones_like(i, dtype=torch.bool), torch.zeros_like(x)
                for e in range(3):
                    a, b = (e + 1) % 3, (e + 2) % 3

                    def edge(px, py, j):
                        return ((Y[:, a] - Y[:, b])[j] * px + (X[:, b] - X[:, a])[j] * py + (X[:, a] * Y[:, b])[j]
                                - (X[:, b] * Y[:, a])[j])

                    f = edge(X[:, e], Y[:, e], slice(None))
                    tie = f * edge(-1.0, -1.0, slice(None)) > 0
                    g = edge(x, y, i) / f[i]
                    inside &= (g > 0) | ((g == 0) & tie[i])
                    z += g * D[i, e]
                at = (y * W + x).long()[inside]
                depth.scatter_reduce_(0, at, z[inside], "amin")
                start = stop
    return depth.reshape(H, W)


def exact(case, seed):
    scenes = _scenes(case, seed)
    ids = [None] if case["winners"] else []
    if case["kind"] == "readback":
        return [None, _depth64(scenes[0])]
    if case["kind"] == "shards":
        return [None, None, None, _depth64(scenes[0])] + ids
    out = []
    for s in scenes:
        out += [None, _depth64(s)] + ids
    return out
