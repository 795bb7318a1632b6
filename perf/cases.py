"""The work that programs give this library, as a list of measurable cases.

A case is one frame (or one differentiable depth step) of a scene, through
the public entry points: ``Renderer.tessellate / build_accel / trace`` where
the program launches its frames itself, ``tc_renderer_graph_launch`` where it
replays a captured frame, and ``diff.displaced_depth`` with autograd for the
differentiable form.  Scenes, sizes and capacities are those of the
benchmark workloads and the tests of this repository; ``draw`` spreads them
over the ranges between.

``prepare`` holds what such a program keeps between frames: the scene in
device memory, the renderer, the output buffers and, for replayed frames, the
captured graph.  The seed sets the instance layout (where rays are traced), the
height maps and the camera's place on its path.
"""
import ctypes as C
import math

import numpy as np
import torch

from vk_tessellated_clusters_amd import abi, diff, scene
from vk_tessellated_clusters_amd.device import DeviceScene, Renderer

FLAGS = {
    # displacement and instance culling, the flags of abi.default_config
    "plain": abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING,
    # the reference renderer's defaults: PN base surface, 1X and 2X transient builds
    "defaults": scene.REFERENCE_DEFAULT_FLAGS,
    # the animated surface
    "ripple": abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_ANIMATION,
    # occlusion culling against the previous frame's depth
    "hiz": abi.FLAG_DISPLACEMENT | abi.FLAG_CULLING | abi.FLAG_HIZ,
}


def listed():
    return [
        # the smallest call: one 1280-triangle mesh in a thumbnail view, frames
        # launched one by one; launches and latency are all there is to it
        dict(name="icosphere_180p", scene="icosphere", count=8, tex=512, width=320, height=180, px=8.0, flags="plain",
             graph=False, rays=True),
        # the small benchmark frame, replayed
        dict(name="icosphere_720p", scene="icosphere", count=8, tex=512, width=1280, height=720, px=8.0, flags="plain",
             graph=True, rays=True),
        # a few ragged meshes (50 quads a side: partial clusters at two edges) in an
        # odd viewport, animated, launched frame by frame
        dict(name="grid5_ragged_ripple", scene="grid", count=5, quads=50, tex=512, width=961, height=541, px=3.0,
             flags="ripple", graph=False, rays=True),
        # a mid-size field culled against its own previous frame
        dict(name="grid20_hiz_900p", scene="grid", count=20, quads=120, tex=1024, width=1600, height=900, px=4.0,
             flags="hiz", graph=True, rays=True),
        # the headline frame
        dict(name="grid64_1080p", scene="grid", count=64, quads=256, tex=2048, width=1920, height=1080, px=4.0,
             flags="plain", graph=True, rays=True),
        # the headline frame with the reference renderer's default flags
        dict(name="grid64_defaults_1080p", scene="grid", count=64, quads=256, tex=2048, width=1920, height=1080, px=4.0,
             flags="defaults", graph=True, rays=True),
        # many meshes of all sizes in one frame, each with a height map of its own
        dict(name="batched500_1080p", scene="batched", count=500, tex=1024, width=1920, height=1080, px=4.0,
             flags="plain", graph=True, rays=True),
        # the same meshes tessellated and built, for a consumer that casts rays
        # of its own later or reads the displaced vertices
        dict(name="batched500_build", scene="batched", count=500, tex=1024, width=1920, height=1080, px=4.0,
             flags="plain", graph=True, rays=False),
        # the largest frame: 16.8M base triangles at 3840 x 2160 and 2 px, a
        # camera on its spline
        dict(name="patches64_2160p", scene="patches", count=8, quads=512, tex=4096, width=3840, height=2160, px=2.0,
             flags="plain", graph=True, rays=True),
        # one step of fitting a height map to depths: forward, loss, backward
        dict(name="depth_fit_512", scene="depth", quads=64, tex=512, width=512, px=0.5),
        # the same step on a mesh that is fine enough by itself (no edge is split)
        dict(name="depth_fit_base", scene="depth", quads=64, tex=256, width=384, px=64.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _viewport(rng, lo, hi):
    w = _log_int(rng, lo, hi)
    return w, max(6, int(round(w * rng.choice((9 / 16, 10 / 16, 3 / 4)))))


def draw(rng):
    kind = rng.choice(("icosphere", "grid", "grid", "grid", "batched", "patches", "depth"))
    if kind == "depth":
        return dict(scene=kind, quads=_log_int(rng, 8, 96), tex=_log_int(rng, 64, 1024), width=_log_int(rng, 48, 768),
                    px=round(math.exp(rng.uniform(math.log(0.5), math.log(16.0))), 2))
    graph = rng.random() < 0.7
    if kind == "icosphere":
        w, h = _viewport(rng, 160, 1920)
        return dict(scene=kind, count=8 * rng.randint(1, 12), tex=_log_int(rng, 64, 1024), width=w, height=h,
                    px=round(rng.uniform(2.0, 12.0), 2), flags=rng.choice(("plain", "defaults", "ripple")), graph=graph,
                    rays=True)
    if kind == "grid":
        w, h = _viewport(rng, 240, 1920)
        return dict(scene=kind, count=_log_int(rng, 1, 90), quads=_log_int(rng, 16, 256), tex=_log_int(rng, 128, 2048),
                    width=w, height=h, px=round(rng.uniform(2.0, 10.0), 2),
                    flags=rng.choice(("plain", "plain", "defaults", "ripple", "hiz")), graph=graph,
                    rays=rng.random() < 0.85)
    if kind == "batched":
        w, h = _viewport(rng, 480, 1920)
        return dict(scene=kind, count=_log_int(rng, 20, 500), tex=_log_int(rng, 128, 1024), width=w, height=h,
                    px=round(rng.uniform(3.0, 10.0), 2), flags=rng.choice(("plain", "defaults")), graph=graph,
                    rays=rng.random() < 0.7)
    w, h = _viewport(rng, 960, 3200)
    return dict(scene=kind, count=rng.randint(2, 7), quads=2 * _log_int(rng, 60, 256), tex=_log_int(rng, 512, 4096),
                width=w, height=h, px=round(rng.uniform(2.0, 6.0), 2), flags=rng.choice(("plain", "defaults")),
                graph=graph, rays=True)


# ------------------------------------------------------------------ frames


def _host_scene(case, seed):
    """The case's scene; `seed` lays out its instances, fills its height maps
    and places its camera.  Height maps are generated on the device.  Without
    rays the layout is fixed and the height maps alone are the seed's: the
    consumer of the geometry has sized its buffers for the scene."""
    w, h, px, tex = case["width"], case["height"], case["px"], case["tex"]
    s = seed % 100003
    if not case["rays"]:
        host = _host_scene(dict(case, rays=True), 2)
        for i, t in enumerate(host.textures):
            host.textures[i] = scene.FbmTexture(t.size, 1000 * s + i, t.octaves, t.format)
        return host
    if case["scene"] == "icosphere":
        host = scene.scene_icosphere(segments=case["count"], tex_size=16, seed=s, width=w, height=h, tess_rate_pixels=px)
        host.textures = [scene.FbmTexture(tex, s, 4, abi.TEXTURE_R32_FLOAT)]
    elif case["scene"] == "grid":
        host = scene.scene_grid_instances(num_instances=case["count"], quads=case["quads"], tex_size=16, seed=s, width=w,
                                          height=h, tess_rate_pixels=px)
        host.textures = [scene.FbmTexture(tex, s, 6, abi.TEXTURE_R16_UNORM)]
    elif case["scene"] == "batched":
        host = scene.scene_batched(num_meshes=case["count"], seed=s, tex_size=tex, width=w, height=h, tess_rate_pixels=px)
    else:
        host = scene.scene_large(patches=case["count"], quads_x=case["quads"], quads_z=case["quads"] // 2, seed=s,
                                 tex_size=tex, width=w, height=h, tess_rate_pixels=px)
        host.camera.eye, host.camera.center = scene.camera_spline(s % 100, 100, *host.spline)
    return host


_STREAM = None


def _stream():
    """The program's one rendering stream (graphs need a created one)."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM


class _DeviceArray:
    """A device array of the renderer's, for torch.as_tensor; the tensor
    keeps this object and with it the renderer that owns the memory."""

    def __init__(self, renderer, addr, shape, typestr):
        self.renderer = renderer
        self.__cuda_array_interface__ = {"data": (int(addr), False), "shape": shape, "typestr": typestr, "version": 2}


def _view(renderer, addr, shape, typestr):
    t = torch.as_tensor(_DeviceArray(renderer, addr, shape, typestr), device="cuda")
    if t.numel() and t.data_ptr() != int(addr):
        raise RuntimeError("the tensor is a copy of the renderer's array")
    return t


class _Frame:
    """Scene, renderer, output buffers and (for replays) captured graph."""

    def __init__(self, case, seed):
        host = _host_scene(case, seed)
        cfg = scene.workload_config(case["scene"] == "patches", FLAGS[case["flags"]])
        self.case, self.stream = case, _stream()
        self.dscene = DeviceScene(host)
        self.r = Renderer(self.dscene, cfg)
        ripple = case["flags"] == "ripple"
        self.fc = host.frame(animation_time=(seed % 997) * 0.5 / 60.0) if ripple else host.frame()
        w, h = case["width"], case["height"]
        self.tp = None
        # counters of the frame: the first twelve words of its readback record
        self.out = {"counters": _view(self.r, self.r.bindings.readback, (12,), "<i4")}
        if case["rays"]:
            hits = torch.empty(w * h, 6, dtype=torch.float32, device="cuda")
            dec = torch.empty(w * h, 12, dtype=torch.float32, device="cuda")
            self.tp = abi.TraceParams()
            self.tp.width, self.tp.height, self.tp.flags = w, h, abi.TRACE_CULL_BACK | abi.TRACE_SHADOW
            self.tp.hits, self.tp.decoded = hits.data_ptr(), dec.data_ptr()
            hi, di = hits.view(torch.int32), dec.view(torch.int32)
            self.out.update(hit_tuv=hits[:, :3], hit_ids=hi[:, 3:], base_ids=di[:, :4], base_bary=dec[:, 4:7],
                            depth=dec[:, 7], position=dec[:, 8:11], shadowed=di[:, 11])
        else:
            # a consumer of the built geometry knows its extent from a first frame
            self.launch()
            torch.cuda.synchronize()
            rb, sb, accel = self.r.readback(), self.r.scene_building(), self.r.accel()[0]
            clas = int(sb.tempInstantiateCounter)
            self.out.update(vertices=_view(self.r, sb.genVertices, (int(rb.numGenVertices), 3), "<f4"),
                            instance_of_cluster=_view(self.r, sb.tempInstanceIDs, (clas,), "<i4"),
                            cluster_bytes=_view(self.r, sb.tempClusterSizes, (clas,), "<i4"),
                            leaves=_view(self.r, accel.blasLeafInfo, (int(sb.blasClusterCounter),), "<i8"))
        if case["graph"]:
            tp = C.byref(self.tp) if self.tp is not None else None
            abi.check(self.r.L.tc_renderer_graph_capture(self.r.handle, C.byref(self.fc), tp, self.handle()),
                      "graph capture")

    def handle(self):
        return C.c_void_p(self.stream.cuda_stream)

    def launch(self):
        self.r.tessellate(self.fc, self.stream)
        self.r.build_accel(self.stream)
        if self.tp is not None:
            self.r.trace(self.tp, self.stream)

    def run(self):
        if self.case["graph"]:
            abi.check(self.r.L.tc_renderer_graph_launch(self.r.handle, C.byref(self.fc), self.handle()), "graph launch")
        else:
            self.launch()
        return self.out


# ------------------------------------------------------- differentiable depth

EYE, SCALE = 2.0, 0.1


def _depth_inputs(case, seed):
    """Height map to fit (rough, as in the middle of a fit) and the measured
    depths of a smoother surface, both float32 on the host."""
    n, m = case["tex"], case["width"]
    rng = np.random.default_rng(seed)
    heights = scene.fbm_height(n, seed % 100003, 4).astype(np.float64) + rng.normal(0.0, 0.01, (n, n))
    c = (np.arange(m) + 0.5) / m
    x, z = np.meshgrid(c, c, indexing="xy")
    a, b, p, q = rng.uniform(0.1, 0.4), rng.uniform(0.1, 0.4), rng.integers(1, 5), rng.integers(1, 5)
    target = EYE - SCALE * (0.5 + a * np.sin(2 * math.pi * p * x) + b * np.cos(2 * math.pi * q * z))
    return heights.astype(np.float32), target.reshape(-1).astype(np.float32)


class _Depth:
    def __init__(self, case, seed):
        heights, target = _depth_inputs(case, seed)
        self.heights = torch.from_numpy(heights).cuda().requires_grad_(True)
        self.target = torch.from_numpy(target).cuda()
        self.r = diff.DepthRenderer(self.heights, quads=case["quads"], rays=case["width"], height_scale=SCALE,
                                    eye_height=EYE, tess_rate_pixels=case["px"])

    def run(self):
        depth = diff.displaced_depth(self.heights, self.r)
        loss = diff.depth_loss(depth, self.target)
        (grad,) = torch.autograd.grad(loss, self.heights)
        return {"depth": depth.detach(), "loss": loss.detach(), "grad": grad}


# ------------------------------------------------------------------ interface


def prepare(case, seed):
    return _Depth(case, seed) if case["scene"] == "depth" else _Frame(case, seed)


def run(state):
    return state.run()


def _geometry(case):
    """(bytes of the distinct geometry, displaced base vertices of a frame)."""
    def grid(qx, qz):
        v = (qx + -(-qx // 8)) * (qz + -(-qz // 8))
        return 32 * v + 6 * qx * qz, v

    n = case.get("count", 1)
    if case["scene"] == "icosphere":
        v = 20 * (n // 8) ** 2 * 45
        return 32 * v + 60 * n * n, v
    if case["scene"] == "batched":
        # counts log-uniform over 200 .. 200000 triangles, up to about 32 distinct
        # meshes, 81 vertices for 128 triangles
        mean = (200000 - 200) / math.log(1000.0)
        return int(min(n, 32) * mean * (32 * 81 / 128 + 3)), int(n * mean * 81 / 128)
    if case["scene"] == "patches":
        b, v = grid(case["quads"], case["quads"] // 2)
        return b, n * n * v
    b, v = grid(case["quads"], case["quads"])
    return b, n * v


def work(case):
    """Compulsory work of a pass: the distinct geometry and the height maps
    read once, the results written once; about 60 operations for a displaced
    vertex and 60 each to make, intersect and decode a ray."""
    geo, verts = _geometry(case)
    if case["scene"] == "depth":
        rays, texels = case["width"] ** 2, case["tex"] ** 2
        return {"bytes": geo + 8 * texels + (32 + 4 + 4) * rays, "flops": 60 * verts + 180 * rays}
    maps = case["count"] if case["scene"] == "batched" else 1
    tex = maps * case["tex"] ** 2 * (4 if case["scene"] == "icosphere" else 2)
    if not case["rays"]:
        return {"bytes": geo + tex + 12 * verts, "flops": 60 * verts}
    rays = case["width"] * case["height"]
    return {"bytes": geo + tex + 72 * rays, "flops": 60 * verts + 180 * rays}


def exact(case, seed):
    """Depths, loss and gradient in 64 bits where no edge is split: the
    surface is then the grid's own triangles with displaced corners, and a
    vertical ray's depth is linear in them.  None elsewhere (a frame's hits
    depend on tessellation decisions)."""
    if case["scene"] != "depth" or case["px"] < 32.0:
        return None
    heights, target = _depth_inputs(case, seed)
    q, n, m = case["quads"], case["tex"], case["width"]
    h = heights.astype(np.float64)
    # bilinear samples at the vertices, REPEAT, texel centres at (i + 0.5) / n
    s = np.arange(q + 1) / q * n - 0.5
    i0 = np.floor(s).astype(np.int64)
    f = s - i0
    ia, ib = i0 % n, (i0 + 1) % n
    w = np.zeros((q + 1, n))
    np.add.at(w, (np.arange(q + 1), ia), 1.0 - f)
    np.add.at(w, (np.arange(q + 1), ib), f)
    y = SCALE * (w @ h @ w.T)  # [z vertex, x vertex]
    c = (np.arange(m) + 0.5) / m * q
    j = np.minimum(c.astype(np.int64), q - 1)
    fr = c - j
    jx, jz = np.meshgrid(j, j, indexing="xy")
    fx, fz = np.meshgrid(fr, fr, indexing="xy")
    low = fx + fz <= 1.0
    # weights of the quad's corners (z, x): 00, 01, 10, 11
    w00 = np.where(low, 1.0 - fx - fz, 0.0)
    w01 = np.where(low, fx, 1.0 - fz)
    w10 = np.where(low, fz, 1.0 - fx)
    w11 = np.where(low, 0.0, fx + fz - 1.0)
    depth = EYE - (w00 * y[jz, jx] + w01 * y[jz, jx + 1] + w10 * y[jz + 1, jx] + w11 * y[jz + 1, jx + 1])
    d = depth.reshape(-1) - target.astype(np.float64)
    loss = float((d ** 2).sum() / d.size)
    g = -SCALE * (2.0 * d / d.size).reshape(m, m)
    gy = np.zeros((q + 1, q + 1))
    for wk, dz, dx in ((w00, 0, 0), (w01, 0, 1), (w10, 1, 0), (w11, 1, 1)):
        np.add.at(gy, (jz + dz, jx + dx), g * wk)
    return {"depth": depth.reshape(-1), "loss": np.float64(loss), "grad": w.T @ gy @ w}
