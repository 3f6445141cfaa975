"""The framework's measured workloads.

Each case is one call pattern of a program that uses the C ABI through restirpt.py:

  frame   one rendered frame of a camera walk: G-buffer, a direct method, an indirect method and, where the
          program shows the image, post-processing. History (previous G-buffer and reservoirs) is in hand.
  batch   one rt_batch_frame over independent square views of two scenes
  rays    ray queries over device arrays (rt_trace_rays)
  bvh     the LBVH of geometry that moves every frame (rt_bvh_build_noalloc)
  scene   loading: host arrays to a device scene with its acceleration structure, and the first G-buffer
  infer   the radiance network at many positions (rt_mlp_infer)
  train   one online training step of it (rt_mlp_train_step) and the updated network's predictions
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vulkan-restir-pt_amd"))
import restirpt as rt  # noqa: E402

# triangles of the procedural scenes (rt_scenegen) that the cases use
TRIANGLES = {0: 20506, 1: 1112592, 3: 224016}
WALK = 16  # frames of the camera walk that a state holds
NETWORK_LO, NETWORK_HI = (-12.0, -12.0, -2.0), (12.0, 12.0, 6.0)


def _frame(name, scene, width, height, **kw):
    c = dict(name=name, kind="frame", scene=scene, width=width, height=height, direct=0, indirect=0, depth=6, shift=2,
             temporal=True, spatial=True, neighbors=3, radius=20.0, learned=False, unbiased=False, guided=False,
             di_shift=0, di_sample=0, di_temporal=False, post=False)
    c.update(kw)
    return c


def listed():
    return [
        # a preview or test render: launches and latency, hardly any work
        _frame("gris_64", 0, 64, 64, indirect=3, depth=4),
        # ReSTIR PT at full HD, hybrid shift, both reuses: the benchmark's own frame
        _frame("gris_1080p", 1, 1920, 1080, indirect=3),
        # every learned and unbiased option at once (target, proposal, 1/Z weights), an odd window size
        _frame("full_form_853x481", 3, 853, 481, indirect=3, depth=8, radius=30.0, learned=True, unbiased=True,
               guided=True),
        # the reference's two naive estimators at thumbnail size
        _frame("plain_256", 0, 256, 256, direct=1, indirect=1, depth=4),
        # ReSTIR DI with the reference's defaults at full HD
        _frame("di_1080p", 1, 1920, 1080, direct=2),
        # the whole image a viewer shows: ReSTIR DI (temporal, both sample types) + ReSTIR GI + tone mapping
        _frame("image_1365x767", 3, 1365, 767, direct=2, indirect=2, di_sample=2, di_temporal=True, post=True),
        # a serving batch: 16 cameras of ragged sizes over two scenes
        dict(name="batch_16", kind="batch", views=16, low=96, high=512, mix=5),
        # another program's own ray queries against a loaded scene
        dict(name="rays_closest_1m", kind="rays", scene=1, rays=1000003, mode=0, skip_lights=False),
        # dynamic geometry: the tree rebuilt from device triangles inside a frame
        dict(name="bvh_rebuild_100k", kind="bvh", triangles=100003),
        # loading a scene of ordinary size
        dict(name="scene_load_224k", kind="scene", scene=3, width=640, height=360),
        # the network alone: predictions at 300k points, and the largest training batch
        dict(name="infer_300k", kind="infer", points=300007, log2_table=19),
        dict(name="train_65536", kind="train", points=65536, log2_table=19),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame"] * 6 + ["batch", "rays", "rays", "bvh", "scene", "infer", "train"])
    if kind == "frame":
        scene = rng.choice([0, 1, 3])
        method = rng.choice(["pt", "pt", "pt_unbiased", "full", "naive", "di", "image"])
        most = {"pt": 1 << 21, "pt_unbiased": 1 << 20, "full": 1 << 19, "naive": 1 << 18, "di": 1 << 20,
                "image": 1 << 20}[method]
        pixels, aspect = _log(rng, 48 * 48, most), rng.uniform(0.8, 2.0)
        width = max(24, int(math.sqrt(pixels * aspect)))
        c = _frame("", scene, width, max(24, pixels // width), depth=rng.randint(3, 8))
        c.pop("name")
        if method in ("pt", "pt_unbiased", "full"):
            c.update(indirect=3, shift=rng.choice([0, 1, 2, 2]), temporal=rng.random() < 0.7, radius=rng.choice([20.0, 30.0]),
                     neighbors=rng.randint(1, 3), unbiased=method != "pt")
            if method == "full":
                c.update(shift=2, temporal=True, learned=True, guided=True)
        elif method == "naive":
            c.update(direct=1, indirect=1)
        else:
            c.update(direct=2, di_shift=rng.choice([0, 0, 1]) if method == "di" else 0, di_sample=rng.randint(0, 2),
                     di_temporal=rng.random() < 0.5)
            if method == "image":
                c.update(indirect=rng.choice([1, 2]), post=True, depth=4)
        return c
    if kind == "batch":
        return dict(kind="batch", views=rng.randint(2, 16), low=64, high=rng.randint(160, 512), mix=rng.randint(0, 1 << 20))
    if kind == "rays":
        return dict(kind="rays", scene=rng.choice([0, 1, 3]), rays=_log(rng, 1000, 1000000), mode=rng.randint(0, 1),
                    skip_lights=rng.random() < 0.3)
    if kind == "bvh":
        return dict(kind="bvh", triangles=_log(rng, 200, 131072))
    if kind == "scene":
        return dict(kind="scene", scene=rng.choice([0, 3]), width=rng.randint(64, 700), height=rng.randint(64, 400))
    return dict(kind=kind, points=_log(rng, 1000, 300000 if kind == "infer" else 65536), log2_table=rng.choice([15, 17, 19]))


# ---- states -----------------------------------------------------------------------------------------


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _zeros(nbytes):
    return torch.zeros(max(16, nbytes), dtype=torch.uint8, device="cuda")


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed & 0x7FFFFFFF)
    return g


def _batch_sizes(case):
    g = np.random.default_rng(case["mix"])
    return [int(v) for v in np.exp(g.uniform(np.log(case["low"]), np.log(case["high"] + 1), case["views"]))]


def _camera_frames(host, width, height):
    return [host.camera(k, width, height) for k in range(WALK)]


class _View:
    """One view's images and reservoirs, as rt_frame binds them for either parity."""

    def __init__(self, scene, width, height, gris, di=False, gi=False, guided=False):
        L, n = rt.core(), width * height
        self.scene, self.width, self.height, self.parity = scene, width, height, 0
        self.depth_normal = [_zeros(16 * n) for _ in range(2)]
        self.albedo_mat = [_zeros(8 * n) for _ in range(2)]
        self.motion = _zeros(4 * n)
        self.direct, self.indirect = _zeros(16 * n), _zeros(16 * n)

        def reservoirs(count, name):
            size = getattr(L, f"rt_{name}_reservoir_bytes")(width, height)
            got = [_zeros(size) for _ in range(count)]
            for b in got:
                rt.check(getattr(L, f"rt_{name}_reservoir_reset")(b.data_ptr(), width, height, _stream()), "reset")
            return got

        self.gris = reservoirs(3, "gris") if gris else []
        self.di = reservoirs(3, "di") if di else []
        self.gi = reservoirs(2, "gi") if gi else []
        lobes = L.rt_guide_lobe_bytes(width, height) if guided else 0
        self.lobes = [_zeros(lobes) for _ in range(2)] if guided else []
        self.samples = _zeros(16 * n) if guided else None
        self.frames = [self._bind(p) for p in range(2)]

    def _bind(self, c):
        l, f = c ^ 1, rt.Frame()
        f.width, f.height = self.width, self.height
        f.directOutput, f.indirectOutput = self.direct.data_ptr(), self.indirect.data_ptr()
        f.depthNormal, f.depthNormalPrev = self.depth_normal[c].data_ptr(), self.depth_normal[l].data_ptr()
        f.albedoMatId, f.albedoMatIdPrev = self.albedo_mat[c].data_ptr(), self.albedo_mat[l].data_ptr()
        f.motionVector = self.motion.data_ptr()
        if self.gris:
            f.grisReservoir, f.grisReservoirPrev = self.gris[c].data_ptr(), self.gris[l].data_ptr()
            f.grisReservoirTemp = self.gris[2].data_ptr()
        if self.lobes:
            f.guideLobes, f.guideLobesPrev = self.lobes[c].data_ptr(), self.lobes[l].data_ptr()
            f.guideSamples = self.samples.data_ptr()
        return f

    def images(self, c):
        """The frame of parity c: floats as floats, packed words and reservoirs as whole numbers."""
        size = (self.height, self.width)
        got = {"depth_normal": self.depth_normal[c].view(torch.float32).view(*size, 4),
               "albedo_mat": self.albedo_mat[c].view(torch.int32).view(*size, 2),
               "motion": self.motion.view(torch.int32).view(*size)}
        if self.gris:
            got["gris"] = self.gris[c].view(torch.int32)
        if self.di:
            got["di"] = self.di[c].view(torch.int32)
        if self.gi:
            got["gi"] = self.gi[c].view(torch.int32)
        return got


def _network(log2_table, seed, guide=False):
    return rt.Mlp(rt.mlp_config(NETWORK_LO, NETWORK_HI, log2_table=log2_table, seed=seed & 0xFFFF), guide=guide)


class _FrameState:
    def __init__(self, case, seed):
        self.case = case
        self.host = rt.HostScene(case["scene"], seed & 0xFFFFFF)
        self.scene = rt.DeviceScene(self.host.arrays)
        w, h = case["width"], case["height"]
        self.view = _View(self.scene, w, h, gris=case["indirect"] == 3, di=case["direct"] == 2, gi=case["indirect"] == 2,
                          guided=case["guided"])
        self.settings = rt.settings(shift=case["shift"], temporal=case["temporal"], spatial=case["spatial"], cap=20,
                                    max_depth=case["depth"], neighbors=case["neighbors"], radius=case["radius"],
                                    learned=case["learned"], unbiased=case["unbiased"], guided=case["guided"])
        self.di_settings = rt.di_settings(shift=case["di_shift"], sample=case["di_sample"],
                                          temporal=case["di_temporal"])
        self.post = rt.PostSettings(1, 1, int(case["direct"] == 0), int(case["indirect"] == 0))
        self.rgba = _zeros(4 * w * h) if case["post"] else None
        self.target = _network(19, seed) if case["learned"] else None
        self.guide = _network(19, seed + 1, guide=True) if case["guided"] else None
        self.cameras = _camera_frames(self.host, w, h)
        self.frame = 0
        self.draw()  # the history that a walk's later frames find

    def draw(self):
        L, st, case, v = rt.core(), _stream(), self.case, self.view
        scene, cams, f = self.scene.handle, self.cameras[self.frame % WALK], v.frames[v.parity]
        rt.check(L.rt_gbuffer_trace(scene, C.byref(cams[0]), f.depthNormal, f.albedoMatId, f.motionVector, st), "G-buffer")
        c = v.parity
        if case["direct"] == 2:
            r = rt.DIReservoirs(v.di[c].data_ptr(), v.di[c ^ 1].data_ptr(), v.di[2].data_ptr())
            rt.check(L.rt_di_render(scene, cams, C.byref(f), C.byref(r), C.byref(self.di_settings), st), "ReSTIR DI")
        naive = (1 if case["direct"] == 1 else 0) | (2 if case["indirect"] == 1 else 0)
        if naive:
            rt.check(L.rt_pt_plain(scene, cams, C.byref(f), case["depth"], naive, st), "plain path tracer")
        if case["indirect"] == 2:
            r = rt.GIReservoirs(v.gi[c].data_ptr(), v.gi[c ^ 1].data_ptr())
            rt.check(L.rt_gi_temporal(scene, cams, C.byref(f), C.byref(r), st), "ReSTIR GI")
        if case["indirect"] == 3 and not (case["learned"] or case["guided"]):
            rt.check(L.rt_gris_render(scene, cams, C.byref(f), C.byref(self.settings), st), "ReSTIR PT")
        elif case["indirect"] == 3:
            s = C.byref(self.settings)
            if self.guide:
                rt.check(L.rt_gris_guide_refresh(scene, self.guide.handle, cams, C.byref(f), st), "proposal refresh")
            rt.check(L.rt_gris_path_trace(scene, cams, C.byref(f), s, st), "path trace")
            if self.target:
                rt.check(L.rt_gris_learned_refresh(scene, self.target.handle, cams, C.byref(f), st), "target refresh")
            rt.check(L.rt_gris_temporal(scene, cams, C.byref(f), s, st), "temporal reuse")
            rt.check(L.rt_gris_spatial(scene, cams, C.byref(f), s, st), "spatial reuse")
            if self.target:
                rt.check(L.rt_mlp_train_frame(self.target.handle, None, st), "target training")
            if self.guide:
                rt.check(L.rt_gris_guide_train(scene, self.guide.handle, cams, C.byref(f), None, st), "proposal training")
        if self.rgba is not None:
            rt.check(L.rt_post_process(C.byref(f), C.byref(self.post), self.rgba.data_ptr(), st), "post-processing")
        v.parity ^= 1
        self.frame += 1
        return c

    def run(self):
        c = self.draw()
        size = (self.case["height"], self.case["width"], 4)
        got = self.view.images(c)
        if self.case["direct"]:
            got["direct"] = self.view.direct.view(torch.float32).view(size)
        if self.case["indirect"]:
            got["indirect"] = self.view.indirect.view(torch.float32).view(size)
        if self.rgba is not None:
            got["rgba"] = self.rgba.view(size)
        if self.view.lobes:
            got["lobes"] = self.view.lobes[c].view(torch.int32)
            got["samples"] = self.view.samples.view(torch.float32)
        return got


class _BatchState:
    def __init__(self, case, seed):
        self.hosts = [rt.HostScene(0, seed & 0xFFFFFF), rt.HostScene(3, seed & 0xFFFFFF)]
        self.scenes = [rt.DeviceScene(h.arrays) for h in self.hosts]
        g = np.random.default_rng(seed)
        self.sizes = _batch_sizes(case)
        self.views, self.settings, self.cameras, self.starts = [], [], [], []
        for i, n in enumerate(self.sizes):
            self.views.append(_View(self.scenes[i % 2], n, n, gris=True))
            self.settings.append(rt.settings(shift=2, temporal=True, spatial=True, cap=20, max_depth=3 + i % 6,
                                             neighbors=3, radius=20.0))
            self.cameras.append(_camera_frames(self.hosts[i % 2], n, n))
            self.starts.append(int(g.integers(0, WALK)))
        self.array = (rt.View * len(self.sizes))()
        for i, v in enumerate(self.views):
            self.array[i].scene, self.array[i].settings = v.scene.handle.value, self.settings[i]
        self.batch = C.c_void_p()
        rt.check(rt.core().rt_batch_create(len(self.sizes), C.byref(self.batch)), "batch")
        self.frame = 0
        self.draw()

    def __del__(self):
        if getattr(self, "batch", None):
            rt.core().rt_batch_destroy(self.batch)

    def draw(self):
        for i, v in enumerate(self.views):
            cams = self.cameras[i][(self.starts[i] + self.frame) % WALK]
            C.memmove(C.addressof(self.array[i].cams), C.addressof(cams), C.sizeof(cams))
            self.array[i].frame = v.frames[v.parity]
        rt.check(rt.core().rt_batch_frame(self.batch, self.array, len(self.views), _stream()), "batched frame")
        for v in self.views:
            v.parity ^= 1
        self.frame += 1

    def run(self):
        self.draw()
        got = []
        for v in self.views:
            c = v.parity ^ 1
            got.append({"gris": v.gris[c].view(torch.int32),
                        "indirect": v.indirect.view(torch.float32).view(v.height, v.width, 4),
                        "depth_normal": v.depth_normal[c].view(torch.float32).view(v.height, v.width, 4)})
        return got


class _RayState:
    def __init__(self, case, seed):
        self.case = case
        self.host = rt.HostScene(case["scene"], seed & 0xFFFFFF)
        self.scene = rt.DeviceScene(self.host.arrays)
        self.rays, n = _rays(case, seed, self.host), case["rays"]
        self.t = torch.zeros(n, dtype=torch.float32, device="cuda")
        self.bary = torch.zeros((n, 2), dtype=torch.float32, device="cuda")
        self.inst = torch.zeros(n, dtype=torch.int32, device="cuda")
        self.prim = torch.zeros(n, dtype=torch.int32, device="cuda")

    def run(self):
        rt.check(rt.core().rt_trace_rays(self.scene.handle, self.rays.data_ptr(), self.case["rays"], self.case["mode"],
                                         int(self.case["skip_lights"]), self.t.data_ptr(), self.bary.data_ptr(),
                                         self.inst.data_ptr(), self.prim.data_ptr(), _stream()), "trace rays")
        return {"t": self.t, "bary": self.bary, "inst": self.inst, "prim": self.prim}


def _world_triangles(host):
    """(n, 3, 3) world-space corners of the scene's object triangles, in 64 bits."""
    a = host.numpy()
    pos, idx, out = a["vertices"]["pos"].astype(np.float64), a["indices"], []
    for inst in a["instances"]:
        m = np.asarray(inst["transform"], np.float64).reshape(4, 4).T
        p = pos[idx[inst["indexOffset"]:inst["indexOffset"] + inst["indexCount"]]]
        out.append((p @ m[:3, :3].T + m[:3, 3]).reshape(-1, 3, 3))
    return np.concatenate(out)


def _light_triangles(host):
    li = host.numpy()["lights"]
    return np.stack([li["v0"], li["v1"], li["v2"]], 1).astype(np.float64)


def _rays(case, seed, host):
    """Origins over the scene's volume, directions over the sphere: what a probe or baking pass sends."""
    corners = _world_triangles(host).reshape(-1, 3)
    lo = torch.tensor(corners.min(0), dtype=torch.float32, device="cuda")
    hi = torch.tensor(corners.max(0), dtype=torch.float32, device="cuda")
    g, n = _generator(seed), case["rays"]
    o = lo + (hi - lo) * (0.02 + 0.96 * torch.rand((n, 3), generator=g, device="cuda"))
    d = torch.randn((n, 3), generator=g, device="cuda")
    d = d / d.norm(dim=1, keepdim=True)
    tmax = torch.full((n, 1), 1e7, device="cuda") if case["mode"] == 0 else \
        0.25 * (hi - lo).max() * torch.rand((n, 1), generator=g, device="cuda")
    return torch.cat([o, d, torch.full((n, 1), 1e-4, device="cuda"), tmax], 1).contiguous()


class _BvhState:
    """A waving sheet of triangles, three float4 each, as an animation writes them on the device."""

    def __init__(self, case, seed):
        n, g = case["triangles"], _generator(seed)
        side = int(math.ceil(math.sqrt(n / 2)))
        k = torch.arange(n, device="cuda")
        cell, half = k // 2, k % 2
        x, y = (cell % side).float(), (cell // side).float()
        phase = 6.2831853 * torch.rand(4, generator=g, device="cuda")

        def corner(dx, dy):
            u, v = (x + dx) / side, (y + dy) / side
            z = 0.05 * torch.sin(19 * u + phase[0]) * torch.cos(23 * v + phase[1]) + 0.01 * torch.sin(150 * u * v + phase[2])
            return torch.stack([10 * u, 10 * v, 10 * z], 1)

        low = half == 0
        v = [corner(0, 0), torch.where(low[:, None], corner(1, 0), corner(1, 1)),
             torch.where(low[:, None], corner(1, 1), corner(0, 1))]
        self.tris = torch.zeros((n, 3, 4), dtype=torch.float32, device="cuda")
        for c in range(3):
            self.tris[:, c, :3] = v[c]
        words = self.tris.view(torch.int32)
        words[:, 0, 3] = 1
        words[:, 1, 3] = k.to(torch.int32)
        self.n = n
        self.codes = torch.zeros(n, dtype=torch.int64, device="cuda")
        self.order = torch.zeros(n, dtype=torch.int32, device="cuda")
        self.nodes = torch.zeros((max(n - 1, 1), 16), dtype=torch.int32, device="cuda")

    def run(self):
        rt.check(rt.core().rt_bvh_build_noalloc(self.tris.data_ptr(), self.n, self.codes.data_ptr(), self.order.data_ptr(),
                                                self.nodes.data_ptr(), _stream()), "LBVH")
        return {"codes": self.codes, "order": self.order, "nodes": self.nodes}


class _SceneState:
    def __init__(self, case, seed):
        self.case = case
        self.host = rt.HostScene(case["scene"], seed & 0xFFFFFF)
        self.camera = self.host.camera(0, case["width"], case["height"])
        self.scene = None

    def run(self):
        w, h = self.case["width"], self.case["height"]
        self.scene = rt.DeviceScene(self.host.arrays, _stream())
        v = _View(self.scene, w, h, gris=False)
        f = v.frames[0]
        rt.check(rt.core().rt_gbuffer_trace(self.scene.handle, C.byref(self.camera[0]), f.depthNormal, f.albedoMatId,
                                            f.motionVector, _stream()), "G-buffer")
        i = self.scene.info()
        tree = np.array([i.numPrimitives, i.numLights, i.bvhNodes, i.bvhDepth, i.bvh4Nodes, i.bvh4Depth], np.int64)
        return dict(v.images(0), tree=tree, box=np.array([*i.sceneLo, *i.sceneHi], np.float32))


def _network_parameters(case, seed):
    """A network in mid-training: grid features of some tenths, weights of a Glorot start."""
    g = _generator(seed)
    u = lambda n, s: (2 * torch.rand(n, generator=g, device="cuda") - 1) * s  # noqa: E731
    grid = u(16 * 2 * (1 << case["log2_table"]), 0.3)
    weights = torch.cat([u(32 * 64, math.sqrt(6 / 96)), u(64 * 64, math.sqrt(6 / 128)), u(64 * 3, math.sqrt(6 / 67))])
    return grid, weights


def _network_points(case, seed):
    """Points on a rolling ground with objects on it, as reconnection vertices lie, and their radiance."""
    g, n = _generator(seed + 7919), case["points"]
    xy = 19.2 * torch.rand((n, 2), generator=g, device="cuda") - 9.6
    z = torch.sin(0.7 * xy[:, 0]) * torch.cos(0.5 * xy[:, 1]) + 0.4 * torch.rand(n, generator=g, device="cuda") ** 4
    pos = torch.cat([xy, z[:, None]], 1).contiguous()
    base = torch.exp(1.5 * torch.sin(xy[:, :1] * torch.tensor([0.9, 1.0, 1.1], device="cuda") + xy[:, 1:]))
    target = base * torch.exp(0.5 * torch.randn((n, 1), generator=g, device="cuda"))
    return pos, target.contiguous()


class _NetworkState:
    def __init__(self, case, seed):
        self.case = case
        self.net = _network(case["log2_table"], seed)
        grid, weights = _network_parameters(case, seed)
        self.net.set_params(grid.cpu().numpy(), weights.cpu().numpy())
        self.pos, self.target = _network_points(case, seed)
        self.rgb = torch.zeros_like(self.pos)
        self.loss = torch.zeros(1, dtype=torch.float32, device="cuda")
        self.weights = np.zeros(self.net.weight_params, np.float32)

    def run(self):
        L, n, st = rt.core(), self.case["points"], _stream()
        got = {"rgb": self.rgb}
        if self.case["kind"] == "train":
            rt.check(L.rt_mlp_train_step(self.net.handle, self.pos.data_ptr(), self.target.data_ptr(), n,
                                         self.loss.data_ptr(), st), "training step")
            got["loss"] = self.loss
        rt.check(L.rt_mlp_infer(self.net.handle, self.pos.data_ptr(), n, self.rgb.data_ptr(), st), "inference")
        if self.case["kind"] == "train":  # the updated layers, which a checkpoint keeps; the grid shows in rgb
            rt.check(L.rt_mlp_get_params(self.net.handle, None, self.weights.ctypes.data), "weights")
            got["weights"] = self.weights
        return got


STATES = {"frame": _FrameState, "batch": _BatchState, "rays": _RayState, "bvh": _BvhState, "scene": _SceneState,
          "infer": _NetworkState, "train": _NetworkState}


def prepare(case, seed):
    return STATES[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---- what a case cannot do without --------------------------------------------------------------------


def _ray_flops(triangles):
    """One ray: a box test of about 18 operations per child down a four-wide tree, two triangle tests, shading."""
    return 4 * 18 * max(1.0, math.log(max(triangles, 4), 4)) + 2 * 60 + 100


def _frame_work(pixels, triangles, case):
    """Per pixel: images and reservoirs read and written once; rays of the methods that run."""
    size, rays = 28, 1.0  # the G-buffer written, its primary ray
    if case["direct"] == 1:
        size, rays = size + 24 + 16, rays + 2
    if case["direct"] == 2:
        size, rays = size + 24 + 64 + 16 + (64 + 28 if case["di_temporal"] else 0), rays + 2 + 11 + (1 if case["di_temporal"] else 0)
    if case["indirect"] == 1:
        size, rays = size + 24 + 16, rays + 2 * min(case["depth"], 3)
    if case["indirect"] == 2:
        size, rays = size + 24 + 28 + 48 + 48 + 16, rays + 2 * 3 + 1
    if case["indirect"] == 3:
        size, rays = size + 24 + 80 + 16 + (80 + 28 if case["temporal"] else 0), rays + 2 * min(case["depth"], 3) + 1 + case["neighbors"]
        size += 16 if case["learned"] else 0
        size += 64 + 16 if case["guided"] else 0
    if case["post"]:
        size += 4
    return {"bytes": pixels * size + 48 * triangles, "flops": pixels * rays * _ray_flops(triangles)}


def _network_flops(points):
    return points * (2 * (32 * 64 + 64 * 64 + 64 * 3) + 16 * 8 * 10)


def work(case):
    kind = case["kind"]
    if kind == "frame":
        return _frame_work(case["width"] * case["height"], TRIANGLES[case["scene"]], case)
    if kind == "batch":
        one = _frame("", 0, 1, 1, indirect=3, depth=5)
        pixels = sum(n * n for n in _batch_sizes(case))
        return _frame_work(pixels, TRIANGLES[0] + TRIANGLES[3], one)
    if kind == "rays":
        n = case["rays"]
        return {"bytes": (32 + 20) * n + 48 * TRIANGLES[case["scene"]], "flops": n * _ray_flops(TRIANGLES[case["scene"]])}
    if kind == "bvh":
        n = case["triangles"]
        return {"bytes": n * (48 + 8 + 4 + 64), "flops": n * (60 + 20 * math.log2(max(n, 2)))}
    if kind == "scene":
        n = TRIANGLES[case["scene"]]
        return {"bytes": n * (12 + 4 + 16 + 48 + 48) + 28 * case["width"] * case["height"],
                "flops": n * (60 + 20 * math.log2(n)) + case["width"] * case["height"] * _ray_flops(n)}
    n, table = case["points"], 1 << case["log2_table"]
    features = 16 * min(table, 8 * n) * 4
    if kind == "infer":
        return {"bytes": 24 * n + features, "flops": _network_flops(n)}
    return {"bytes": 36 * n + features * 9, "flops": 4 * _network_flops(n)}


def tolerance(case):
    # Rendering is specified operation by operation (no contraction, correctly rounded division and square
    # root, a fixed traversal order), so images, reservoirs and trees are the same bit for bit.
    if case["kind"] not in ("infer", "train"):
        return "exact"
    # FP16 activations and weights with 32-bit sums: 2e-5 from the 64-bit value on these networks.
    if case["kind"] == "infer":
        return {"rel": 8e-5, "max": 4e-3}
    # Adam's first steps move a parameter by the sign of its gradient, so the smallest gradients' rounding shows
    # after the step: up to 3e-3 from the 64-bit weights, 5e-4 from its predictions.
    return {"rel": 1.3e-2, "max": 0.3}


# ---- the same in 64 bits -------------------------------------------------------------------------------


def _exact_rays(case, seed):
    host = rt.HostScene(case["scene"], seed & 0xFFFFFF)
    rays = _rays(case, seed, host).double()
    tris = _world_triangles(host)
    if not case["skip_lights"]:
        tris = np.concatenate([tris, _light_triangles(host)])
    tris = torch.from_numpy(tris).cuda()
    v0, e1, e2 = tris[:, 0], tris[:, 1] - tris[:, 0], tris[:, 2] - tris[:, 0]
    normal = torch.cross(e1, e2, dim=1)
    out = []
    for part in rays.split(1024):
        o, d = part[:, :3], part[:, 3:6]
        det = -(d @ normal.T)
        # with s = o - v0: t = s.n / det, u = e2 . (s x d) / det, v = -e1 . (s x d) / det
        on = o @ normal.T - (v0 * normal).sum(1)
        od = torch.cross(o, d, dim=1)
        u = (od @ e2.T - _triple(v0, d, e2)) / det
        v = (_triple(v0, d, e1) - od @ e1.T) / det
        t = on / det
        hit = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= part[:, 6:7]) & (t < part[:, 7:8])
        out.append(torch.where(hit, t, torch.inf).amin(1))
    t = torch.cat(out)
    return {"t": torch.where(torch.isinf(t), 0.0, t), "bary": None, "inst": None, "prim": None}


def _triple(v0, d, e):
    """(v0 x d) . e for every ray direction and triangle: d . (e x v0)."""
    return d @ torch.cross(e, v0, dim=1).T


class _Network64:
    """The hash-grid network in 64 bits, its parameters as the device holds them (rounded to FP16)."""

    def __init__(self, case, seed):
        grid, weights = _network_parameters(case, seed)
        self.table = 1 << case["log2_table"]
        self.master = [grid.double(), weights.double()]
        b = math.exp((math.log(2048) - math.log(16)) / 15)
        self.res = [int(math.floor(16 * b ** level + 1e-9)) for level in range(16)]

    @staticmethod
    def half(p):
        return p.float().half().double()

    def forward(self, grid, weights, pos):
        lo = torch.tensor(NETWORK_LO, dtype=torch.float64, device="cuda")
        hi = torch.tensor(NETWORK_HI, dtype=torch.float64, device="cuda")
        unit = ((pos.double() - lo) / (hi - lo)).clamp(0, 1)
        feats, table = [], grid.view(16, self.table, 2)
        for level, n in enumerate(self.res):
            x = unit * n
            c = torch.minimum(torch.floor(x), torch.tensor(n - 1.0, dtype=torch.float64, device="cuda"))
            f, c, acc = x - c, c.long(), 0
            for k in range(8):
                bit = [(k >> a) & 1 for a in range(3)]
                p = [c[:, a] + bit[a] for a in range(3)]
                if (n + 1) ** 3 <= self.table:
                    slot = p[0] + (n + 1) * (p[1] + (n + 1) * p[2])
                else:
                    slot = (p[0] ^ (p[1] * 2654435761) ^ (p[2] * 805459861)) & (self.table - 1)
                w = 1
                for a in range(3):
                    w = w * (f[:, a] if bit[a] else 1 - f[:, a])
                acc = acc + w[:, None] * table[level][slot]
            feats.append(acc)
        h = torch.cat(feats, 1)
        h = torch.relu(h @ weights[:2048].view(32, 64))
        h = torch.relu(h @ weights[2048:6144].view(64, 64))
        return torch.exp((h @ weights[6144:].view(64, 3)).clamp(-20, 20))


def _exact_network(case, seed):
    net = _Network64(case, seed)
    pos, target = _network_points(case, seed)
    grid, weights = (net.half(p) for p in net.master)
    if case["kind"] == "infer":
        return {"rgb": torch.cat([net.forward(grid, weights, p) for p in pos.split(1 << 16)])}
    grid.requires_grad_(True)
    weights.requires_grad_(True)
    y = net.forward(grid, weights, pos)
    loss = ((y - target.double()) ** 2 / (y.detach() ** 2 + 0.01)).mean()
    loss.backward()
    # first Adam step: the moments' bias corrections leave g / |g|
    moved = [p - 1e-2 * g / (g.abs() + 1e-15) for p, g in zip(net.master, (grid.grad, weights.grad))]
    with torch.no_grad():
        return {"rgb": net.forward(*(net.half(p) for p in moved), pos), "loss": loss.detach().view(1),
                "weights": moved[1]}


def exact(case, seed):
    if case["kind"] in ("infer", "train"):
        return _exact_network(case, seed)
    # brute force over every triangle; the larger scenes would take minutes
    if case["kind"] == "rays" and case["mode"] == 0 and case["scene"] == 0:
        return _exact_rays(case, seed)
    # a path, a reservoir or a tree is a chain of discrete choices on 32-bit values: it has no 64-bit value
    return None
