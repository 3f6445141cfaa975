"""Ray queries where the traversal's stack, its slab test and its wave-level scheduling can go wrong, bit for bit
against the oracle: overlapping triangles that overflow the LDS part of the stack, directions with zero
components starting on box planes (0 * inf in the slab test), trees of one to a few leaves, ray counts around the
wave size, entry distances that are zero or negative (tmin <= 0)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuhelp  # noqa: E402
import orc  # noqa: E402

rt = gpuhelp.rt


def light_scene(tris):
    """A scene whose primitives are the given triangles (n, 3, 3), all of them emitters."""
    n = len(tris)
    keep = {"mat": rt.Material(), "lights": (rt.TriangleLight * n)(), "table": (rt.LightTableEntry * (n + 1))()}
    keep["mat"].type, keep["mat"].textureIdx = 1, 0xFFFFFFFF
    for i, t in enumerate(tris):
        li = keep["lights"][i]
        li.v0, li.v1, li.v2 = ((C.c_float * 3)(*map(float, v)) for v in t)
        li.nz, li.area = 1.0, 1.0
    keep["table"][0].prob, keep["table"][0].failId = float(n), n
    for i in range(1, n + 1):
        keep["table"][i].prob, keep["table"][i].failId = 1.0, i
    a = rt.SceneArrays()
    a.materials, a.numMaterials = C.addressof(keep["mat"]), 1
    a.lights, a.numLights = C.addressof(keep["lights"]), n
    a.lightTable, a.numLightTable = C.addressof(keep["table"]), n + 1
    return a, keep


def check(arrays, rays, skip=False):
    ds, osc = rt.DeviceScene(arrays), orc.OracleScene(arrays)
    for mode in (0, 1):
        t, bary, inst, prim = gpuhelp.gpu_trace(ds, rays, mode, skip)
        ot, obary, oinst, oprim, _ = osc.trace(rays, mode, skip)
        assert np.array_equal(inst, oinst), f"mode {mode}: hit instance differs"
        if mode == 0:
            assert np.array_equal(prim, oprim)
            assert np.array_equal(t.view(np.uint32), ot.view(np.uint32))
            assert np.array_equal(bary.view(np.uint32), obary.view(np.uint32))


def aligned_rays(points, seed, tmin=1e-4):
    """Rays from the given points along directions with one or two zero components of either sign."""
    g = np.random.default_rng(seed)
    n = len(points)
    d = g.choice(np.array([-1.0, -0.0, 0.0, 1.0, 0.5, -0.25], np.float32), (n, 3))
    d[(d == 0).all(axis=1)] = (0.0, 0.0, -1.0)
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3], rays[:, 3:6], rays[:, 6], rays[:, 7] = points, d, tmin, 1e7
    return rays


def slivers(triangles, g):
    """Long slivers through a common region: a ray's boxes overlap nearly all, so the stack runs deep."""
    centre, axis = g.uniform(-0.2, 0.2, (triangles, 3)), g.normal(size=(triangles, 3))
    axis *= 4 / np.linalg.norm(axis, axis=1, keepdims=True)
    return np.stack([centre - axis, centre + axis, centre + g.uniform(-0.05, 0.05, (triangles, 3))], 1).astype(np.float32)


@pytest.mark.parametrize("triangles", [1, 2, 3, 5, 700, 4000])
def test_overlapping_triangles(triangles):
    print(f"[gpu] overlapping triangles {triangles}", flush=True)
    g = np.random.default_rng(triangles)
    tris = slivers(triangles, g)
    a, keep = light_scene(tris)
    check(a, gpuhelp.random_rays(20000, -1.0, 1.0, seed=3))
    check(a, aligned_rays(tris.reshape(-1, 3)[g.integers(0, 3 * triangles, 5000)], 4))


@pytest.mark.parametrize("count", [1, 63, 64, 65, 4097])
def test_axis_aligned_rays_from_vertices(count):
    print(f"[gpu] axis aligned rays {count}", flush=True)
    hs = rt.HostScene(0, 1)
    v = hs.numpy()["vertices"]["pos"]
    g = np.random.default_rng(count)
    rays = aligned_rays(v[g.integers(0, len(v), count)], count)
    check(hs.arrays, rays)
    check(hs.arrays, rays, skip=True)


@pytest.mark.parametrize("tmin", [0.0, -0.0, -1.0, -100.0, -np.inf, np.nan])
@pytest.mark.parametrize("scene", ["room", "one sliver", "slivers"])
def test_rays_from_inside_leaf_boxes(scene, tmin):
    """Origins in a leaf's box (on surfaces, at vertices) and in free air: the box is entered at max(slabs, tmin),
    which is zero or negative here."""
    print(f"[gpu] {scene}, tmin {tmin}", flush=True)
    g = np.random.default_rng(7)
    if scene == "room":
        keep = rt.HostScene(0, 1)
        a = keep.arrays
    else:
        a, keep = light_scene(slivers(1 if scene == "one sliver" else 700, g))
    tris = orc.OracleScene(a).world_tris()[0].reshape(-1, 3, 3)
    n = 4097
    tri = tris[g.integers(0, len(tris), n)]
    surface = gpuhelp.random_rays(n, 0.0, 1.0, seed=8, tmin=tmin)
    surface[:, :3] = (tri * g.dirichlet((1, 1, 1), n)[:, :, None]).sum(1)
    air = gpuhelp.random_rays(n, -1.0, 1.5, seed=9, tmin=tmin)
    bounded = air.copy()
    bounded[:, 7] = g.choice(np.array([1.0, 1e-3, 0.0, -0.5], np.float32), n)
    rays = np.concatenate([surface, aligned_rays(tri[:, 0], 10, tmin), air, bounded])
    check(a, rays)
    if scene == "room":
        check(a, rays, skip=True)


@pytest.mark.parametrize("counting", [False, True])
def test_deep_stack_of_negative_distances(counting):
    """Overlapping sheets some 100 units behind the origins, at distances that differ by less than a spilled entry's
    16 bits hold: an entry must not be taken to lie beyond a hit that it precedes."""
    print(f"[gpu] negative distances, counting {counting}", flush=True)
    n, m = 3000, 4000
    g = np.random.default_rng(n)
    c = np.stack([g.uniform(-1, 1, n), g.uniform(-1, 1, n), g.uniform(99.5, 100.5, n)], 1)
    u, v = (g.normal(size=(n, 3)) * (2, 2, 0.3) for _ in range(2))
    a, keep = light_scene(np.stack([c - u - v, c + u - v, c + v], 1).astype(np.float32))
    rays = np.zeros((m, 8), np.float32)
    rays[:, :2], rays[:, 3:6] = g.uniform(-1, 1, (m, 2)), g.normal(size=(m, 3)) * 0.02 + (0, 0, -1)
    rays[:, 6], rays[:, 7] = -200.0, 1e7
    rt.check(rt.core().rt_counters_enable(int(counting)), "counters")
    try:
        check(a, rays)
    finally:
        rt.core().rt_counters_enable(0)


@pytest.mark.parametrize("near", [0.0, -0.0, -0.5])
def test_gbuffer_without_near_plane(near):
    print(f"[gpu] gbuffer near {near}", flush=True)
    hs = rt.HostScene(0, 1)
    ds, osc = rt.DeviceScene(hs.arrays), orc.OracleScene(hs.arrays)
    pos, ref = osc.world_tris()
    on_mesh = pos[ref[:, 0] != 0].reshape(-1, 3, 3)
    g = np.random.default_rng(3)
    for i in g.integers(0, len(on_mesh), 4):
        w, h = 97, 61
        cam = hs.camera(0, w, h)[0]
        cam.pos = (C.c_float * 3)(*map(float, on_mesh[i].mean(axis=0)))
        cam.nearZ = near
        run = gpuhelp.GrisRun(ds, w, h)
        run.gbuffer(cam)
        for got, want in zip(run.gbuffer_host(), osc.gbuffer(cam)[:3]):
            assert np.array_equal(got.view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize("tmin", [1e-4, 0.0, -1.0])
@pytest.mark.parametrize("scene", ["room", "one sliver", "slivers"])
def test_counted_visits(scene, tmin):
    """Nodes, triangles and rays of the counting builds, as the oracle counts them."""
    print(f"[gpu] counted visits, {scene}, tmin {tmin}", flush=True)
    g = np.random.default_rng(11)
    if scene == "room":
        keep = rt.HostScene(0, 1)
        a = keep.arrays
    else:
        a, keep = light_scene(slivers(1 if scene == "one sliver" else 700, g))
    ds, osc = rt.DeviceScene(a), orc.OracleScene(a)
    tris = osc.world_tris()[0].reshape(-1, 3, 3)
    rays = gpuhelp.random_rays(4097, -1.0, 1.5, seed=12, tmin=tmin)
    if tmin >= 0:  # else entry distances of -0 and 0, which the counted order keeps apart, precede a hit
        rays[::2, :3] = tris[g.integers(0, len(tris), 2049)].mean(axis=1)
    rt.check(rt.core().rt_counters_enable(1), "counters")
    try:
        for mode in (0, 1):
            out = np.zeros(3, np.uint64)
            rt.check(rt.core().rt_counters_read(out.ctypes.data, 1), "read")
            gpuhelp.gpu_trace(ds, rays, mode)
            rt.check(rt.core().rt_counters_read(out.ctypes.data, 1), "read")
            st = osc.trace(rays, mode)[4]
            assert (out[0], out[1], out[2]) == (st[1], st[2], st[0]), f"mode {mode}"
    finally:
        rt.core().rt_counters_enable(0)
