"""Ray queries where the traversal's stack, its slab test and its wave-level scheduling can go wrong, bit for bit
against the oracle: overlapping triangles that overflow the LDS part of the stack, directions with zero
components starting on box planes (0 * inf in the slab test), trees of one to a few leaves, ray counts around the
wave size."""
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


def aligned_rays(points, seed):
    """Rays from the given points along directions with one or two zero components of either sign."""
    g = np.random.default_rng(seed)
    n = len(points)
    d = g.choice(np.array([-1.0, -0.0, 0.0, 1.0, 0.5, -0.25], np.float32), (n, 3))
    d[(d == 0).all(axis=1)] = (0.0, 0.0, -1.0)
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3], rays[:, 3:6], rays[:, 6], rays[:, 7] = points, d, 1e-4, 1e7
    return rays


@pytest.mark.parametrize("triangles", [1, 2, 3, 5, 700, 4000])
def test_overlapping_triangles(triangles):
    print(f"[gpu] overlapping triangles {triangles}", flush=True)
    g = np.random.default_rng(triangles)
    # long slivers through a common region: a ray's boxes overlap nearly all, so the stack runs deep
    centre, axis = g.uniform(-0.2, 0.2, (triangles, 3)), g.normal(size=(triangles, 3))
    axis *= 4 / np.linalg.norm(axis, axis=1, keepdims=True)
    tris = np.stack([centre - axis, centre + axis, centre + g.uniform(-0.05, 0.05, (triangles, 3))], 1).astype(np.float32)
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
