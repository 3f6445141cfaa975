"""Where a wave hands its rays out to free lanes: the spatial passes of ReSTIR DI and GRIS (visibility rays of a tile's
shifts in an LDS pool, merged afterwards in the neighbours' order) on tiles that the image only partly covers, and ray
queries of more waves than the device holds at once. Bit for bit against the oracle."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuhelp  # noqa: E402
import orc  # noqa: E402
from test_gpu_batch import make_view  # noqa: E402
from test_gpu_di import run_sequence  # noqa: E402
from test_gpu_parity import run_gris_frames  # noqa: E402

rt = gpuhelp.rt


@pytest.fixture(scope="module")
def room():
    hs = rt.HostScene(0, 3)
    return hs, rt.DeviceScene(hs.arrays), orc.OracleScene(hs.arrays)


@pytest.mark.parametrize("size", [(1, 1), (7, 9), (8, 8), (65, 17)])
def test_di_spatial_on_ragged_tiles(room, size):
    for temporal, spatial in ((True, True), (False, False)):
        s = rt.di_settings(shift=0, sample=2, temporal=temporal, spatial=spatial)
        run_sequence(*room, *size, s, 2)


@pytest.mark.parametrize("neighbors", [0, 1, 3, 4])
@pytest.mark.parametrize("size", [(1, 1), (7, 9), (65, 17)])
def test_gris_spatial_on_ragged_tiles(room, size, neighbors):
    """0 to 3 neighbours go through the pool, 4 merge one by one."""
    s = rt.settings(shift=2, temporal=True, spatial=True, cap=20, max_depth=6, neighbors=neighbors, radius=4.0)
    assert run_gris_frames(*room, *size, s, 2) == [(0, 0, 0, 0, 0)] * 2


@pytest.mark.parametrize("shift", [0, 1, 2])
def test_gris_spatial_weights_that_are_not_numbers(room, shift):
    """A shifted weight is divided by the luminance of the neighbour's F: negative, NaN and zero luminances give weights
    that are not valid before the visibility ray, whose merge then depends on the ray, and infinite ones."""
    hs, ds, osc = room
    w, h, cap = 96, 40, 8
    n = w * h
    s = rt.settings(shift=shift, temporal=False, spatial=True, cap=cap, max_depth=5, neighbors=3, radius=6.0)
    run = gpuhelp.GrisRun(ds, w, h)
    cams = hs.camera(0, w, h)
    run.gbuffer(cams[0])
    dn, am, _, _ = osc.gbuffer(cams[0])
    run.path_trace(cams, s)
    run.temporal(cams, s)
    temp = run.reservoirs(run.temp)
    rng = np.random.default_rng(shift)
    kind = rng.integers(0, 8, n)
    for k, v in enumerate((-1.0, np.nan, 0.0)):
        temp["F"][kind == k] = v
    plane = run.temp.view(torch.float32)[12 * n:16 * n].view(n, 4)  # F and the primary ray's random state
    plane[:, :3] = torch.from_numpy(temp["F"].copy()).to(plane.device)
    assert not gpuhelp.compare_reservoirs(run.reservoirs(run.temp), temp).any()
    run.spatial(cams, s)
    out, ref = orc.reset_reservoirs(n), np.zeros((h, w, 4), np.float32)
    osc.gris_spatial(cams, dn, am, s, temp, out, ref)
    assert not gpuhelp.compare_reservoirs(run.reservoirs(run.resv[run.cur]), out).any()
    assert gpuhelp.same_float(run.output(1), ref).all()


@pytest.mark.parametrize("neighbors", [(3, 2, 0), (3, 5, 1)])
def test_batched_gris_spatial(room, neighbors):
    """A batch takes the pool if all its views do; a graph built for one choice is rebuilt for the other."""
    hs, ds, _ = room
    sizes = [(64, 17), (7, 9), (40, 40)]
    b = C.c_void_p()
    L = rt.core()
    rt.check(L.rt_batch_create(len(sizes), C.byref(b)), "batch create")
    try:
        t = rt.BatchTuning()
        t.graph = 1
        rt.check(L.rt_batch_set_tuning(b, C.byref(t)), "tuning")
        single, batched = ([gpuhelp.GrisRun(ds, *z) for z in sizes] for _ in range(2))
        for frame, ns in enumerate(((1, 2, 3), neighbors, neighbors)):
            views = (rt.View * len(sizes))()
            for i, z in enumerate(sizes):
                s = rt.settings(shift=2, temporal=True, spatial=True, cap=20, max_depth=5, neighbors=ns[i], radius=5.0)
                cams = hs.camera(frame, *z)
                single[i].frame(cams, s)
                views[i] = make_view(batched[i], ds, cams, s)
            rt.check(L.rt_batch_frame(b, views, len(sizes), gpuhelp.stream()), "batch frame")
            torch.cuda.synchronize()
            for a, z in zip(single, batched):
                assert not gpuhelp.compare_reservoirs(a.reservoirs(a.resv[a.cur]), z.reservoirs(z.resv[z.cur])).any()
                assert gpuhelp.same_float(a.output(1), z.output(1)).all()
                a.flip()
                z.flip()
    finally:
        L.rt_batch_destroy(b)


@pytest.mark.parametrize("count", [524287, 524288, 524289, 600001])
def test_rays_beyond_the_waves_in_flight(room, count):
    print(f"[gpu] rays {count}", flush=True)
    _, ds, osc = room
    rays = gpuhelp.random_rays(count, -0.9, 1.5, seed=count)
    for mode, skip in ((0, False), (0, True), (1, False)):
        t, bary, inst, prim = gpuhelp.gpu_trace(ds, rays, mode, skip)
        ot, obary, oinst, oprim, _ = osc.trace(rays, mode, skip)
        assert np.array_equal(inst, oinst)
        if mode == 0:
            assert np.array_equal(prim, oprim)
            assert np.array_equal(t.view(np.uint32), ot.view(np.uint32))
            assert np.array_equal(bary.view(np.uint32), obary.view(np.uint32))
