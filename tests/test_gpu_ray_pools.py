"""Where a wave hands its rays out to free lanes: ReSTIR DI's spatial pass (visibility rays of a tile's shifts in
an LDS pool, merged afterwards in the neighbours' order) on tiles that the image only partly covers, and ray queries
beyond the count from which a lane takes more than one ray. Bit for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuhelp  # noqa: E402
import orc  # noqa: E402
from test_gpu_di import run_sequence  # noqa: E402

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


@pytest.mark.parametrize("count", [524287, 524288, 524289, 600001])
def test_rays_beyond_one_per_lane(room, count):
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
