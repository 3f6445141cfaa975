"""LBVH builds at the sizes where the sort's and the refit's split changes: the one-workgroup sort up to 4096 keys,
the sort's tiles of 512, 1024 and 4096 keys, the refit's blocks of 1024 and 4096 leaves. Codes, order and nodes bit
for bit against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuhelp  # noqa: E402
import orc  # noqa: E402
from test_gpu_traversal import light_scene  # noqa: E402

rt = gpuhelp.rt


@pytest.mark.parametrize("n", [2, 3, 1023, 1024, 1025, 4095, 4096, 4097, 8191, 131072, 131073, 262144, 262145, 524288, 524289,
                               786432, 786433])
def test_build_matches_oracle(n):
    print(f"[gpu] lbvh {n}", flush=True)
    g = np.random.default_rng(n)
    corner = np.round(g.uniform(-4, 4, (n, 1, 3)) * 64) / 64  # a coarse lattice: equal codes occur
    tris = (corner + g.uniform(-0.05, 0.05, (n, 3, 3)) * (g.random((n, 1, 1)) < 0.7)).astype(np.float32)
    tris += np.float32(0.0)  # no -0.0: which zero a minimum of -0.0 and 0.0 gives is left open
    a, keep = light_scene(tris)
    codes, order, nodes, info = gpuhelp.gpu_bvh(rt.DeviceScene(a))
    ocodes, oorder, onodes = orc.OracleScene(a).bvh()[:3]
    assert np.array_equal(codes, ocodes)
    assert np.array_equal(order, oorder)
    assert np.array_equal(nodes, onodes)
