"""The grid gradients of a batch that k_mlp_scatter adds (up to 65536 samples) against those that the training kernel
adds itself: the same samples with masked ones appended until the batch is beyond that limit. The sums are fixed
point, so the two are the same bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import gpuhelp  # noqa: E402

rt = gpuhelp.rt
LO, HI = (-1.0, -2.0, 0.5), (3.0, 2.0, 4.5)


def grid_gradient(m, pos, target):
    d_pos, d_t = torch.from_numpy(pos).cuda(), torch.from_numpy(target).cuda()
    rt.check(rt.core().rt_mlp_gradients(m.handle, d_pos.data_ptr(), d_t.data_ptr(), len(pos), None, gpuhelp.stream()),
             "gradients")
    torch.cuda.synchronize()
    return m.read_gradients()[0]


@pytest.mark.parametrize("guide", [False, True], ids=["radiance", "proposal"])
@pytest.mark.parametrize("n", [1, 31, 33, 4097, 65536])
def test_scatter_matches_training_kernel(n, guide):
    print(f"[gpu] scatter {n} guide {guide}", flush=True)
    g = np.random.default_rng(n)
    m = rt.Mlp(rt.mlp_config(LO, HI, log2_table=14, base_res=4, max_res=256, seed=5), guide=guide)
    beyond = 65537
    pos = g.uniform(np.array(LO) - 0.3, np.array(HI) + 0.3, (beyond, 3)).astype(np.float32)
    target = g.uniform(0.1, 2.0, (beyond, 4 if guide else 3)).astype(np.float32)
    if guide:
        target[:, :3] /= np.linalg.norm(target[:, :3], axis=1, keepdims=True)
    target[7:n:5] = np.nan  # masked samples within the batch
    target[n:] = -1.0
    a = grid_gradient(m, pos[:n].copy(), target[:n].copy())
    b = grid_gradient(m, pos, target)
    assert np.count_nonzero(a) > 0
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
