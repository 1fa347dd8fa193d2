"""The training loss bit for bit: FP32 squares of the network's output against
the target, summed by a tree over 256 consecutive voxels each and those sums
one after the other.  The order belongs to the result, so there is no
tolerance."""
import numpy as np
import pytest

from conftest import random_br0, small_mesh

pytestmark = pytest.mark.gpu


def _loss(out, tgt):
    d = out - tgt
    sq = np.zeros(-(-d.size // 256) * 256, np.float32)
    sq[:d.size] = d * d
    t = sq.reshape(-1, 256)
    while t.shape[1] > 1:
        h = t.shape[1] // 2
        t = t[:, :h] + t[:, h:]
    # (cumsum adds in order)
    total = np.cumsum(t[:, 0], dtype=np.float32)[-1]
    return total * (np.float32(1.0) / np.float32(d.size))


# voxels: fewer than 256; one past a group; more groups than the kernel has
# blocks (1024), than the sum takes in one piece (4096)
@pytest.mark.parametrize("dims", [(5, 6, 10), (13, 13, 31), (51, 91, 181), (103, 104, 107)])
def test_loss_in_its_order(dims):
    from pot3d_amd.warmstart import WarmStartNet
    mesh = small_mesh(*dims)
    net = WarmStartNet(mesh, seed=2)
    net.set_scales(2.0, 0.5)
    rng = np.random.default_rng(3)
    for seed in range(3):
        br0 = random_br0(mesh, seed=seed)
        x = 0.3 * rng.standard_normal(net.N)
        # predict returns 0.5 (the scale of the solutions) times the FP32 output
        out = (net.predict(br0) / 0.5).astype(np.float32)
        ref = _loss(out, (x / 0.5).astype(np.float32))
        loss, _ = net.loss_grad(br0, x)
        assert loss == float(ref), (dims, seed, loss, float(ref))
    net.add_sample(br0, x)
    assert net.train(1, 1e-4)[0] == ref, dims
    net.close()
