"""The network's convolutions in every tile size.  How many voxels and channels a
wave takes depends on the grid's size, up to grids for which the oracle takes
minutes.  But phi is periodic: on a grid of m times the planes, with data that
repeat m times, every voxel has the value that it has on the small grid, which
takes the smallest tiles (compared with the oracle in test_gpu_nn_shapes).

Forward: the sums of a voxel have one order in every tile size, so the values
are the same bit for bit.

Gradient: with m a power of two every gradient of a voxel is 1/m of the small
grid's, exactly.  Only the sums over voxels differ, in their FP32 order.  The
target differs from the output at 300 voxels at the grid's end and at every
101st voxel, so a wrong value at either of them shows.  The sums' error is a few
hundred roundings of 6e-8 at worst, of partial sums not larger than a few times
the total: 1e-4 of a layer's gradient (a tile left out at the end of the largest
grid, one of m copies, would be 1/m, 2e-3 and more)."""
import numpy as np
import pytest

from conftest import random_br0, small_mesh

pytestmark = pytest.mark.gpu


def _net(dims, p):
    from pot3d_amd.warmstart import WarmStartNet
    a, b, c = dims
    net = WarmStartNet(small_mesh(a + 2, b + 2, c + 2), seed=1)
    net.set_params(p)
    net.set_scales(2.0, 0.5)
    return net


def _run(dims, p, br0, delta):
    net = _net(dims, p)
    x = net.predict(br0)
    loss, grads = net.loss_grad(br0, x + delta)
    net.close()
    return x, loss, grads


# first grid: 36 thousand voxels, m = 2, 4, 8 and 16: two and four tiles of 16
# voxels a wave on the finest level with a broken end, 32 channels a wave on the
# next ones; second: 50 thousand, up to four tiles a wave on the two levels below
@pytest.mark.parametrize("dims,m", [((41, 37, 24), 2), ((41, 37, 24), 4), ((41, 37, 24), 8),
                                    ((41, 37, 24), 16), ((81, 77, 8), 32), ((81, 77, 8), 64),
                                    ((81, 77, 8), 512)])
def test_repeated_grid(dims, m):
    import nn_oracle as N
    p = N.init_params(3).astype(np.float32)
    rng = np.random.default_rng(4)
    offs, _ = N.param_offsets()
    for (_, cout, _), (_, bo) in zip(N.SPEC, offs):
        p[bo:bo + cout] = 0.05 * rng.standard_normal(cout)
    a, b, c = dims
    n = a * b * c
    br0 = rng.standard_normal((b + 2, c + 2))
    big = np.zeros((b + 2, m * c + 2))
    big[:, 1:-1] = np.tile(br0[:, 1:-1], (1, m))
    delta = np.zeros(n)
    at = np.unique(np.r_[np.arange(0, n, 101), np.arange(n - 300, n)])
    delta[at] = 0.3 * rng.standard_normal(at.size) + 0.3
    x, loss, g = _run(dims, p, br0, delta)
    xb, lossb, gb = _run((a, b, m * c), p, big, np.tile(delta, m))
    assert np.array_equal(xb.reshape(m, n), np.broadcast_to(x, (m, n)))
    # (the loss adds the sums of 256 voxels one after the other)
    assert abs(lossb - loss) <= (1e-5 + 6e-8 * m * n / 256) * loss
    for (_, cout, _), (wo, bo) in zip(N.SPEC, offs):
        for lo, hi in ((wo, bo), (bo, bo + cout)):
            err = np.linalg.norm(gb[lo:hi].astype(float) - g[lo:hi])
            assert err <= 1e-4 * np.linalg.norm(g[lo:hi].astype(float)), (dims, m, lo, err)
