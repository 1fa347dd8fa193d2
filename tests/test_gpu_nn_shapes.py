"""The network's convolutions and weight gradients where their tiles end: grids
of whole and broken steps of 64, 96, 128 and 256 voxels, an r axis too long for
the staged rows, few theta rows, against the oracle's bf16 mode.  The same
tolerances as for the oracle comparison of the ordinary grids."""
import numpy as np
import pytest

from conftest import random_br0, small_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(402, 9, 10), (5, 42, 9), (18, 34, 66), (10, 10, 6),
                                  (4, 4, 5)])
def test_network_shapes_match_oracle(dims):
    import nn_oracle as N

    from pot3d_amd.warmstart import WarmStartNet
    nr, nt, np_ = dims
    mesh = small_mesh(nr=nr, nt=nt, np_=np_)
    net = WarmStartNet(mesh, seed=1)
    p = N.init_params(3).astype(np.float32)
    rng = np.random.default_rng(4)
    offs, _ = N.param_offsets()
    for (_, cout, _), (_, bo) in zip(N.SPEC, offs):
        p[bo:bo + cout] = 0.05 * rng.standard_normal(cout)
    net.set_params(p)
    net.set_scales(2.0, 0.5)
    br0 = random_br0(mesh, seed=4)
    a, b, c = nr - 2, nt - 2, np_ - 2
    x = 0.3 * rng.standard_normal(a * b * c)
    x0 = N.features(br0, np.asarray(mesh.rh), 2.0, mode="bf16")
    tgt = np.asarray(x / 0.5, np.float32).astype(np.float64).reshape(c, b, a)
    L_o, g_o, out_o = N.loss_and_grad(p.astype(np.float64), x0, tgt, mode="bf16")
    ref = 0.5 * out_o[..., 0].ravel()
    assert np.linalg.norm(net.predict(br0) - ref) <= 5e-3 * np.linalg.norm(ref)
    L_g, g_g = net.loss_grad(br0, x)
    assert abs(L_g - L_o) <= 5e-3 * L_o
    for (_, cout, _), (wo, bo) in zip(N.SPEC, offs):
        for lo, hi in ((wo, bo), (bo, bo + cout)):
            assert np.linalg.norm(g_g[lo:hi] - g_o[lo:hi]) < 3e-2 * max(
                np.linalg.norm(g_o[lo:hi]), 1e-30), (dims, lo)
    net.close()
