"""ILU sweeps by columns (P3D_OPT_COLUMN): the same bits as the hyperplane and
tile schedules at the edges of its columns (8x8 points), chunks (8 steps) and
rounds (32 steps), with and without a block-Jacobi cut, on uniform and
non-uniform phi meshes, in FP64 and in the FP32 recurrence.  Bit equality: no
tolerance."""
import numpy as np
import pytest

from conftest import random_br0, small_mesh

pytestmark = pytest.mark.gpu

# interior r, theta: one column, one point over, several with remainders;
# phi: shorter than a lane's delay, at and around whole rounds of 32 steps
DIMS = [(8, 8, 6), (9, 17, 7), (3, 5, 40), (16, 8, 32 - 21), (17, 24, 33 - 21), (24, 16, 64 - 28),
        (25, 31, 65 - 28), (40, 9, 96), (12, 70, 131), (50, 50, 180)]


def _mesh(dims, uniform):
    from p3d_driver import inputs
    a, b, c = dims
    if uniform:
        return small_mesh(a + 2, b + 2, c + 2)
    return inputs.global_mesh(a + 2, b + 2, c + 2, 1.0, 2.5, rfrac=(0.0, 1.0), drratio=(1.5,),
                              pfrac=(0.2, 0.6), dpratio=(1.7, 1.0 / 1.7))


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("dims", DIMS)
def test_columns_match_other_schedules(dims, uniform):
    from pot3d_amd import _lib, solver
    with solver.Pot3dSolver(_mesh(dims, uniform), -1.0, 2) as s:
        x = np.random.default_rng(11).standard_normal(s.N)
        for blocks in ((1, 1, 1), (2, 2, 1), (2, 1, 2)):
            for key, v in zip((_lib.OPT_ILU_BLOCKS_R, _lib.OPT_ILU_BLOCKS_T,
                               _lib.OPT_ILU_BLOCKS_P), blocks):
                s.set_option(key, v)
            s.set_option(_lib.OPT_SWEEP, 1)
            ref = s.prec_inv(x)
            s.set_option(_lib.OPT_SWEEP, 0)
            for tk in (16, 32, 64):
                s.set_option(_lib.OPT_TILE_K, tk)
                s.set_option(_lib.OPT_COLUMN, 0)
                assert np.array_equal(s.prec_inv(x), ref), ("tiles", dims, blocks, tk)
                s.set_option(_lib.OPT_COLUMN, 1)
                for rep in range(3):
                    assert np.array_equal(s.prec_inv(x), ref), (dims, blocks, tk, rep)


@pytest.mark.parametrize("blocks", [(1, 1, 1), (2, 2, 2)])
@pytest.mark.parametrize("dims", [(9, 17, 7), (25, 31, 65 - 28), (50, 50, 180)])
def test_columns_in_the_solves(dims, blocks):
    """FP64 and FP32-recurrence solves with tiles and columns, the residual
    update folded into the forward sweep or on its own: the same iterates."""
    from pot3d_amd import _lib, solver
    mesh = _mesh(dims, True)
    with solver.Pot3dSolver(mesh, -1.0, 2) as s:
        s.set_br0(random_br0(mesh, 2))
        s.set_option(_lib.OPT_STOP, 1)
        for key, v in zip((_lib.OPT_ILU_BLOCKS_R, _lib.OPT_ILU_BLOCKS_T, _lib.OPT_ILU_BLOCKS_P),
                          blocks):
            s.set_option(key, v)
        for mixed in (0, 1, 2):
            s.set_option(_lib.OPT_MIXED, mixed)
            got = []
            for col, fuse in ((0, 0), (1, 0), (1, 1), (1, 1)):
                s.set_option(_lib.OPT_COLUMN, col)
                s.set_option(_lib.OPT_FUSE_RESIDUAL, fuse)
                x = np.zeros(s.N)
                assert s.solve(x, None, 1e-9, ncgmax=5000)[0] == 0
                got.append((s.stats()["ncg"], x))
            for n, x in got[1:]:
                assert n == got[0][0] and np.array_equal(x, got[0][1]), (dims, blocks, mixed)
