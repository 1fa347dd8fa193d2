"""The tile schedules of the ILU sweeps with the column sweeps switched off
(P3D_OPT_COLUMN 0): every tile shape and staging, block-persistent or one launch
per diagonal, with and without the residual update in the forward sweep.  The
same bits as the hyperplanes, the same iterates as the default tiles and as the
columns: no tolerance."""
import numpy as np
import pytest

from conftest import random_br0, small_mesh

pytestmark = pytest.mark.gpu

# waves per tile, planes per tile, staging
SHAPES = [(1, 16, 0), (1, 32, 0), (1, 64, 0), (4, 16, 0), (4, 32, 0), (4, 64, 0), (8, 16, 0),
          (8, 32, 0), (1, 16, 1), (1, 32, 1), (1, 64, 1), (1, 16, 2), (1, 32, 2)]


def _set(s, waves, tk, stage):
    """(a stage-2 tile needs one wave and 16 or 32 planes at every step)"""
    from pot3d_amd import _lib
    s.set_option(_lib.OPT_TILE_STAGE, 0)
    s.set_option(_lib.OPT_TILE_WAVES, 1)
    s.set_option(_lib.OPT_TILE_K, tk)
    s.set_option(_lib.OPT_TILE_WAVES, waves)
    s.set_option(_lib.OPT_TILE_STAGE, stage)


def _blocks(s, blocks):
    from pot3d_amd import _lib
    for key, v in zip((_lib.OPT_ILU_BLOCKS_R, _lib.OPT_ILU_BLOCKS_T, _lib.OPT_ILU_BLOCKS_P),
                      blocks):
        s.set_option(key, v)


@pytest.mark.parametrize("blocks", [(1, 1, 1), (2, 2, 2), (2, 1, 3)])
@pytest.mark.parametrize("dims", [(9, 8, 12), (21, 31, 48), (33, 45, 70), (41, 81, 160)])
def test_tiles_match_hyperplanes(dims, blocks):
    from pot3d_amd import _lib, solver
    with solver.Pot3dSolver(small_mesh(*dims), -1.0, 2) as s:
        _blocks(s, blocks)
        x = np.random.default_rng(8).standard_normal(s.N)
        s.set_option(_lib.OPT_SWEEP, 1)
        ref = s.prec_inv(x)
        s.set_option(_lib.OPT_SWEEP, 0)
        s.set_option(_lib.OPT_COLUMN, 0)
        for shape in SHAPES:
            _set(s, *shape)
            for persist in ((-1, 0, 1, 2) if shape[2] == 2 else (-1,)):
                s.set_option(_lib.OPT_BLOCK_SWEEP, persist)
                for rep in range(2):
                    assert np.array_equal(s.prec_inv(x), ref), (shape, persist, rep)
            s.set_option(_lib.OPT_BLOCK_SWEEP, -1)


@pytest.mark.parametrize("blocks", [(1, 1, 1), (2, 4, 2)])
@pytest.mark.parametrize("mixed", [0, 1, 2])
def test_solves_of_every_schedule(mixed, blocks):
    from pot3d_amd import _lib, solver
    mesh = small_mesh(41, 81, 160)
    with solver.Pot3dSolver(mesh, -1.0, 2) as s:
        s.set_br0(random_br0(mesh, 3))
        s.set_option(_lib.OPT_STOP, 1)
        s.set_option(_lib.OPT_MIXED, mixed)
        _blocks(s, blocks)

        def solve():
            x = np.zeros(s.N)
            assert s.solve(x, None, 1e-9, ncgmax=5000)[0] == 0
            return s.stats()["ncg"], x

        for tk in (16, 32):
            _set(s, 1, tk, 0)
            s.set_option(_lib.OPT_COLUMN, 1)
            ref = solve()
            s.set_option(_lib.OPT_COLUMN, 0)
            for stage in (0, 1, 2):
                _set(s, 1, tk, stage)
                for fuse in (0, 1):
                    s.set_option(_lib.OPT_FUSE_RESIDUAL, fuse)
                    for persist in ((-1, 0, 1, 2) if stage == 2 else (-1,)):
                        s.set_option(_lib.OPT_BLOCK_SWEEP, persist)
                        n, x = solve()
                        assert n == ref[0] and np.array_equal(x, ref[1]), (
                            tk, stage, fuse, persist)
                s.set_option(_lib.OPT_FUSE_RESIDUAL, -1)
                s.set_option(_lib.OPT_BLOCK_SWEEP, -1)
