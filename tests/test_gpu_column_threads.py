"""Solves of several threads at once, each with its own handle: the iterates of
each alone, bit for bit, without a wait that runs into its bound."""
import threading

import numpy as np
import pytest

from conftest import random_br0, small_mesh

pytestmark = pytest.mark.gpu

# columns of 8x8 points: 84 (several calls fit the device together), 289 (two
# do not), 722
MESHES = {"84": (51, 91, 60), "289": (132, 132, 40), "722": (151, 301, 24)}


@pytest.mark.parametrize("names", [("84", "84", "84"), ("289", "289"), ("722", "84", "722"),
                                   ("722", "722")])
@pytest.mark.parametrize("mixed", [0, 2])
def test_threads_solve_at_once(names, mixed, capfd):
    from pot3d_amd import _lib, solver
    handles, ref = [], []
    for q, name in enumerate(names):
        mesh = small_mesh(*MESHES[name])
        s = solver.Pot3dSolver(mesh, -1.0, 2)
        s.set_br0(random_br0(mesh, q))
        s.set_option(_lib.OPT_STOP, 1)
        s.set_option(_lib.OPT_MIXED, mixed)
        handles.append(s)
        x = np.zeros(s.N)
        assert s.solve(x, None, 1e-8, ncgmax=5000)[0] == 0
        v = np.random.default_rng(q).standard_normal(s.N)
        ref.append((s.stats()["ncg"], x, v, s.prec_inv(v)))
    got, start = [None] * len(names), threading.Barrier(len(names))

    def work(q):
        s, out = handles[q], []
        start.wait()
        for _ in range(3):
            x = np.zeros(s.N)
            assert s.solve(x, None, 1e-8, ncgmax=5000)[0] == 0
            out.append((s.stats()["ncg"], x, s.prec_inv(ref[q][2])))
        got[q] = out

    ts = [threading.Thread(target=work, args=(q,)) for q in range(len(names))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for q in range(len(names)):
        assert got[q] is not None, q
        for ncg, x, z in got[q]:
            assert ncg == ref[q][0] and np.array_equal(x, ref[q][1]), (names, q)
            assert np.array_equal(z, ref[q][3]), (names, q)
        handles[q].close()
    assert "a wait ran into its bound" not in capfd.readouterr().err
