"""FP64 recurrence with the solution updated once per group of iterations: the
iterates after every count of iterations, also where a solve ends inside a
group, against the same recurrence in numpy with the library's operator and
preconditioner."""
import numpy as np
import pytest

from conftest import random_br0, small_mesh

pytestmark = pytest.mark.gpu

# The two sides differ in the order of their sums and in fused multiply-adds:
# a few eps64 of relative change per iteration, grown by the recurrence by well
# under 1e3 over these few iterations.
TOL = 1e-11


def _pcg(s, b, x, n):
    r = b - s.ax(x)
    z = s.prec_inv(r)
    p, rz = z.copy(), r @ z
    for _ in range(n):
        ap = s.ax(p)
        alpha = rz / (p @ ap)
        x = x + alpha * p
        r = r - alpha * ap
        z = s.prec_inv(r)
        rz, old = r @ z, rz
        p = z + rz / old * p
    return x


@pytest.mark.parametrize("ifprec", [0, 1, 2])
@pytest.mark.parametrize("dims", [(5, 5, 8), (9, 19, 33), (34, 18, 64)])
def test_solution_after_every_count(dims, ifprec):
    from pot3d_amd import _lib, solver
    mesh = small_mesh(*dims)
    with solver.Pot3dSolver(mesh, 1.0, ifprec) as s:
        s.set_br0(random_br0(mesh, 5))
        b = s.rhs()
        x0 = np.random.default_rng(6).standard_normal(s.N) * 1e-2
        for n in range(1, 10):
            ref = _pcg(s, b, x0, n)
            for chunk, graph in ((0, 1), (1, 0), (5, 1), (8, 1)):
                s.set_option(_lib.OPT_CHUNK, chunk)
                s.set_option(_lib.OPT_GRAPH, graph)
                x = x0.copy()
                ierr, ncg, _ = s.solve(x, None, 1e-30, ncgmax=n)
                assert ierr == 1 and ncg == n, (dims, ifprec, n, ierr, ncg)
                err = np.abs(x - ref).max() / np.abs(ref).max()
                assert err < TOL, (dims, ifprec, n, chunk, graph, err)
