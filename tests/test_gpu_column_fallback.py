"""Column sweeps whose waits run into their bound: the call starts over with the
tile schedules and returns what they return, bit for bit.  P3D_COLUMN_POLLS=0
makes every wait that has to poll give up; the kernels end as always."""
import numpy as np
import pytest

from conftest import random_br0, small_mesh

pytestmark = pytest.mark.gpu

MESSAGE = "a wait ran into its bound"


def _solver(mesh, column, monkeypatch):
    from pot3d_amd import _lib, solver
    s = solver.Pot3dSolver(mesh, -1.0, 2)
    s.set_br0(random_br0(mesh, 2))
    s.set_option(_lib.OPT_COLUMN, column)
    if column:
        monkeypatch.setenv("P3D_COLUMN_POLLS", "0")
    else:
        monkeypatch.delenv("P3D_COLUMN_POLLS", raising=False)
    return s


@pytest.mark.parametrize("mixed", [0, 1, 2])
@pytest.mark.parametrize("blocks", [(1, 1, 1), (2, 1, 2)])
@pytest.mark.parametrize("dims", [(42, 60, 80), (19, 91, 181)])
def test_solve_starts_over(dims, blocks, mixed, monkeypatch, capfd):
    from pot3d_amd import _lib
    mesh = small_mesh(*dims)
    got = []
    for column in (0, 1):
        with _solver(mesh, column, monkeypatch) as s:
            s.set_option(_lib.OPT_STOP, 1)
            s.set_option(_lib.OPT_MIXED, mixed)
            s.set_option(_lib.OPT_VERBOSE, 1)
            for key, v in zip((_lib.OPT_ILU_BLOCKS_R, _lib.OPT_ILU_BLOCKS_T,
                               _lib.OPT_ILU_BLOCKS_P), blocks):
                s.set_option(key, v)
            x, rhs = np.zeros(s.N), s.rhs()
            assert s.solve(x, rhs, 1e-9, ncgmax=5000, ncghist=50)[0] == 0
            out, err = capfd.readouterr()
            assert (MESSAGE in err) == (column == 1)
            # the history of the call's one valid run
            assert out.count("Iteration:        0 ") == (1 if mixed == 0 else 0), out
            got.append((s.stats()["ncg"], x, rhs))
            y = np.zeros(s.N)
            assert s.solve(y, None, 1e-9, ncgmax=5000)[0] == 0
            assert MESSAGE not in capfd.readouterr().err
            assert np.array_equal(y, x)
    assert got[0][0] == got[1][0]
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])


def test_solve_that_does_not_converge(monkeypatch):
    """An error of the call is the tiles' error, not that of the void attempt."""
    from pot3d_amd import _lib
    mesh = small_mesh(42, 60, 80)
    for mixed in (0, 1, 2):
        got = []
        for column in (0, 1):
            with _solver(mesh, column, monkeypatch) as s:
                s.set_option(_lib.OPT_MIXED, mixed)
                x = np.zeros(s.N)
                assert s.solve(x, None, 1e-9, ncgmax=7)[0] == 1
                got.append((s.stats()["ncg"], s.stats()["true_relres"], x))
        assert got[0][:2] == got[1][:2] and np.array_equal(got[0][2], got[1][2]), mixed


def test_single_calls(monkeypatch, capfd):
    from pot3d_amd import _lib
    mesh = small_mesh(42, 60, 80)
    with _solver(mesh, 0, monkeypatch) as s:
        x = np.random.default_rng(1).standard_normal(s.N)
        ref = s.prec_inv(x)
    with _solver(mesh, 1, monkeypatch) as s:
        for rep in range(3):
            # the tiles from then on, until the option is set again
            assert np.array_equal(s.prec_inv(x), ref)
            assert (MESSAGE in capfd.readouterr().err) == (rep != 1)
            if rep == 1:
                s.set_option(_lib.OPT_COLUMN, 1)
    for kid in (2, 3, 7):
        with _solver(mesh, 1, monkeypatch) as s:
            assert s.time_kernel(kid, 1) > 0
            assert MESSAGE in capfd.readouterr().err, kid
            assert np.array_equal(s.prec_inv(x), ref), kid


@pytest.mark.parametrize("on_device", [False, True])
def test_legacy_lu_starts_over(on_device, monkeypatch, capfd):
    import ctypes as C

    from pot3d_amd import _lib
    from test_gpu_legacy_columns import _matrix
    L = _lib.load()
    ia, ja, av, _, _, _ = _matrix((24, 17, 36), True, 7)
    n = len(ia) - 1
    x = np.random.default_rng(8).standard_normal(n)
    dev = C.c_void_p()  # (the library's own HIP runtime)
    assert L.hipMalloc(C.byref(dev), C.c_size_t(8 * n)) == 0
    out = []
    for polls in (None, "0"):
        if polls is None:
            monkeypatch.delenv("P3D_COLUMN_POLLS", raising=False)
        else:
            monkeypatch.setenv("P3D_COLUMN_POLLS", polls)
        a = av.copy()
        L.load_external_lu_solver(a.ctypes.data, ia.ctypes.data, ja.ctypes.data, n, len(a))
        for rep in range(2):
            y = x.copy()
            host = C.c_void_p(y.ctypes.data)
            if on_device:
                assert L.hipMemcpy(dev, host, C.c_size_t(8 * n), 1) == 0
                L.external_lu_solver(dev)
                assert L.hipMemcpy(host, dev, C.c_size_t(8 * n), 2) == 0
            else:
                L.external_lu_solver(host)
            out.append(y)
            assert (MESSAGE in capfd.readouterr().err) == (polls == "0" and rep == 0)
        L.unload_external_lu_solver()
    assert L.hipFree(dev) == 0
    for y in out[1:]:
        assert np.array_equal(y, out[0])
