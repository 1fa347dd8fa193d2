"""Calls on a card with little memory left: what a solve keeps only for speed
(the direction buffers of the FP64 recurrence, the column sweeps' plan) is given
back to the calls that follow it, which return the same as with memory to
spare."""
import contextlib
import ctypes as C

import numpy as np
import pytest

from conftest import random_br0, small_mesh

pytestmark = pytest.mark.gpu

MB = 1 << 20


@contextlib.contextmanager
def _leave(nbytes):
    """Allocates device memory until about nbytes are free."""
    from pot3d_amd import _lib
    L = _lib.load()
    L.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t)] * 2
    free, total, held = C.c_size_t(), C.c_size_t(), []
    try:
        for _ in range(64):
            assert L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
            size = int(free.value) - int(nbytes)
            if size < 4 * MB:
                break
            p = C.c_void_p()
            if L.hipMalloc(C.byref(p), C.c_size_t(min(size, 32 << 30) // (2 * MB) * (2 * MB))):
                L.hipGetLastError()
                break
            held.append(p)
        assert L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        if abs(int(free.value) - int(nbytes)) >= 64 * MB:
            pytest.skip("the device's memory is not this test's alone")
        yield
    finally:
        for p in held:
            L.hipFree(p)


def _calls(s, x0, rhs):
    """A solve and what a program does with its result."""
    x = x0.copy()
    s.solve(x, rhs.copy(), 1e-9, ncgmax=9)
    phi = s.fill_phi()
    return [x, phi, s.magnetic_energy(), *s.getb()]


@pytest.mark.parametrize("ifprec", [1, 2])
def test_solve_and_fields_in_little_memory(ifprec):
    from pot3d_amd import solver
    mesh = small_mesh(152, 202, 402)  # 12 M unknowns, 96 MB a vector
    with solver.Pot3dSolver(mesh, -1.0, ifprec) as s:
        s.set_br0(random_br0(mesh, 1))
        rhs, x0 = s.rhs(), np.zeros(s.N)
        want = _calls(s, x0, rhs)
    with solver.Pot3dSolver(mesh, -1.0, ifprec) as s:
        s.set_br0(random_br0(mesh, 1))
        # phi (100 MB), then the three fields (300 MB) and what the runtime
        # takes; a solve's direction buffers take 290 MB, its plan about 110
        with _leave(480 * MB):
            got = _calls(s, x0, rhs)
        again = _calls(s, x0, rhs)
    for w, g, a in zip(want, got, again):
        assert np.array_equal(np.asarray(g), np.asarray(w))
        assert np.array_equal(np.asarray(a), np.asarray(w))


def test_options_in_little_memory():
    """A new factorisation and tile plan, and the FP32 operator, after a solve."""
    from pot3d_amd import _lib, solver
    mesh = small_mesh(152, 202, 402)
    out = []
    for leave in (None, 16 * MB):
        with solver.Pot3dSolver(mesh, -1.0, 2) as s:
            s.set_br0(random_br0(mesh, 1))
            x = np.zeros(s.N)
            s.solve(x, None, 1e-9, ncgmax=9)
            with _leave(leave) if leave else contextlib.nullcontext():
                s.set_option(_lib.OPT_APPLY_FP32, 1)
                y = s.ax(x)
                s.set_option(_lib.OPT_ILU_BLOCKS_T, 2)
                out.append((x, y, s.prec_inv(x)))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_kernel_timing_that_takes_the_columns_plan():
    """Timing the residual update in the forward sweep needs the columns (or
    register tiles): an error where the vectors take their plan's memory."""
    from pot3d_amd import _lib, solver
    with solver.Pot3dSolver(small_mesh(152, 202, 402), -1.0, 2) as s:
        s.prec_inv(np.zeros(s.N))  # builds the plan, about 130 MB
        with _leave(150 * MB):  # the vectors take 250 MB
            for _ in range(2):
                with pytest.raises(_lib.Pot3dError) as e:
                    s.time_kernel(11, 1)
                assert e.value.code == _lib.P3D_ESTATE
        s.set_option(_lib.OPT_COLUMN, -1)
        assert s.time_kernel(11, 1) > 0


def test_mixed_solve_after_one_without_memory():
    """A call that finds memory for some of the FP32 vectors only, twice, and
    then for all."""
    from pot3d_amd import _lib, solver
    mesh = small_mesh(152, 202, 402)  # the five vectors take 48 MB each and more
    out = []
    for leave in (None, 130 * MB):
        with solver.Pot3dSolver(mesh, -1.0, 1) as s:
            s.set_br0(random_br0(mesh, 1))
            s.set_option(_lib.OPT_MIXED, 2)
            x = np.zeros(s.N)
            if leave:
                with _leave(leave):
                    for _ in range(2):
                        with pytest.raises(_lib.Pot3dError) as e:
                            s.solve(x, None, 1e-9, ncgmax=9)
                        assert e.value.code == _lib.P3D_ENOMEM
            s.solve(x, None, 1e-9, ncgmax=9)
            out.append(x)
    assert np.array_equal(out[0], out[1])


def test_legacy_lu_host_vector_in_little_memory():
    from pot3d_amd import _lib
    L = _lib.load()
    a, b, c = 64, 128, 512
    n, ab = a * b * c, a * b
    rng = np.random.default_rng(3)
    p = np.arange(n, dtype=np.int64).reshape(c, b, a)
    off = [ab - n, -ab, -a, -1, 0, 1, a, ab, n - ab]
    on = np.ones((n, 9), bool).reshape(c, b, a, 9)
    on[:-1, :, :, 0] = on[1:, :, :, 8] = on[0, :, :, 1] = on[-1, :, :, 7] = False
    on[:, 0, :, 2] = on[:, -1, :, 6] = on[:, :, 0, 3] = on[:, :, -1, 5] = False
    cols = np.stack([p + o for o in off], axis=-1)
    vals = -rng.uniform(0.2, 1.0, on.shape)
    vals[..., 4] = 8.5
    ja = (cols[on] + 1).astype(np.int32)
    av = vals[on].astype(np.float32)
    ia = np.concatenate([[1], 1 + np.cumsum(on.reshape(n, 9).sum(axis=1))]).astype(np.int32)
    x = rng.standard_normal(n)
    out = []
    for leave in (None, 16 * MB):  # (a staging vector takes 32 MB)
        v = av.copy()
        L.load_external_lu_solver(v.ctypes.data, ia.ctypes.data, ja.ctypes.data, n, len(v))
        y = x.copy()
        with _leave(leave) if leave else contextlib.nullcontext():
            L.external_lu_solver(y.ctypes.data)
        L.unload_external_lu_solver()
        out.append(y)
    assert np.array_equal(out[0], out[1])
