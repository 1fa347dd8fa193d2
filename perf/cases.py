"""Cases for timing the library through its public entry points.

Seven kinds of call, each as a user's program makes it:

  readbr   solver.readbr: a surface Br map onto the solver's mesh (host arrays)
  potfld   solver.potfld: the whole driver-side call on host arrays: solve,
           phi with boundary values, magnetic energy
  solve    Pot3dSolver.solve_dev: one PCG solve, vectors resident on the GPU;
           with guess=True the learned initial guess is made inside the pass
  extlu    external_lu_solver: one application of the drop-in LU interface
           that an unmodified driver calls once per CG iteration
  guess    the learned initial guess alone: network prediction on the coarse
           grid, boundary values, prolongation to the fine grid
  train    WarmStartNet.loss_grad: one forward and backward of the network
  field    fill_phi, magnetic_energy and getb of a solution (host arrays)

Inputs come from the seeded synthetic Br maps of the repository's workloads.
``exact`` gives the outputs in float64 from plain torch and numpy: the
operator separates (uniform phi mesh), so a solution is an FFT in phi, an
eigenbasis in r and tridiagonal systems in theta.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

from p3d_driver import inputs, workloads
from pot3d_amd import _lib, solver, warmstart

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WEIGHTS = os.path.join(ROOT, "pot3d_amd", "weights", "warmstart_pfss_51x91x181.npz")
DEV = "cuda:0"
BLOCKS = (8, 16, 16)  # the block-Jacobi cut of the fast paths


def _solve(name, grid, option, mixed, blocks, guess=False):
    nr, nt, np_ = grid
    return dict(name=name, kind="solve", nr=nr, nt=nt, np=np_, option=option, ifprec=2,
                mixed=mixed, blocks=blocks, guess=guess, tol=1e-10 if mixed else 1e-9)


def listed():
    return [
        # the driver's start: a 1-degree map onto the small grid's surface
        dict(name="readbr_91x181", kind="readbr", nt=91, np=181, ntn=181, npn=361, option="ss"),
        # the reference's source-surface deck: diagonal preconditioner
        dict(name="potfld_diag_55x181x361", kind="potfld", nr=55, nt=181, np=361, option="ss",
             ifprec=1),
        # the smallest grid, Neumann outer boundary, single-rank ILU0
        dict(name="potfld_ilu_51x91x181", kind="potfld", nr=51, nt=91, np=181,
             option="potential", ifprec=2),
        # mixed precision on the smallest grid, single-rank ILU0
        _solve("solve_mixed_51x91x181", (51, 91, 181), "ss", 2, False),
        # FP64 with the ILU0 of a decomposed grid (current-sheet deck's grid, |Br|)
        _solve("solve_fp64_bj_101x181x361", (101, 181, 361), "open", 0, True),
        # the drop-in baseline: FP64, single-rank ILU0
        _solve("solve_fp64_151x301x601", (151, 301, 601), "ss", 0, False),
        # the fast path: mixed precision, block-Jacobi ILU0, learned guess
        _solve("solve_fast_151x301x601", (151, 301, 601), "ss", 2, True, guess=True),
        # the fast path on a grid of more than 2^26 unknowns
        _solve("solve_fast_205x409x815", (205, 409, 815), "ss", 2, True),
        # the drop-in LU interface on device vectors
        dict(name="extlu_51x91x181", kind="extlu", nr=51, nt=91, np=181),
        # the learned guess for the middle grid
        dict(name="guess_51x91x181", kind="guess", nr=51, nt=91, np=181, fnr=151, fnt=301,
             fnp=601),
        # one training step's forward and backward
        dict(name="train_51x91x181", kind="train", nr=51, nt=91, np=181),
        # post-processing of a solution on the current-sheet deck's grid
        dict(name="field_101x181x361", kind="field", nr=101, nt=181, np=361, option="open"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """(nr, nt, np) with about lo..hi unknowns, np : nt : nr near 4 : 2 : 1."""
    n = _log(rng, lo, hi)
    s = (n / 8.0) ** (1.0 / 3.0)
    f, h = rng.uniform(0.7, 1.3), rng.uniform(0.85, 1.15)
    return (max(12, round(s * f)) + 2, max(20, round(2 * s * h)) + 2,
            max(40, round(4 * s / f / h)) + 2)


def draw(rng):
    kind = rng.choice(["readbr", "potfld", "potfld", "solve", "solve", "solve", "solve", "solve",
                       "extlu", "guess", "train", "field"])
    option = rng.choice(["ss", "ss", "open", "potential"])
    if kind == "readbr":
        deg = rng.choice([1.0, 1.0, 2.0, 0.5])
        return dict(kind=kind, nt=_log(rng, 40, 601), np=_log(rng, 80, 1201),
                    ntn=int(180 / deg) + 1, npn=int(360 / deg) + 1, option=option)
    if kind == "potfld":
        nr, nt, np_ = _grid(rng, 1e5, 4e6)
        return dict(kind=kind, nr=nr, nt=nt, np=np_, option=option, ifprec=rng.choice([1, 2]))
    if kind == "solve":
        mixed = rng.choice([0, 2, 2])
        nr, nt, np_ = _grid(rng, 2e5, 1.2e7 if mixed == 0 else 3e7)
        return dict(kind=kind, nr=nr, nt=nt, np=np_, option=rng.choice(["ss", "ss", "open"]),
                    ifprec=2, mixed=mixed, blocks=rng.random() < 0.6, guess=False,
                    tol=1e-10 if mixed else 1e-9)
    nr, nt, np_ = _grid(rng, 1e5, 2e6)
    if kind == "guess":
        fnr, fnt, fnp = _grid(rng, 3e6, 3e7)
        return dict(kind=kind, nr=nr, nt=nt, np=np_, fnr=fnr, fnt=fnt, fnp=fnp)
    if kind == "field":
        nr, nt, np_ = _grid(rng, 2e5, 1e7)
        return dict(kind=kind, nr=nr, nt=nt, np=np_, option=rng.choice(["ss", "open"]))
    return dict(kind=kind, nr=nr, nt=nt, np=np_)


# -- inputs --------------------------------------------------------------------
def _domain(option):
    d = dict(workloads.DOMAINS["open" if option == "open" else "pfss"])
    return dict(d, option=option)


def _mesh(nr, nt, np_, option):
    d = _domain(option)
    return inputs.global_mesh(nr, nt, np_, d["r0"], d["r1"], rfrac=(0.0, 1.0),
                              drratio=(workloads.PFSS_DRRATIO,))


def _map(option, seed, ntn=181, npn=361):
    return inputs.synthetic_br_map(seed, _domain(option)["n_bipoles"], ntn, npn)


def _readbr(mesh, option, tn, pn, bn):
    """The map on the mesh in plain numpy: bilinear interpolation, seam, pole
    averages, flux balance, |Br| for 'open'; (br0, fluxp, fluxm, area, err)."""
    def table(x, v):
        i = np.clip(np.searchsorted(x, v, side="left") - 1, 0, x.size - 2)
        return i, (v - x[i]) / (x[i + 1] - x[i])
    it, at = table(tn, mesh.th[1:-1])
    ip, ap = table(pn, mesh.ph[1:-1])
    at, ap = at[:, None], ap[None, :]
    f = lambda a, b: bn[np.ix_(it + a, ip + b)]  # noqa: E731
    br0 = np.empty((mesh.nt, mesh.np))
    br0[1:-1, 1:-1] = ((1 - at) * ((1 - ap) * f(0, 0) + ap * f(0, 1))
                       + at * ((1 - ap) * f(1, 0) + ap * f(1, 1)))
    br0[:, 0], br0[:, -1] = br0[:, -2], br0[:, 1]
    for row, inner in ((0, 1), (-1, -2)):
        s = float(np.sum(br0[inner, 1:-1] * mesh.dph[1:-1])) / (2.0 * math.pi)
        br0[row] = 2.0 * s - br0[inner]
    da = (mesh.sth * mesh.dth)[1:-1, None] * mesh.dph[None, 1:-1]
    v = br0[1:-1, 1:-1]
    fp, fm = float(np.sum(np.where(v > 0, v * da, 0.0))), float(np.sum(np.where(v > 0, 0.0, v * da)))
    area = float(np.sum(da))
    err = (fp + fm) / area
    br0 = br0 - err
    return (np.abs(br0) if option == "open" else br0), fp, fm, area, err


def _br0(mesh, option, seed):
    return _readbr(mesh, option, *_map(option, seed))[0]


def _net(mesh):
    """The warm-start network with the trained weights (it is convolutional:
    the weights fit every grid)."""
    z = np.load(WEIGHTS, allow_pickle=False)
    net = warmstart.WarmStartNet(mesh)
    net.set_params(z["params"])
    net.set_scales(float(z["bscale"]), float(z["phiscale"]))
    return net


def _csr(mesh):
    """The ILU matrix of the mesh as the driver hands it over (1-based CSR,
    FP32, phi wrap kept, r and theta boundary couplings dropped), on the GPU."""
    low, up, diag = _couplings(mesh, -1.0)
    c, b, a = diag.shape
    n = a * b * c
    p = torch.arange(n, device=DEV).reshape(c, b, a)
    off = [-a * b, -a, -1, 0, 1, a, a * b]
    val = [low[0], low[1], low[2], diag, up[2], up[1], up[0]]
    on = torch.ones((9, c, b, a), dtype=torch.bool, device=DEV)
    cols = torch.stack([p] + [p + o for o in off] + [p])
    vals = torch.stack([up[0]] + val + [low[0]])
    cols[0] += a * b - n   # plane c-1 to plane 0
    cols[8] += n - a * b   # plane 0 to plane c-1
    on[0, :-1] = on[8, 1:] = on[1, 0] = on[7, -1] = False
    on[2, :, 0] = on[6, :, -1] = False
    on[3, :, :, 0] = on[5, :, :, -1] = False
    flat = lambda t: t.reshape(9, n).T  # noqa: E731
    on = flat(on)
    ia = torch.ones(n + 1, dtype=torch.int32, device=DEV)
    ia[1:] += torch.cumsum(on.sum(1), 0).int()
    return ia, (flat(cols)[on] + 1).int().contiguous(), flat(vals)[on].float().contiguous()


def _residual(case, seed):
    n = (case["nr"] - 2) * (case["nt"] - 2) * (case["np"] - 2)
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    return torch.randn(n, dtype=torch.float64, device=DEV, generator=g)


def _handle(mesh, case):
    s = solver.Pot3dSolver(mesh, inputs.pm_r1_for(case["option"]), case["ifprec"])
    if case.get("blocks"):
        for key, v in zip((_lib.OPT_ILU_BLOCKS_R, _lib.OPT_ILU_BLOCKS_T, _lib.OPT_ILU_BLOCKS_P),
                          BLOCKS):
            s.set_option(key, v)
        s.set_option(_lib.OPT_TILE_K, 16)
        s.set_option(_lib.OPT_TILE_STAGE, 2)
    return s


def _guess_state(nr, nt, np_, fmesh, seed):
    cmesh = _mesh(nr, nt, np_, "ss")
    br0 = _br0(cmesh, "ss", seed)
    sc = solver.Pot3dSolver(cmesh, -1.0, 2)
    sc.set_br0(br0)
    return dict(net=_net(cmesh), coarse=sc, cbr0=br0, tab=warmstart.prolong_tables(cmesh, fmesh),
                phic=torch.empty(nr * nt * np_, dtype=torch.float64, device=DEV),
                x=torch.zeros(fmesh.N, dtype=torch.float64, device=DEV))


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind == "readbr":
        mesh = _mesh(32, case["nt"], case["np"], case["option"])
        return dict(st, mesh=mesh, map=_map(case["option"], seed, case["ntn"], case["npn"]))
    if kind == "extlu":
        L = _lib.load()
        ia, ja, av = _csr(_mesh(case["nr"], case["nt"], case["np"], "ss"))
        torch.cuda.synchronize()
        L.unload_external_lu_solver()
        n = ia.numel() - 1
        L.load_external_lu_solver(av.data_ptr(), ia.data_ptr(), ja.data_ptr(), n, av.numel() + 1)
        r = _residual(case, seed)
        return dict(st, L=L, r=r, z=torch.empty_like(r), keep=(ia, ja, av))
    option = case.get("option", "ss")
    mesh = _mesh(case["nr"], case["nt"], case["np"], option)
    if kind == "guess":
        fmesh = _mesh(case["fnr"], case["fnt"], case["fnp"], "ss")
        return dict(st, **_guess_state(case["nr"], case["nt"], case["np"], fmesh, seed))
    br0 = _br0(mesh, option, seed)
    pm = inputs.pm_r1_for(option)
    if kind == "potfld":
        w = workloads.Workload("case", mesh, br0, pm, option, 1e-9, case["ifprec"])
        return dict(st, w=w, s=_handle(mesh, case))
    if kind == "solve":
        if case["guess"]:
            st.update(_guess_state(*workloads.COARSE_GRID, mesh, seed))
        else:
            st.update(x=torch.zeros(mesh.N, dtype=torch.float64, device=DEV))
        s = _handle(mesh, case)
        s.set_br0(br0)
        s.set_option(_lib.OPT_STOP, 1)
        s.set_option(_lib.OPT_MIXED, case["mixed"])
        s.set_option(_lib.OPT_GUESS_CHECK, 2 if case["guess"] else 0)
        return dict(st, s=s)
    x = _solution(mesh, pm, br0).cpu().numpy().ravel()
    if kind == "train":
        return dict(st, net=_net(mesh), br0=br0, x=x)
    s = solver.Pot3dSolver(mesh, pm, 0)
    s.set_br0(br0)
    return dict(st, s=s, x=x)


# -- one pass ---------------------------------------------------------------------
def _guess(st):
    xc = st["net"].predict(st["cbr0"])
    phic = st["coarse"].fill_phi(xc)
    st["phic"].copy_(torch.from_numpy(phic))
    torch.cuda.current_stream().synchronize()
    warmstart.prolong_dev_noalloc(st["tab"], st["phic"].data_ptr(), st["x"].data_ptr())
    return st["x"]


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "readbr":
        br0, flux = solver.readbr(st["mesh"], *st["map"], True, case["option"] == "open")
        return dict(br0=br0, **flux)
    if kind == "potfld":
        r = solver.potfld(st["w"], solver=st["s"])
        return dict(x=r.x, phi=r.phi, energy=r.energy, ierr=r.ierr)
    if kind == "solve":
        x = st["x"]
        if case["guess"]:
            _guess(st)
        else:
            x.zero_()
            torch.cuda.current_stream().synchronize()  # the solver has a stream of its own
        ierr, _, _ = st["s"].solve_dev(x.data_ptr(), None, case["tol"])
        return dict(x=x, ierr=ierr)
    if kind == "extlu":
        st["z"].copy_(st["r"])
        torch.cuda.current_stream().synchronize()
        st["L"].external_lu_solver(st["z"].data_ptr())
        return st["z"]
    if kind == "guess":
        return _guess(st)
    if kind == "train":
        loss, grads = st["net"].loss_grad(st["br0"], st["x"])
        return dict(loss=loss, grads=grads)
    phi = st["s"].fill_phi(st["x"])
    w = st["s"].magnetic_energy()
    br, bt, bp = st["s"].getb()
    return dict(phi=phi, energy=w, br=br, bt=bt, bp=bp)


# -- what a pass cannot do without ----------------------------------------------
# Multiply-adds per voxel of the finest level: (Cin, Cout, level) of the network
_CONVS = [(16, 16, 0), (16, 32, 1), (32, 64, 2), (64, 128, 3), (128, 64, 2), (64, 32, 1),
          (32, 16, 0), (16, 16, 0)]


def _net_work(nr, nt, np_):
    """(bytes, flops) of one forward: every layer's input and output in BF16."""
    by = fl = 0
    for ci, co, lev in _CONVS:
        v = 1
        for n in (nr - 2, nt - 2, np_ - 2):
            v *= -(-n // (1 << lev))
        by += 2 * v * (ci + co)
        fl += 2 * 27 * v * ci * co
    return by, fl


def _iterations(n, case):
    """PCG iterations, roughly: they grow with the longest axis."""
    per = 7.5 if case["ifprec"] == 1 else 1.5
    return per * case["np"] * (1.1 if case.get("mixed") else 1.0)


def work(case):
    kind = case["kind"]
    if kind == "readbr":
        n = case["nt"] * case["np"]
        return dict(bytes=8.0 * (case["ntn"] * case["npn"] + n), flops=20.0 * n)
    n = float((case["nr"] - 2) * (case["nt"] - 2) * (case["np"] - 2))
    if kind in ("potfld", "solve"):
        # per iteration: A p, two vector updates and dots, the preconditioner
        if case.get("mixed"):
            by, fl = 60.0, 60.0
        else:
            by, fl = (80.0, 50.0) if case["ifprec"] == 1 else (112.0, 60.0)
        it = _iterations(n, case)
        return dict(bytes=by * n * it, flops=fl * n * it)
    if kind == "extlu":
        return dict(bytes=n * (16.0 + 2 * (16.0 + 4.0) + 8.0), flops=20.0 * n)
    if kind == "guess":
        by, fl = _net_work(case["nr"], case["nt"], case["np"])
        nf = float((case["fnr"] - 2) * (case["fnt"] - 2) * (case["fnp"] - 2))
        return dict(bytes=by + 24.0 * n + 8.0 * nf, flops=fl + 30.0 * nf)
    if kind == "train":
        by, fl = _net_work(case["nr"], case["nt"], case["np"])
        return dict(bytes=3.0 * by + 8.0 * n, flops=3.0 * fl)
    return dict(bytes=8.0 * 5 * n, flops=60.0 * n)


# -- float64 from plain torch and numpy ------------------------------------------
def _t(v):
    return torch.as_tensor(np.ascontiguousarray(v, dtype=np.float64), device=DEV)


def _factors(mesh):
    """The operator's 1-D factors (r, theta, phi)."""
    drh, cr = mesh.drh[1:-1], mesh.r ** 2 / mesh.dr
    sd, cp = (mesh.sth * mesh.dth)[1:-1], (mesh.dth / mesh.sth)[1:-1]
    ct = mesh.st / mesh.dt
    return drh, cr, sd, cp, ct, mesh.dph[1:-1], 1.0 / mesh.dp[:-1]


def _couplings(mesh, pm):
    """((k, j, i) lower, (k, j, i) upper couplings, diagonal) on the GPU, (c, b, a)."""
    drh, cr, sd, cp, ct, dph, rdp = _factors(mesh)
    o = lambda k, j, i: (_t(k)[:, None, None] * _t(j)[:, None]) * _t(i)  # noqa: E731
    low = [-o(rdp[:-1], cp, drh), -o(dph, ct[:-1], drh), -o(dph, sd, cr[:-1])]
    up = [-o(rdp[1:], cp, drh), -o(dph, ct[1:], drh), -o(dph, sd, cr[1:])]
    return low, up, -(sum(low) + sum(up))


def _solution(mesh, pm, br0):
    """x (c, b, a) of the boundary-value problem: FFT in phi, eigenbasis in r,
    tridiagonal in theta (pm = +1, singular: the solution without constant)."""
    import scipy.linalg
    drh, cr, sd, cp, ct, dph, _ = _factors(mesh)
    a, b, c = drh.size, sd.size, dph.size
    h = float(dph[0])
    d = cr[:-1] + cr[1:]
    d[0] = cr[1]
    d[-1] = cr[-2] + (1.0 - pm) * cr[-1]
    R = np.diag(d) - np.diag(cr[1:-1], 1) - np.diag(cr[1:-1], -1)
    mu, V = scipy.linalg.eigh(R, np.diag(drh))
    g = _t(br0[1:-1, 1:-1].T * (sd * h)) * (-cr[0] * mesh.dr[0])  # rhs at i = 0, (c, b)
    G = torch.fft.rfft(g, dim=0)
    m = torch.arange(c // 2 + 1, dtype=torch.float64, device=DEV)
    lam = (2.0 - 2.0 * torch.cos(2.0 * math.pi * m / c)) / h
    ct = ct.copy()
    ct[0] = ct[-1] = 0.0  # no flux through the poles
    dj, e = _t(h * (ct[:-1] + ct[1:])), -h * ct
    mu_t = _t(mu)
    if pm > 0:
        mu_t[0] = 0.0
    cpt, sdt, v0 = _t(cp), _t(sd), _t(V[0])
    dg = lambda j: dj[j] + cpt[j] * lam[:, None] + h * sdt[j] * mu_t  # noqa: E731
    w = torch.empty((b, m.numel(), a), dtype=torch.complex128, device=DEV)
    q = torch.empty((b, m.numel(), a), dtype=torch.float64, device=DEV)
    for j in range(b):
        rhs, den = G[:, j, None] * v0, dg(j)
        if j:
            rhs, den = rhs - e[j] * w[j - 1], den - e[j] * q[j - 1]
        if pm > 0 and j == b - 1:
            den[0, 0] = math.inf  # the constant
        q[j], w[j] = e[j + 1] / den, rhs / den
    for j in range(b - 2, -1, -1):
        w[j] -= q[j] * w[j + 1]
    del q
    x = torch.empty((c, b, a), dtype=torch.float64, device=DEV)
    for j in range(b):
        x[:, j] = torch.fft.irfft(w[j], n=c, dim=0) @ _t(V.T)
    if pm > 0:
        vol = _t(dph)[:, None, None] * _t(sd)[:, None] * _t(drh)
        x -= (x * vol).sum() / vol.sum()
    return x


def _phi(mesh, pm, br0, x):
    """The padded potential (np, nt, nr): boundary values, poles, seam."""
    phi = torch.empty((mesh.np, mesh.nt, mesh.nr), dtype=torch.float64, device=DEV)
    phi[1:-1, 1:-1, 1:-1] = x
    i = phi[1:-1, 1:-1]
    i[..., 0] = i[..., 1] - _t(br0.T)[1:-1, 1:-1] * mesh.dr[0]
    i[..., -1] = pm * i[..., -2]
    for row, inner in ((0, 1), (-1, -2)):
        s = (phi[1:-1, inner] * _t(mesh.dph)[1:-1, None]).sum(0) / (2.0 * math.pi)
        phi[1:-1, row] = 2.0 * s - phi[1:-1, inner]
    phi[0], phi[-1] = phi[-2], phi[1]
    return phi


def _b(mesh, phi):
    rh, sth = _t(mesh.rh), _t(mesh.sth)[:, None]
    br = (phi[..., 1:] - phi[..., :-1]) / _t(mesh.dr)
    bt = (phi[:, 1:] - phi[:, :-1]) / (rh * _t(mesh.dt)[:, None])
    bp = (phi[1:] - phi[:-1]) / (rh * sth * _t(mesh.dp)[:-1, None, None])
    return br, bt, bp


def _energy(mesh, phi):
    br, bt, bp = _b(mesh, phi)
    dv = (_t(mesh.dph)[1:-1, None, None] * _t(mesh.dth * mesh.sth)[1:-1, None]
          * _t(mesh.rh ** 2 * mesh.drh)[1:-1])
    av = (0.5 * (br[1:-1, 1:-1, 1:] + br[1:-1, 1:-1, :-1]),
          0.5 * (bt[1:-1, 1:, 1:-1] + bt[1:-1, :-1, 1:-1]),
          0.5 * (bp[1:, 1:-1, 1:-1] + bp[:-1, 1:-1, 1:-1]))
    return torch.stack([(0.5 * v * v * dv).sum() for v in av])


def _ilu_apply(mesh, r):
    """The ILU(0) solve of _csr's FP32 matrix in float64, by hyperplanes."""
    low, up, diag = _couplings(mesh, -1.0)
    low, up, diag = [[t.float().double().reshape(-1) for t in v] for v in (low, up, [diag])]
    c, b, a = mesh.np - 2, mesh.nt - 2, mesh.nr - 2
    n, ab = a * b * c, a * b
    p = torch.arange(n, device=DEV)
    i, j, k = p % a, (p // a) % b, p // ab
    order = torch.argsort(i + j + k, stable=True)
    ends = torch.cumsum(torch.bincount(i + j + k, minlength=a + b + c - 2), 0).tolist()
    levels = [order[s:e] for s, e in zip([0] + ends[:-1], ends)]
    pad = lambda on, q: torch.where(on, q, torch.full_like(q, n))  # noqa: E731
    lo = [pad(k > 0, p - ab), pad(j > 0, p - a), pad(i > 0, p - 1), pad(k == c - 1, p % ab)]
    hi = [pad(k < c - 1, p + ab), pad(j < b - 1, p + a), pad(i < a - 1, p + 1),
          pad(k == 0, p + n - ab)]
    cl, cu = low + [up[0]], up + [low[0]]
    dinv, y, z = (torch.zeros(n + 1, dtype=torch.float64, device=DEV) for _ in range(3))
    for q in levels:
        dinv[q] = 1.0 / (diag[0][q] - sum(v[q] ** 2 * dinv[s[q]] for s, v in zip(lo, cl)))
    for q in levels:
        y[q] = r[q] - sum(v[q] * dinv[s[q]] * y[s[q]] for s, v in zip(lo, cl))
    for q in reversed(levels):
        z[q] = (y[q] - sum(v[q] * z[s[q]] for s, v in zip(hi, cu))) * dinv[q]
    return z[:n]


def _conv(x, W, bias):
    """3x3x3 convolution of x (Z, Y, X, C): periodic in z, zero-padded in y, x."""
    Z, Y, X, C = x.shape
    xp = torch.nn.functional.pad(torch.cat([x[-1:], x, x[:1]]), (0, 0, 1, 1, 1, 1))
    y = bias
    for t in range(27):
        dx, dy, dz = t % 3, (t // 3) % 3, t // 9
        y = y + xp[dz:dz + Z, dy:dy + Y, dx:dx + X].reshape(-1, C) @ W[t].T
    return y.reshape(Z, Y, X, -1)


def _pool(x):
    Z, Y, X, _ = x.shape
    odd = (0, 0, 0, X % 2, 0, Y % 2, 0, Z % 2)
    one = torch.nn.functional.pad(torch.ones((Z, Y, X, 1), dtype=x.dtype, device=DEV), odd)
    s = lambda t: sum(t[u::2, v::2, w::2] for u in (0, 1) for v in (0, 1) for w in (0, 1))  # noqa: E731
    return s(torch.nn.functional.pad(x, odd)) / s(one)


def _up(x, like):
    Z, Y, X, _ = like.shape
    i = lambda n: torch.arange(n, device=DEV) // 2  # noqa: E731
    return x[i(Z)][:, i(Y)][:, :, i(X)]


def _forward(mesh, br0, params):
    """The network's output (c, b, a) and the scale of its target."""
    scale = float(np.sqrt(np.mean(br0[1:-1, 1:-1] ** 2)))
    bb = (_t(br0[1:-1, 1:-1].T) / scale)[..., None]
    rh = mesh.rh
    r = _t(rh[1:-1])
    c, b, a = mesh.np - 2, mesh.nt - 2, mesh.nr - 2
    r0, r1 = 0.5 * (rh[0] + rh[1]), 0.5 * (rh[-2] + rh[-1])
    x0 = torch.zeros((c, b, a, 16), dtype=torch.float64, device=DEV)
    x0[..., 0], x0[..., 1] = bb * (r0 / r) ** 2, bb
    x0[..., 2] = (r - r0) / (r1 - r0)
    W, at = [], 0
    for ci, co, _ in _CONVS:
        W.append((params[at:at + 27 * ci * co].reshape(27, co, ci),
                  params[at + 27 * ci * co:at + 27 * ci * co + co]))
        at += 27 * ci * co + co
    f = lambda x, i: torch.relu(_conv(x, *W[i]))  # noqa: E731
    e0 = f(x0, 0)
    e1 = f(_pool(e0), 1)
    e2 = f(_pool(e1), 2)
    e3 = f(_pool(e2), 3)
    s2 = f(_up(e3, e2), 4) + e2
    s1 = f(_up(s2, e1), 5) + e1
    s0 = f(_up(s1, e0), 6) + e0
    return _conv(s0, *W[7])[..., 0], scale


def _predicted(mesh, fmesh, br0):
    z = np.load(WEIGHTS, allow_pickle=False)
    with torch.no_grad():
        out, scale = _forward(mesh, br0, _t(z["params"]))
    phi = _phi(mesh, -1.0, br0, out * (scale * float(z["phiscale"])))
    for dim, (cv, fv) in enumerate(((mesh.ph, fmesh.ph), (mesh.th, fmesh.th),
                                    (mesh.rh, fmesh.rh))):
        v = fv[1:-1]
        i = np.clip(np.searchsorted(cv, v, side="right") - 1, 0, cv.size - 2)
        w = _t((v - cv[i]) / (cv[i + 1] - cv[i])).reshape([-1 if q == dim else 1 for q in range(3)])
        lo = torch.as_tensor(i, device=DEV)
        phi = (1.0 - w) * phi.index_select(dim, lo) + w * phi.index_select(dim, lo + 1)
    return phi.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "readbr":
        mesh = _mesh(32, case["nt"], case["np"], case["option"])
        v = _readbr(mesh, case["option"], *_map(case["option"], seed, case["ntn"], case["npn"]))
        return dict(zip(("br0", "fluxp", "fluxm", "area", "br00err"), v))
    option = case.get("option", "ss")
    mesh = _mesh(case["nr"], case["nt"], case["np"], option)
    if kind == "extlu":
        return _ilu_apply(mesh, _residual(case, seed))
    pm = inputs.pm_r1_for(option)
    br0 = _br0(mesh, option, seed)
    if kind == "guess":
        return _predicted(mesh, _mesh(case["fnr"], case["fnt"], case["fnp"], "ss"), br0)
    if kind == "potfld" and pm > 0:
        # the constant of a Neumann solution is the iteration's own; its energy is not
        phi = _phi(mesh, pm, br0, _solution(mesh, pm, br0))
        return dict(x=None, phi=None, energy=_energy(mesh, phi), ierr=None)
    x = _solution(mesh, pm, br0)
    if kind == "solve":
        return dict(x=x.reshape(-1), ierr=None)
    if kind == "train":
        z = np.load(WEIGHTS, allow_pickle=False)
        params = _t(z["params"]).requires_grad_(True)
        out, scale = _forward(mesh, br0, params)
        loss = torch.mean((out - x / (scale * float(z["phiscale"]))) ** 2)
        loss.backward()
        return dict(loss=loss.detach(), grads=params.grad)
    phi = _phi(mesh, pm, br0, x)
    w = _energy(mesh, phi)
    if kind == "potfld":
        return dict(x=x.reshape(-1), phi=phi.reshape(-1), energy=w, ierr=None)
    br, bt, bp = _b(mesh, phi)
    return dict(phi=phi.reshape(-1), energy=w, br=br.reshape(-1), bt=bt.reshape(-1),
                bp=bp.reshape(-1))
