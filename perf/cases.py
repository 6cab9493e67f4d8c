"""The workloads this framework's speed is measured on, with their inputs, the
work that cannot be left out, tolerances and a plain 64-bit restatement.

A case is one whole run of a CANS time loop ``cfl_m -> t=t+dt -> engine ->
bnd`` from a given initial state (or the gradient through one), called as a
program calls the package: the initial state goes into the run's buffers, the
steps run, the final state and time come back.  Kinds:

  tube1d   one Brio-Wu tube, 1D mlw_m, free ends: the smallest runs, bound by
           launches and latency (cans1d/md_mhdshktb)
  spicule  the UTRIP flux-tube loop (cans1d/md_spicule) of a few realizations
  calls2d  a main.f loop that calls the routines one by one (cfl_m, roe_m and
           one bd* call per field and face), 2D Roe-MUSCL in a periodic box
  box2d    Orszag-Tang vortex, 2D mlw_m in a periodic box (the benchmark)
  open2d   2D mlw_m on a stretched grid between a mirror wall and free faces,
           the boundaries of most CANS models
  box25d   the three-component 2D mlw_m3 in a periodic box
  runs2d   many uneven periodic 2D runs in one call, each to its own end
  mlw3d    3D blast wave, mlw_m, periodic box
  roe3d    the same, Roe-MUSCL in FP64
  hlld3d   the same, HLLD with FP32 face fluxes
  cyl3d    3D mlw_m_c in cylindrical (r, phi, z) coordinates, periodic in phi
  grad2d   forward and backward of the final density of the 2D mlw_m loop
"""
import math

import numpy as np
import torch

from utrip_amd import cans, problems, spicule
from utrip_amd.adjoint import FinalDensity, PeriodicMlwAdjoint

PI = math.pi
GM = 5.0 / 3.0
SQ4PI = math.sqrt(4.0 * PI)
F4_PI = float(np.float32(PI))           # REAL*4 acos(-1.0) of the 3D cfl_m
F4_1EM4 = float(np.float32(1.0e-4))     # REAL*4 1.0e-4 of the artificial viscosity
QAV = 3.0

FRE, SPP, SPN, PER = cans.BD_FRE, cans.BD_SPP, cans.BD_SPN, cans.BD_PER


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one tube of the benchmark's shock-tube size: 1028 cells a step
        dict(name="tube1d_1024", kind="tube1d", nx=1024, margin=2, steps=200),
        # the shipped spicule model, 1026 cells, one realization
        dict(name="spicule_1026", kind="spicule", nx=1026, runs=1, steps=400),
        # a main.f that calls cfl_m, roe_m and bd* itself, an ordinary 2D size
        dict(name="calls2d_roe_512", kind="calls2d", nx=512, ny=512, margin=3, steps=4),
        # the benchmark's grid
        dict(name="box2d_1024", kind="box2d", nx=1024, ny=1024, margin=1, steps=40),
        # an odd, ragged model grid with walls and free faces
        dict(name="open2d_603x401", kind="open2d", nx=603, ny=401, margin=1, steps=40),
        # the benchmark's 2.5D grid
        dict(name="box25d_1024", kind="box25d", nx=1024, ny=1024, margin=1, steps=15),
        # a parameter study: runs of 32-256 cells a side, 3-80 steps each
        dict(name="runs2d_192", kind="runs2d", nx=256, ny=32, margin=1, runs=192, tend=0.2),
        # the blast wave of the benchmark on grids that one step fills the card with
        dict(name="mlw3d_256", kind="mlw3d", nx=256, ny=256, nz=256, margin=2, steps=3),
        dict(name="roe3d_192", kind="roe3d", nx=192, ny=192, nz=192, margin=3, steps=3),
        dict(name="hlld3d_mixed_192", kind="hlld3d", nx=192, ny=192, nz=192, margin=3, steps=3),
        # a cylindrical stellar-wind sized grid (r, phi, z)
        dict(name="cyl3d_160x64x128", kind="cyl3d", nx=160, ny=64, nz=128, margin=1, steps=3),
        # gradient of the final density, checkpoints every 20 steps
        dict(name="grad2d_256", kind="grad2d", nx=256, ny=256, margin=1, steps=40, ckpt=20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tube1d", "spicule", "calls2d", "box2d", "open2d", "box25d", "runs2d", "mlw3d", "roe3d",
                       "hlld3d", "cyl3d", "grad2d"])
    if kind == "tube1d":
        return dict(kind=kind, nx=_log(rng, 200, 8000), margin=rng.choice([1, 2]), steps=rng.randint(100, 200))
    if kind == "spicule":
        return dict(kind=kind, nx=rng.randint(800, 1100), runs=_log(rng, 1, 64), steps=rng.randint(200, 400))
    if kind == "calls2d":
        return dict(kind=kind, nx=_log(rng, 100, 640), ny=_log(rng, 100, 640), margin=3, steps=rng.randint(2, 4))
    if kind in ("box2d", "box25d"):
        return dict(kind=kind, nx=_log(rng, 90, 1500), ny=_log(rng, 90, 1500), margin=rng.choice([1, 2]),
                    steps=rng.randint(10, 15))
    if kind == "open2d":
        return dict(kind=kind, nx=_log(rng, 90, 1100), ny=_log(rng, 90, 1100), margin=rng.choice([1, 2]),
                    steps=rng.randint(20, 40))
    if kind == "runs2d":
        return dict(kind=kind, nx=rng.randint(96, 256), ny=rng.randint(24, 64), margin=1, runs=_log(rng, 32, 192),
                    tend=round(rng.uniform(0.05, 0.2), 4))
    if kind in ("mlw3d", "roe3d", "hlld3d"):
        n = [_log(rng, 48, 190) for _ in range(3)]
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], margin=2 if kind == "mlw3d" else 3, steps=rng.randint(1, 3))
    if kind == "cyl3d":
        return dict(kind=kind, nx=_log(rng, 48, 160), ny=_log(rng, 24, 96), nz=_log(rng, 48, 160), margin=1,
                    steps=rng.randint(1, 3))
    return dict(kind=kind, nx=_log(rng, 64, 320), ny=_log(rng, 64, 320), margin=1, steps=rng.randint(10, 40),
                ckpt=rng.choice([0, 20]))


# ------------------------------------------------------------------ inputs
def _centres(n, margin, lo, hi):
    return lo + (np.arange(n + 2 * margin) - margin + 0.5) * ((hi - lo) / n)


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64).cuda()


def _spacings(x):
    """Cell and face spacings dx, dxm and face positions xm of cell positions x (grdrdy)."""
    dxm = np.append(x[1:] - x[:-1], x[-1] - x[-2])
    dx = 0.5 * (dxm[:-2] + dxm[1:-1])
    dx = np.concatenate([dx[:1], dx, dx[-1:]])
    xm = np.append(0.5 * (x[:-1] + x[1:]), 0.5 * (x[-2] + x[-1]) + dx[-1])
    return dx, dxm, xm


def _metric(x):
    dx, dxm, _ = _spacings(x)
    return _dev(dx), _dev(dxm)


def _waves(rng, amp, *axes):
    """A smooth random field on [0, 2 pi) periodic axes (x last): a few long waves."""
    out = 0.0
    for _ in range(6):
        ph = sum(float(rng.integers(-2, 3)) * a for a in axes)
        out = out + amp * float(rng.uniform(0.3, 1.0)) * torch.sin(ph + float(rng.uniform(0, 2 * PI)))
    return out


def _fill_per(q, margin, dims):
    for d in dims:
        n = q.shape[d]
        q.narrow(d, 0, margin).copy_(q.narrow(d, n - 2 * margin, margin).clone())
        q.narrow(d, n - margin, margin).copy_(q.narrow(d, margin, margin).clone())


def _vortex(nx, ny, margin, rng, comp3=False, pscale=1.0):
    """The Orszag-Tang vortex with seeded long waves on its velocities and
    pressure, and its grid; tensors (ny, nx) with periodic ghosts filled."""
    x, y = _centres(nx, margin, 0.0, 2 * PI), _centres(ny, margin, 0.0, 2 * PI)
    X, Y = _dev(x)[None, :], _dev(y)[:, None]
    one = torch.ones_like(X + Y)
    ro = one * (25.0 / (36.0 * PI))
    pr = one * (5.0 / (12.0 * PI) * pscale) * (1.0 + _waves(rng, 0.02, X, Y))
    vx = -torch.sin(Y) * one + _waves(rng, 0.03, X, Y)
    vy = torch.sin(X) * one + _waves(rng, 0.03, X, Y)
    bx, by = -torch.sin(Y) * one, torch.sin(2.0 * X) * one
    az = (torch.cos(Y) + 0.5 * torch.cos(2.0 * X)) * one
    f = [ro, pr, vx, vy, bx, by, az]
    if comp3:
        f = [ro, pr, vx, vy, 0.2 * torch.sin(X + Y), bx, by, 0.3 * torch.cos(X - Y), az]
    f = [(q * one).contiguous() for q in f]
    for q in f:
        _fill_per(q, margin, (1, 0))
    return f, (x, y)


def _blast(nx, ny, nz, margin, rng, gauss):
    """An over-pressure sphere in a periodic box, with seeded long waves on the
    velocities; tensors (nz, ny, nx)."""
    h = 1.0 / max(nx, ny, nz)
    ax = [_centres(n, margin, 0.0, n * h) for n in (nx, ny, nz)]
    X, Y, Z = _dev(ax[0])[None, None, :], _dev(ax[1])[None, :, None], _dev(ax[2])[:, None, None]
    c = [0.5 * n * h for n in (nx, ny, nz)]
    r2 = (X - c[0]) ** 2 + (Y - c[1]) ** 2 + (Z - c[2]) ** 2
    one = torch.ones_like(r2)
    P = [2 * PI * q / (n * h) for q, n in ((X, nx), (Y, ny), (Z, nz))]
    b0 = (SQ4PI if gauss else 1.0) / math.sqrt(2.0)
    r0 = 0.3 * min(nx, ny, nz) * h
    f = [one, torch.where(r2 < r0 * r0, 10.0 * one, 0.1 * one), _waves(rng, 0.02, *P) * one,
         _waves(rng, 0.02, *P) * one, _waves(rng, 0.02, *P) * one, one * b0, one * b0, one * 0.0]
    f = [q.clone().contiguous() for q in f]
    for q in f:
        _fill_per(q, margin, (2, 1, 0))
    return f, ax


def _inputs(case, seed):
    """State (list of tensors), axes (cell positions), boundary kinds per
    (axis, side, field) or None, engine constants."""
    rng = np.random.default_rng(seed)
    k, m = case["kind"], case.get("margin", 1)
    if k == "tube1d":
        pb = problems.shock_tube_1d(nx=case["nx"], margin=m, p_l=float(rng.uniform(0.8, 1.2)),
                                    x0=float(rng.uniform(0.4, 0.6)))
        f = [_dev(pb.fields[q]) for q in ("ro", "pr", "vx", "vy", "by")]
        return dict(f=f, axes=[pb.grid["x"]], bc=[FRE] * 10, gm=2.0, bx=_dev(pb.fields["bx"]),
                    bxm=_dev(pb.fields["bxm"]))
    if k in ("box2d", "calls2d", "grad2d"):
        f, axes = _vortex(case["nx"], case["ny"], m, rng)
        return dict(f=f, axes=axes, bc=[PER] * 28, gm=GM)
    if k == "box25d":
        f, axes = _vortex(case["nx"], case["ny"], m, rng, comp3=True)
        return dict(f=f, axes=axes, bc=[PER] * 36, gm=GM)
    if k == "open2d":
        # mirror wall below (vy, bx odd), free faces elsewhere, y cells growing upwards
        nx, ny = case["nx"], case["ny"]
        x = _centres(nx, m, 0.0, 4.0)
        dy = np.full(ny + 2 * m, 4.0 / nx) * (1.0 + 0.5 * np.arange(ny + 2 * m) / ny)
        y = np.cumsum(dy) - dy[:m].sum() - 0.5 * dy[m]
        X, Y = _dev(x)[None, :] - 2.0, _dev(y)[:, None]
        one = torch.ones_like(X + Y)
        top = float(y[-1])
        ro = torch.exp(-Y.abs() / top) * one
        pr = (0.6 * ro + 2.0 * torch.exp(-(X ** 2 + (Y - 0.3 * top) ** 2) / (0.1 * top) ** 2)) * one
        wx, wy = (X + 2.0) * (PI / 2), Y * (2 * PI / top)
        f = [ro, pr, _waves(rng, 0.05, wx, wy) * one, _waves(rng, 0.05, wx, wy) * one, 0.3 * one * (Y > 0),
             1.5 * one, -1.5 * X * one]
        f = [q.clone().contiguous() for q in f]
        lo = [SPP, SPP, SPP, SPN, SPN, SPP, SPP]
        bc = [FRE] * 14 + lo + [FRE] * 7
        _fill(f, bc, m)
        return dict(f=f, axes=[x, y], bc=bc, gm=GM)
    if k in ("mlw3d", "roe3d", "hlld3d"):
        f, axes = _blast(case["nx"], case["ny"], case["nz"], m, rng, gauss=k != "hlld3d")
        return dict(f=f, axes=axes, bc=[PER] * 48, gm=GM)
    if k == "cyl3d":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        x, y, z = _centres(nx, m, 1.0, 3.0), _centres(ny, m, 0.0, 2 * PI), _centres(nz, m, -1.0, 1.0)
        X, Y, Z = _dev(x)[None, None, :], _dev(y)[None, :, None], _dev(z)[:, None, None]
        one = torch.ones_like(X + Y + Z)
        ro = one / X ** 2
        pr = 0.5 * ro + torch.exp(-((X - 2.0) ** 2 + Z ** 2 + (1.0 - torch.cos(Y))) / 0.1)
        w = [(X - 1.0) * PI, Y, (Z + 1.0) * PI]
        f = [ro, pr, 0.5 * one + _waves(rng, 0.05, *w), _waves(rng, 0.05, *w), _waves(rng, 0.05, *w),
             2.0 / X, 0.5 / X, one]
        f = [(q * one).contiguous() for q in f]
        bc = [FRE] * 16 + [PER] * 16 + [FRE] * 16
        _fill(f, bc, m)
        return dict(f=f, axes=[x, y, z], bc=bc, gm=GM)
    raise ValueError(k)


def _run_sizes(case):
    """Sizes, pressure scales of the runs of a runs2d case (not of the seed:
    the same study with other perturbations)."""
    r = np.random.default_rng(20160811)
    lo, hi, n = case["ny"], case["nx"], case["runs"]
    return (r.integers(lo, hi + 1, n), r.integers(lo, hi + 1, n), 10.0 ** r.uniform(-1.0, 1.0, n))


def _runs(case, seed):
    rng = np.random.default_rng(seed)
    return [_vortex(int(a), int(b), case["margin"], rng, pscale=float(p)) for a, b, p in zip(*_run_sizes(case))]


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    k = case["kind"]
    s = dict(kind=k, case=dict(case))
    if k == "spicule":
        rng = np.random.default_rng(seed)
        seeds = [int(v) for v in rng.integers(1, 2 ** 31 - 1, case["runs"])]
        r = spicule.SpiculeRuns(spicule.setup(case["nx"], 1), seeds)
        s.update(run=r, seed0=r.seed.clone(), init=[t.clone() for t in r.f])
        return s
    if k == "runs2d":
        runs = []
        for f, axes in _runs(case, seed):
            d = {q: t.cpu().numpy().T for q, t in zip(cans.Batch2D.FIELDS, f)}
            for n, a in zip("xy", axes):
                d["d" + n], d[f"d{n}m"], _ = _spacings(a)
            runs.append(d)
        b = cans.Batch2D(runs, GM, QAV, 0.4, case["margin"], tune_room=False)
        s.update(run=b, init=[t.clone() for t in b.f])
        return s
    v = _inputs(case, seed)
    s["init"] = v["f"]
    g = {}
    for n, a in zip("xyz", v["axes"]):
        g["d" + n], g[f"d{n}m"] = _metric(a)
    s["grid"] = g
    state = [t.clone() for t in v["f"]]
    m = case["margin"]
    if k == "tube1d":
        s["run"] = cans.Run(1, cans.ENGINE_MLW, state, g, 2.0, 0.4, qav=QAV, margin=m, bc=v["bc"], bx1d=v["bx"],
                            bxm1d=v["bxm"])
    elif k == "box2d":
        s["run"] = cans.MlwRun2D(state, g["dx"], g["dxm"], g["dy"], g["dym"], QAV, GM, 0.4, margin=m)
    elif k == "open2d":
        s["run"] = cans.MlwRun2D(state, g["dx"], g["dxm"], g["dy"], g["dym"], QAV, GM, 0.4, margin=m, bc=v["bc"])
    elif k == "box25d":
        s["run"] = cans.Run(2, cans.ENGINE_MLW3, state, g, GM, 0.4, qav=QAV, margin=m, bc=v["bc"])
    elif k in ("mlw3d", "roe3d", "hlld3d"):
        e = dict(mlw3d=cans.ENGINE_MLW, roe3d=cans.ENGINE_ROE, hlld3d=cans.ENGINE_HLLD)[k]
        s["run"] = cans.Run(3, e, state, g, GM, 0.4, qav=QAV, margin=m, bc=v["bc"], mixed=k == "hlld3d")
    elif k == "cyl3d":
        x = v["axes"][0]
        s["run"] = cans.Run(3, cans.ENGINE_MLWC, state, g, GM, 0.4, qav=QAV, margin=m, bc=v["bc"], bx1d=_dev(x),
                            bxm1d=_dev(_spacings(x)[2]))
    elif k == "calls2d":
        s["state"] = state
    elif k == "grad2d":
        c = (slice(m, -m), slice(m, -m))
        s["solver"] = PeriodicMlwAdjoint(g["dx"], g["dxm"], g["dy"], g["dym"], QAV, GM, 0.4, m, case["steps"],
                                         ckpt=case["ckpt"])
        s["par"] = [state[2][c].clone().requires_grad_(True), state[3][c].clone().requires_grad_(True),
                    torch.ones((), dtype=torch.float64, device="cuda", requires_grad=True)]
        s["target"] = state[0][c] * 1.1
    return s


def run(s):
    k, c = s["kind"], s["case"]
    if k == "spicule":
        r = s["run"]
        for dst, src in zip(r.f, s["init"]):
            dst.copy_(src)
        r.seed.copy_(s["seed0"])
        for q in (r.t, r.ns, r.merr):
            q.zero_()
        r.run(nstop=c["steps"])
        return [*r.f, r.t, r.ns, r.merr, r.seed]
    if k == "runs2d":
        b = s["run"]
        for dst, src in zip(b.f, s["init"]):
            dst.copy_(src)
        b.run(c["tend"])
        return [*b.f, b.t, b.ns, b.merr]
    if k == "calls2d":
        st, g, t, m = s["state"], s["grid"], 0.0, c["margin"]
        for dst, src in zip(st, s["init"]):
            dst.copy_(src)
        for _ in range(c["steps"]):
            dt, merr = cans.cfl_m_2d(0.4, 1e-10, GM, *st[:6], g["dx"], g["dy"])
            if merr:
                break
            t = t + dt
            cans.roe_m_2d(*st, dt, GM, g["dx"], g["dy"])
            for d in (0, 1):
                for q in st:
                    cans.bnd_2d(d, PER, m, m, q)
        return [*st, t]
    if k == "grad2d":
        vx, vy, beta = s["par"]
        rho = FinalDensity.apply(vx, vy, beta, s["solver"], s["init"])
        loss = 0.5 * ((rho - s["target"]) ** 2).sum()
        return [rho.detach(), *torch.autograd.grad(loss, s["par"])]
    r = s["run"]
    for dst, src in zip(r.a, s["init"]):
        dst.copy_(src)
    r.reset()
    r.steps(c["steps"])
    state, info = r.state()
    return [*state, info["t"], info["nexec"], info["merr"]]


# ------------------------------------------------------------------ work and tolerances
# Operations per cell and step: the adds, multiplies and (as one) divisions
# and roots of the scheme's formulas, counted from the loops.
_FLOPS = dict(tube1d=190, spicule=300, calls2d=2600, box2d=430, open2d=430, box25d=620, runs2d=430, mlw3d=1500,
              roe3d=6000, hlld3d=3600, cyl3d=1800, grad2d=2200)
_FIELDS = dict(tube1d=5, spicule=5, calls2d=7, box2d=7, open2d=7, box25d=9, runs2d=7, mlw3d=8, roe3d=8, hlld3d=8,
               cyl3d=8, grad2d=7)


def work(case):
    k = case["kind"]
    cells = case["nx"] * case.get("ny", 1) * case.get("nz", 1)
    steps = case.get("steps", 1)
    if k == "spicule":
        cells *= case["runs"]
    if k == "runs2d":
        nx, ny, ps = _run_sizes(case)
        # steps of a run to tend: the fastest waves over the smallest spacing
        c = np.sqrt(2.0 + GM * (5.0 / (12.0 * PI)) * ps / (25.0 / (36.0 * PI)) + 2.0 / (4 * PI * 25.0 / (36.0 * PI)))
        n = np.ceil(case["tend"] / (0.4 * 2 * PI / np.maximum(nx, ny) / c))
        cells, steps = float(np.sum(nx * ny * n)), 1
    # every step reads each field once and writes it once, 8 bytes each; the
    # backward reads the states of the trajectory and carries six adjoints
    per = 16.0 * _FIELDS[k] + (8.0 * (7 + 12) if k == "grad2d" else 0.0)
    return {"bytes": per * cells * steps, "flops": float(_FLOPS[k]) * cells * steps}


def tolerance(case):
    # Measured against exact() and taken about four times: FP64 sums in
    # another order give some 1e-15 and up to 3e-14 in the weak components; the
    # spicule's vx starts as the rounding of a hydrostatic balance (5e-7);
    # FP32 face fluxes give 9e-7 in the transverse velocities.
    if case["kind"] == "hlld3d":
        return {"rel": 4e-6}
    if case["kind"] == "spicule":
        return {"rel": 2e-6}
    return {"rel": 1e-13, "max": 1e-11}


# ------------------------------------------------------------------ plain 64-bit restatement
def _cut(q, dim, lo, hi):
    return q.narrow(dim, lo, q.shape[dim] - lo - hi)


def _dim(q, a):
    return q.dim() - 1 - a


def _along(v, q, a):
    """1D values along axis a (0 = x, the last dimension) against tensor q."""
    s = [1] * q.dim()
    s[_dim(q, a)] = v.numel()
    return v.reshape(s)


def _fill(f, bc, m):
    """bd* of every field and face, x then y then z, in place."""
    nf = len(f)
    for a in range(f[0].dim()):
        for n, q in enumerate(f):
            d, size = _dim(q, a), q.shape[_dim(q, a)]
            for side in (0, 1):
                k = bc[(2 * a + side) * nf + n]
                if k == PER:
                    if side == 0:
                        _fill_per(q, m, (d,))
                    continue
                sgn = -1.0 if k == SPN else 1.0
                for i in range(m):
                    dst = m - 1 - i if side == 0 else size - m + i
                    src = (m + i if side == 0 else size - m - 1 - i) if k in (SPP, SPN) else (m if side == 0 else size - m - 1)
                    q.select(d, dst).copy_(sgn * q.select(d, src))


def _cfl(P, grid, gm, safety):
    ro, pr, v, b = P[0], P[1], P[2:5], P[5:8]
    D = ro.dim()
    pi4i = 0.25 / (F4_PI if D == 3 else PI)
    a2 = gm * pr / ro + (b[0] ** 2 + b[1] ** 2 + b[2] ** 2) * pi4i / ro
    if D == 1:
        return torch.amin((safety * grid[0][0] / (v[0].abs() + torch.sqrt(a2)))[1:-1])
    d = _along(grid[0][0], ro, 0)
    for a in range(1, D):
        d = torch.minimum(d, _along(grid[a][0], ro, a))
    return torch.amin(safety * d / torch.sqrt(v[0] ** 2 + v[1] ** 2 + v[2] ** 2 + a2))


def _cons(P, gm, em=1.0 / (8.0 * PI)):
    ro, pr, v, b = P[0], P[1], P[2:5], P[5:8]
    v2, b2 = v[0] ** 2 + v[1] ** 2 + v[2] ** 2, b[0] ** 2 + b[1] ** 2 + b[2] ** 2
    return [ro, pr / (gm - 1.0) + 0.5 * ro * v2 + em * b2, ro * v[0], ro * v[1], ro * v[2], *b]


def _prim(u, gm, em=1.0 / (8.0 * PI)):
    v = [u[2] / u[0], u[3] / u[0], u[4] / u[0]]
    b2, v2 = u[5] ** 2 + u[6] ** 2 + u[7] ** 2, v[0] ** 2 + v[1] ** 2 + v[2] ** 2
    return [u[0], (gm - 1.0) * (u[1] - 0.5 * u[0] * v2 - em * b2), *v, u[5], u[6], u[7]]


def _efield(P):
    v, b = P[2:5], P[5:8]
    return [-v[1] * b[2] + v[2] * b[1], -v[2] * b[0] + v[0] * b[2], -v[0] * b[1] + v[1] * b[0]]


def _fluxes(P, gm, r):
    """Fluxes F[axis][equation] and sources (cylindrical: radius r) or None."""
    ro, pr, v, b = P[0], P[1], P[2:5], P[5:8]
    p4, p8 = 1.0 / (4.0 * PI), 1.0 / (8.0 * PI)
    e = _efield(P)
    ep = pr * gm / (gm - 1.0) + 0.5 * ro * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
    pt = pr + p8 * (b[0] ** 2 + b[1] ** 2 + b[2] ** 2)
    F = []
    for a in range(ro.dim()):
        n, t = (a + 1) % 3, (a + 2) % 3
        f = [ro * v[a], ep * v[a] + (b[t] * e[n] - b[n] * e[t]) * p4]
        f += [ro * v[a] * v[q] - p4 * b[a] * b[q] + (pt if q == a else 0.0) for q in range(3)]
        ind = [torch.zeros_like(ro)] * 3
        ind[n], ind[t] = -e[t], e[n]
        F.append(f + ind)
    if r is None:
        return F, None
    z = torch.zeros_like(ro)
    S = [-F[0][0] / r, -F[0][1] / r, -ro / r * (v[0] ** 2 - v[1] ** 2) + p4 / r * (b[0] ** 2 - b[1] ** 2),
         -2.0 * ro / r * v[0] * v[1] + 2.0 * p4 / r * b[0] * b[1], -F[0][4] / r, z, z, -F[0][7] / r]
    F[1] = [q / r for q in F[1]]
    return F, S


def _mean(q, axes):
    for a in axes:
        q = 0.5 * (_cut(q, _dim(q, a), 0, 1) + _cut(q, _dim(q, a), 1, 0))
    return q


def _diff(q, a):
    return _cut(q, _dim(q, a), 1, 0) - _cut(q, _dim(q, a), 0, 1)


def _inner(q, axes):
    for a in axes:
        q = _cut(q, _dim(q, a), 1, 1)
    return q


def _weigh(q, grid, axes):
    """Corner values interpolated to the cells along the axes."""
    for a in axes:
        d, dm = grid[a]
        q = (_along(0.5 * dm[1:-1] / d[1:-1], q, a) * _cut(q, _dim(q, a), 0, 1)
             + _along(0.5 * dm[:-2] / d[1:-1], q, a) * _cut(q, _dim(q, a), 1, 0))
    return q


def _put(q, new, m):
    """q with its inside (m cells from every face) replaced."""
    out = q.clone()
    out[(slice(m, -m),) * q.dim()] = new
    return out


def _mlw(P, az, dt, qav, gm, grid, r=None, rm=None):
    D = P[0].dim()
    axes = list(range(D))
    u = _cons(P, gm)
    F, S = _fluxes(P, gm, r)
    uh = []
    for q in range(8):
        h = _mean(u[q], axes)
        for a in axes:
            others = [o for o in axes if o != a]
            t = _diff(_mean(F[a][q], others), a)
            h = h - dt * t / _along(grid[a][1][:-1], t, a)
        if S is not None:
            h = h + dt * _mean(S[q], axes)
        uh.append(h)
    Ph = _prim(uh, gm)
    H, SH = _fluxes(Ph, gm, rm)
    visc = []
    for a in axes:
        dv = _diff(P[2 + a], a)
        visc.append(qav * torch.clamp(dv.abs() - F4_1EM4, min=0.0))     # q over the face's dm
    un = []
    for q in range(8):
        n = _inner(u[q], axes)
        for a in axes:
            others = [o for o in axes if o != a]
            di = _along(grid[a][0][1:-1], n, a)
            f = _inner(F[a][q], others)
            dim = _dim(f, a)
            n = n - 0.25 * dt * (_cut(f, dim, 2, 0) - _cut(f, dim, 0, 2)) / di
            n = n - 0.5 * dt * _diff(_weigh(H[a][q], grid, others), a) / di
            n = n + dt * _diff(_inner(visc[a] * _diff(u[q], a), others), a) / di
        if S is not None:
            n = n + 0.5 * dt * (_inner(S[q], axes) + _weigh(SH[q], grid, axes))
        un.append(n)
    out = [_put(q, n, 1) for q, n in zip(P, _prim(un, gm))]
    if az is not None:
        e, eh = _efield(P)[2], _efield(Ph)[2]
        az = _put(az, _inner(az, axes) - 0.5 * dt * (_inner(e, axes) + _weigh(eh, grid, axes)), 1)
    return out, az


def _minmod(a, b):
    return torch.where(a * b > 0, torch.sign(a) * torch.minimum(a.abs(), b.abs()), torch.zeros_like(a))


def _faces(P, a, muscl):
    """Left and right states of the faces along axis a (between cells c and
    c+1); minmod slopes where the face has two cells on each side."""
    L, R = [], []
    for q in P:
        d = _dim(q, a)
        lo, hi = _cut(q, d, 0, 1), _cut(q, d, 1, 0)
        if muscl:
            g = _diff(q, a)
            sl = 0.5 * _minmod(_cut(g, d, 0, 1), _cut(g, d, 1, 0))       # slopes of cells 1..n-2
            z = torch.zeros_like(q.narrow(d, 0, 1))
            sl = torch.cat([z, sl, z], dim=d)
            keep = torch.ones(q.shape[d] - 1, dtype=q.dtype, device=q.device)
            keep[0] = keep[-1] = 0.0
            keep = _along(keep, q, a)
            lo, hi = lo + keep * _cut(sl, d, 0, 1), hi - keep * _cut(sl, d, 1, 0)
        L.append(lo)
        R.append(hi)
    return L, R


def _roe_flux(L, R, a, gm, fix):
    """Linearised Roe flux along axis a, by equation of _cons (normal field 0)."""
    p4i, p8i, p4 = 1.0 / (4.0 * PI), 1.0 / (8.0 * PI), 4.0 * PI
    c = [a, (a + 1) % 3, (a + 2) % 3]
    rl, pl, rr, pr = L[0], L[1], R[0], R[1]
    vl, bl, vr, br = [L[2 + q] for q in c], [L[5 + q] for q in c], [R[2 + q] for q in c], [R[5 + q] for q in c]
    g1, g2 = gm - 1.0, (gm - 2.0) / (gm - 1.0)
    s0, s1 = torch.sqrt(rl), torch.sqrt(rr)
    si, rb = 1.0 / (s0 + s1), s0 * s1
    v = [(s0 * x + s1 * y) * si for x, y in zip(vl, vr)]
    b = [(s0 * y + s1 * x) * si for x, y in zip(bl, br)]

    def enth(ro, p, w, f):
        return 0.5 * (w[0] ** 2 + w[1] ** 2 + w[2] ** 2) + gm * p / (g1 * ro) + (b[0] ** 2 + f[1] ** 2 + f[2] ** 2) / (p4 * ro)

    hl, hr = enth(rl, pl, vl, bl), enth(rr, pr, vr, br)
    hb = (s0 * hl + s1 * hr) * si
    db = [br[1] - bl[1], br[2] - bl[2]]
    delb = g2 * (db[0] ** 2 + db[1] ** 2) * si ** 2 * p8i
    v2, b2, bt = v[0] ** 2 + v[1] ** 2 + v[2] ** 2, b[0] ** 2 + b[1] ** 2 + b[2] ** 2, b[1] ** 2 + b[2] ** 2
    cs2 = g1 * (hb - 0.5 * v2 - delb - b2 * p4i / rb)
    ast = g1 * (hb - 0.5 * v2 - delb) - (gm - 2.0) * b2 * p4i / rb
    ca2, cb2 = b[0] ** 2 / (p4 * rb), bt * p4i / rb
    cf2 = 0.5 * (ast + torch.sqrt(cb2 * (ast + cs2 + ca2) + (cs2 - ca2) ** 2))
    cl2 = cs2 * ca2 / cf2
    cf, cl, ca, cs = torch.sqrt(cf2), torch.sqrt(cl2), torch.sqrt(ca2), torch.sqrt(cs2)
    sp = (bt - 1e-12 >= 0).to(bt.dtype)
    rbt, sqh = torch.sqrt(1.0 / (bt + 1.0 - sp)), math.sqrt(0.5)
    ty, tz = sp * b[1] * rbt + sqh * (1.0 - sp), sp * b[2] * rbt + sqh * (1.0 - sp)
    sp2 = (bt / (p4 * rb) + (ca2 - cs2).abs() - 1e-12 >= 0).to(bt.dtype)
    den = torch.clamp(cf2 - cl2, min=0.0) + 1.0 - sp2
    af = sp2 * torch.sqrt(torch.clamp(cf2 - ca2, min=0.0) / den) + 1.0 - sp2
    al = sp2 * torch.sqrt(torch.clamp(cf2 - cs2, min=0.0) / den) + ((1.0 - sp2) if fix else 0.0)
    sg = torch.copysign(torch.ones_like(b[0]), b[0])
    dvx = vr[0] - vl[0]
    ent = (dvx + dvx.abs()) * 0.25

    def lam(x):
        return -torch.maximum(x.abs(), ent)

    t1 = ty * db[0] + tz * db[1]
    t2 = (pr - pl + (0.5 * (bl[1] + br[1]) * db[0] + 0.5 * (bl[2] + br[2]) * db[1]) * p4i
          + (gm - 2.0) * (b[1] * db[0] + b[2] * db[1]) * p4i) / g1
    t3 = tz * db[0] - ty * db[1]
    dy, dz = rb * (vr[1] - vl[1]), rb * (vr[2] - vl[2])
    w1, w2, w3 = rb * dvx, ty * dy + tz * dz, tz * dy - ty * dz
    sq = torch.sqrt(p4 / rb)
    p11, p12, p21, p22 = al * cf * sq, -af * cs2 / cf * sq, af * (cf2 - cs2 * g2), al * (cl2 - cs2 * g2)
    q11, q12, q21, q22 = af * cf, al * cl, -al * ca * sg, af * cs * sg
    dp, dq = p11 * p22 - p12 * p21, q11 * q22 - q12 * q21
    a1, b1 = (p22 * t1 - p12 * t2) / dp, (q22 * w1 - q12 * w2) / dq
    a2, bb = (-p21 * t1 + p11 * t2) / dp, (-q21 * w1 + q11 * w2) / dq
    wf, mf, ws, ms = 0.5 * (a1 + b1), 0.5 * (a1 - b1), 0.5 * (a2 + bb), 0.5 * (a2 - bb)
    sr = torch.sqrt(rb * p4i)
    wa, ma = 0.5 * (sr * t3 - sg * w3), 0.5 * (sr * t3 + sg * w3)
    wz = rr - rl - af * (wf + mf) - al * (ws + ms)
    bv = ty * v[1] + tz * v[2]
    z = torch.zeros_like(rl)
    e0 = 0.5 * v2 + delb

    def phys(ro, p, w, f, h):
        return [ro * w[0], ro * w[0] * h - b[0] * (b[0] * w[0] + f[1] * w[1] + f[2] * w[2]) * p4i,
                ro * w[0] ** 2 + p + (-b[0] ** 2 + f[1] ** 2 + f[2] ** 2) * p8i,
                ro * w[0] * w[1] - b[0] * f[1] * p4i, ro * w[0] * w[2] - b[0] * f[2] * p4i,
                w[0] * f[1] - w[1] * b[0], w[0] * f[2] - w[2] * b[0]]

    def fast(s):
        return [af, af * (e0 + s * cf * v[0] + cf2 / g1 + (cf2 - cs2) * g2) - s * al * ca * bv * sg, af * (v[0] + s * cf),
                af * v[1] - s * al * ty * ca * sg, af * v[2] - s * al * tz * ca * sg, al * ty * cf * sq, al * tz * cf * sq]

    def slow(s):
        return [al, al * (e0 + s * cl * v[0] + cl2 / g1 + (cl2 - cs2) * g2) + s * af * cs * bv * sg, al * (v[0] + s * cl),
                al * v[1] + s * cs * sg * af * ty, al * v[2] + s * cs * sg * af * tz, -sq * cs2 * af * ty / cf,
                -sq * cs2 * af * tz / cf]

    def alfven(s):
        return [z, -s * (tz * v[1] - ty * v[2]) * sg, z, -s * sg * tz, s * sg * ty, sq * tz, -sq * ty]

    waves = [(lam(v[0] + cf) * wf, fast(1.0)), (lam(v[0] - cf) * mf, fast(-1.0)), (lam(v[0] + cl) * ws, slow(1.0)),
             (lam(v[0] - cl) * ms, slow(-1.0)), (lam(v[0] + ca) * wa, alfven(1.0)), (lam(v[0] - ca) * ma, alfven(-1.0)),
             (lam(v[0]) * wz, [torch.ones_like(rl), e0, v[0], v[1], v[2], z, z])]
    f = [0.5 * (x + y + sum(k * w[n] for k, w in waves))
         for n, (x, y) in enumerate(zip(phys(rl, pl, vl, bl, hl), phys(rr, pr, vr, br, hr)))]
    return _frame(f, c, z)


def _frame(f, c, zero):
    """Sweep-frame fluxes (ro ee normal t1 t2 bt1 bt2) by equation of _cons."""
    out = [f[0], f[1], None, None, None, None, None, None]
    for n in range(3):
        out[2 + c[n]] = f[2 + n]
    out[5 + c[0]], out[5 + c[1]], out[5 + c[2]] = zero, f[5], f[6]
    return out


def _sweep(u, F, a, dt, grid, m):
    """u - dt dF/dx of axis a on cells m+1..n-m of that axis (every other cell as it is)."""
    d = _dim(u[0], a)
    out = []
    for q, f in zip(u, F):
        di = _along(grid[a][0][m:q.shape[d] - m], q, a)
        mid = _cut(q, d, m, m) - dt * _diff(_cut(f, d, m - 1, m - 1), a) / di
        out.append(torch.cat([q.narrow(d, 0, m), mid, q.narrow(d, q.shape[d] - m, m)], dim=d))
    return out


def _roe(P, az, dt, gm, grid):
    D = P[0].dim()
    keep = range(8) if D == 3 else (0, 1, 2, 3, 5, 6)
    u = _cons(P, gm)
    w = u
    for a in range(D):
        F = _roe_flux(*_faces(P, a, False), a, gm, D == 3)
        w = _sweep(w, F, a, 0.5 * dt, grid, 1)
    Ph = [_put(q, _inner(h, range(D)), 1) if n in keep else q for n, (q, h) in enumerate(zip(P, _prim(w, gm)))]
    w = u
    for a in range(D):
        F = _roe_flux(*_faces(Ph, a, True), a, gm, D == 3)
        w = _sweep(w, F, a, dt, grid, 2)
    new = _prim(w, gm)
    out = []
    for n, (q, h) in enumerate(zip(P, new)):
        for d in range(D):
            h = _cut(h, d, 2, 2)
        out.append(_put(q, h, 2) if n in keep else q)
    if az is not None:
        t = (az - dt * _efield(Ph)[2])[2:-2, 2:-2]
        az = _put(az, t, 2)
    return out, az


def _hlld_flux(L, R, a, gm, bn):
    c = [a, (a + 1) % 3, (a + 2) % 3]
    side = []
    for S in (L, R):
        ro, p, v, b = S[0], S[1], [S[2 + q] for q in c], [bn] + [S[5 + q] for q in c[1:]]
        pb = 0.5 * (b[0] ** 2 + b[1] ** 2 + b[2] ** 2)
        pt = p + pb
        u = [ro, p / (gm - 1.0) + 0.5 * ro * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2) + pb, ro * v[0], ro * v[1], ro * v[2],
             b[1], b[2]]
        f = [u[2], v[0] * (u[1] + pt - bn ** 2) - bn * (v[1] * b[1] + v[2] * b[2]), u[2] * v[0] + pt - bn ** 2,
             u[2] * v[1] - bn * b[1], u[2] * v[2] - bn * b[2], b[1] * v[0] - bn * v[1], b[2] * v[0] - bn * v[2]]
        gp = gm * p + 2.0 * pb
        cf = torch.sqrt((gp + torch.sqrt(gp ** 2 - 4.0 * gm * p * bn ** 2)) / (2.0 * ro))
        side.append((ro, v, b, pt, u, f, cf))
    cm = torch.maximum(side[0][6], side[1][6])
    sl = torch.minimum(side[0][1][0], side[1][1][0]) - cm
    sr = torch.maximum(side[0][1][0], side[1][1][0]) + cm
    (rl, vl, _, ptl, *_), (rr, vr, _, ptr, *_) = side
    dl, dr = sl - vl[0], sr - vr[0]
    den = dr * rr - dl * rl
    sm = (dr * rr * vr[0] - dl * rl * vl[0] - ptr + ptl) / den
    pst = (dr * rr * ptl - dl * rl * ptr + rl * rr * dr * dl * (vr[0] - vl[0])) / den
    star = []
    for (ro, v, b, pt, u, f, cf), s in zip(side, (sl, sr)):
        sd, sdm = s - v[0], s - sm
        tf = ro * sd * sdm - bn ** 2
        ok = tf.abs() > 1e-10
        tf = torch.where(ok, tf, torch.ones_like(tf))
        r1 = ro * sd / sdm
        k, g = bn * (sd - sdm) / tf, (ro * sd ** 2 - bn ** 2) / tf
        w = [torch.where(ok, x, y) for x, y in zip([r1, sm, v[1] - b[1] * k, v[2] - b[2] * k, b[1] * g, b[2] * g],
                                                   [ro, v[0], v[1], v[2], b[1], b[2]])]
        vb = w[1] * bn + w[2] * w[4] + w[3] * w[5]
        e = (sd * u[1] - pt * v[0] + pst * sm + bn * (v[0] * bn + v[1] * b[1] + v[2] * b[2] - vb)) / sdm
        e = torch.where(ok, e, u[1])
        star.append((w, vb, [w[0], e, w[0] * w[1], w[0] * w[2], w[0] * w[3], w[4], w[5]]))
    (wl, vbl, ul), (wr, vbr, ur) = star
    ql, qr, sg = torch.sqrt(wl[0]), torch.sqrt(wr[0]), torch.copysign(torch.ones_like(bn), bn)
    inv = 1.0 / (ql + qr)
    vt = [inv * (ql * wl[2 + n] + qr * wr[2 + n] + sg * (wr[4 + n] - wl[4 + n])) for n in (0, 1)]
    bt = [inv * (ql * wr[4 + n] + qr * wl[4 + n] + sg * ql * qr * (wr[2 + n] - wl[2 + n])) for n in (0, 1)]
    vb = sm * bn + vt[0] * bt[0] + vt[1] * bt[1]
    dd = []
    for w, q, v, u, s in ((wl, ql, vbl, ul, -1.0), (wr, qr, vbr, ur, 1.0)):
        x = [u[0], u[1] + s * q * sg * (v - vb), u[2], w[0] * vt[0], w[0] * vt[1], bt[0], bt[1]]
        dd.append([torch.where(bn == 0, y, z) for y, z in zip(u, x)])
    tl, tr = sm - bn.abs() / ql, sm + bn.abs() / qr
    out = []
    for n in range(7):
        fl, fr, u0, u1 = side[0][5][n], side[1][5][n], side[0][4][n], side[1][4][n]
        f = fr + sr * (ur[n] - u1)
        f = torch.where(tr > 0, f + tr * (dd[1][n] - ur[n]), f)
        left = fl + sl * (ul[n] - u0)
        f = torch.where(sm >= 0, left + tl * (dd[0][n] - ul[n]), f)
        f = torch.where(tl >= 0, left, f)
        f = torch.where(sr <= 0, fr, f)
        out.append(torch.where(sl >= 0, fl, f))
    return _frame(out, c, torch.zeros_like(bn))


def _hlld(P, dt, gm, grid):
    u = _cons(P, gm, 0.5)
    Q = P
    for stage, h in ((1, 0.5 * dt), (2, dt)):
        w = u
        for a in range(3):
            bn = _mean(Q[5 + a], (a,))
            w = _sweep(w, _hlld_flux(*_faces(Q, a, stage == 2), a, gm, bn), a, h, grid, 1)
        Q = _prim(w, gm, 0.5)
    return Q


def _loop(f, axes, bc, gm, kind, margin, steps=None, tend=None, radii=None):
    """The time loop on tensors f (fields as the package holds them)."""
    D = f[0].dim()
    grid = [_metric(a) for a in axes]
    az = None
    z = torch.zeros_like(f[0])
    if D == 1:
        pos = [0, 1, 2, 3, 6]
    elif D == 2:
        pos = [0, 1, 2, 3, 5, 6] if len(f) == 7 else list(range(8))
        az = f[-1].clone()
    else:
        pos = list(range(8))
    P = [z.clone() for _ in range(8)]
    for n, p in enumerate(pos):
        P[p] = f[n].clone()
    if kind == "tube1d":
        P[5] = radii
    r = rm = None
    if kind == "cyl3d":
        r, rm = (_along(q, z, 0) for q in radii)
        rm = rm[..., :-1]
    t, n = 0.0, 0
    while (steps is None or n < steps) and (tend is None or t < tend):
        dt = _cfl(P, grid, gm, 0.4)
        t, n = t + float(dt), n + 1
        if kind in ("roe3d", "calls2d"):
            P, az = _roe(P, az, dt, gm, grid)
        elif kind == "hlld3d":
            P = _hlld(P, dt, gm, grid)
        else:
            P, az = _mlw(P, az, dt, QAV, gm, grid, r, rm)
        new = [P[p].clone() for p in pos] + ([az.clone()] if az is not None else [])
        _fill(new, bc, margin)
        for q, p in enumerate(pos):
            P[p] = new[q]
        az = new[-1] if az is not None else None
    return [P[p] for p in pos] + ([az] if az is not None else []), t, n


def _per_fill(q, m):
    for d in (1, 0):
        q = torch.cat([q.narrow(d, q.shape[d] - 2 * m, m), q.narrow(d, m, q.shape[d] - 2 * m), q.narrow(d, m, m)], dim=d)
    return q


def _grad(case, seed):
    v = _inputs(case, seed)
    m, f, grid = case["margin"], v["f"], [_metric(a) for a in v["axes"]]
    c = (slice(m, -m), slice(m, -m))
    par = [f[2][c].clone().requires_grad_(True), f[3][c].clone().requires_grad_(True),
           torch.ones((), dtype=torch.float64, device="cuda", requires_grad=True)]
    z = torch.zeros_like(f[0])
    P = [f[0], f[1] * par[2], _per_fill(_put(f[2], par[0], m), m), _per_fill(_put(f[3], par[1], m), m), z, f[4], f[5], z]
    for _ in range(case["steps"]):
        P, _ = _mlw(P, None, _cfl(P, grid, GM, 0.4), QAV, GM, grid)
        P = [_per_fill(q, m) for q in P]
    rho = P[0][c]
    loss = 0.5 * ((rho - f[0][c] * 1.1) ** 2).sum()
    return [rho.detach(), *torch.autograd.grad(loss, par)]


def _spicule(case, seed):
    """mlw_m_bg, the torque, the mirror and free ends and the floors, in numpy
    on (realization, cell) arrays."""
    n = case["nx"]
    sp = spicule.setup(n, 1)
    seeds = np.random.default_rng(seed).integers(1, 2 ** 31 - 1, case["runs"]).astype(np.int64)
    ro, pr, vx, vy, by = (np.tile(sp.state[q], (case["runs"], 1)) for q in ("ro", "pr", "vx", "vy", "by"))
    g, gm, p4, p8 = sp.geom, sp.gm, 0.25 / PI, 0.125 / PI
    bx, bxm, dx, dxm, sc, rr = g["bx"], g["bxm"], g["dx"], g["dxm"], g["sc"], g["rr"]
    trq, pw = spicule.torque_table(sp.x), spicule.draw_powers(n)
    t = np.zeros(case["runs"])
    low = dict(gx="gx", dsc="dsc", drr="drr", sc="sc", rr="rr")
    high = dict(gx="gxm", dsc="dscm", drr="drrm", sc="scm", rr="rrm")

    def terms(ro, pr, vx, vy, by, bx, names, cut):
        q = {k: g[v][:cut] for k, v in names.items()}
        ez = -vx * by + vy * bx
        ep = pr * gm / (gm - 1.0) + 0.5 * ro * (vx * vx + vy * vy)
        F = [ro * vx * q["sc"], (ep * vx - by * ez * p4) * q["sc"], (ro * vx * vx + pr + (by * by - bx * bx) * p8) * q["sc"],
             (ro * vx * vy - bx * by * p4) * q["sc"] * q["rr"], -ez * q["sc"] / q["rr"]]
        S = [0.0 * ro, ro * vx * q["gx"] * q["sc"],
             (ro * q["gx"] + (ro * vy * vy - by * by * p4) / q["rr"] * q["drr"]) * q["sc"]
             + (pr + (by * by + bx * bx) * p8) * q["dsc"], 0.0 * ro, 0.0 * ro]
        return F, S

    for _ in range(case["steps"]):
        a2 = gm * pr / ro + (bx * bx + by * by) * p4 / ro
        dt = np.min((0.8 * dx / (np.abs(vx) + np.sqrt(a2)))[:, 1:-1], axis=1)
        t = t + dt
        d = dt[:, None]
        u = [ro * sc, (pr / (gm - 1.0) + 0.5 * ro * (vx * vx + vy * vy) + p8 * (bx * bx + by * by)) * sc, ro * vx * sc,
             ro * vy * sc * rr, by * sc / rr]
        F, S = terms(ro, pr, vx, vy, by, bx, low, None)
        h = [0.5 * (q[:, 1:] + q[:, :-1]) - d * (f[:, 1:] - f[:, :-1]) / dxm[:-1] + d * 0.5 * (s[:, 1:] + s[:, :-1])
             for q, f, s in zip(u, F, S)]
        scm, rrm = g["scm"][:-1], g["rrm"][:-1]
        rh, vxh, vyh, byh = h[0] / scm, h[2] / h[0], h[3] / h[0] / rrm, h[4] / scm * rrm
        ph = (gm - 1.0) * (h[1] / scm - 0.5 * rh * (vxh ** 2 + vyh ** 2) - p8 * (bxm[:-1] ** 2 + byh ** 2))
        H, T = terms(rh, ph, vxh, vyh, byh, bxm[:-1], high, -1)
        di, w0, w1 = dx[1:-1], 0.5 * dxm[1:-1] / dx[1:-1], 0.5 * dxm[:-2] / dx[1:-1]
        q = 1.0 * np.maximum(0.0, np.abs(vx[:, 1:] - vx[:, :-1]) - F4_1EM4)
        nu = []
        for v, f, s, fh, sh in zip(u, F, S, H, T):
            c = v[:, 1:-1] - 0.25 * d * (f[:, 2:] - f[:, :-2]) / di + 0.5 * d * s[:, 1:-1]
            c = c - 0.5 * d * (fh[:, 1:] - fh[:, :-1]) / di + 0.5 * d * (w0 * sh[:, :-1] + w1 * sh[:, 1:])
            e = q * (v[:, 1:] - v[:, :-1])
            nu.append(c + d * (e[:, 1:] - e[:, :-1]) / di)
        i = slice(1, -1)
        ro[:, i] = nu[0] / sc[i]
        vx[:, i], vy[:, i] = nu[2] / nu[0], nu[3] / rr[i] / nu[0]
        by[:, i] = nu[4] / sc[i] * rr[i]
        pr[:, i] = (gm - 1.0) * (nu[1] / sc[i] - 0.5 * ro[:, i] * (vx[:, i] ** 2 + vy[:, i] ** 2)
                                 - p8 * (bx[i] ** 2 + by[:, i] ** 2))
        noise = 2.0 * rr * ((seeds[:, None] * pw[None, :] % 2147483647) * 4.656612875245796924105750827168e-10 - 0.5)
        noise[:, -1] = noise[:, -3]
        seeds = seeds * pw[-1] % 2147483647
        vy = vy + d * 30.0 * noise * trq
        for v, sg in ((pr, 1.0), (ro, 1.0), (vx, -1.0), (vy, 1.0), (by, 1.0)):
            v[:, 0] = sg * v[:, 1]
            v[:, -1] = v[:, -2]
        for v in (ro, pr):
            vx[v < 1e-9] = 0.0
            v[v < 1e-9] = 1e-9
    return [q.reshape(-1) for q in (ro, pr, vx, vy, by)] + [t, None, None, None]


def exact(case, seed):
    k = case["kind"]
    if k == "spicule":
        return _spicule(case, seed)
    if k == "grad2d":
        return _grad(case, seed)
    if k == "runs2d":
        done = [_loop(f, axes, [PER] * 28, GM, k, case["margin"], tend=case["tend"]) for f, axes in _runs(case, seed)]
        out = [torch.cat([r[0][q].reshape(-1) for r in done]) for q in range(7)]
        return out + [torch.tensor([r[1] for r in done], dtype=torch.float64), None, None]
    v = _inputs(case, seed)
    radii = None
    if k == "tube1d":
        radii = v["bx"]
    if k == "cyl3d":
        x = v["axes"][0]
        radii = (_dev(x), _dev(_spacings(x)[2]))
    f, t, n = _loop(v["f"], v["axes"], v["bc"], v["gm"], k, case["margin"], steps=case["steps"], radii=radii)
    return f + [t] if k == "calls2d" else f + [t, None, None]
