"""GPU parity of the modified Lax-Wendroff engines, cfl_m and bnd against the
C restatement of the reference (bit-identical FP64 is the bar: the kernels
keep the reference's operation order and use no FMA contraction)."""
import numpy as np
import pytest

from tests.helpers import assert_bitwise, smooth_state_1d, smooth_state_2d, stretched_grid, to_dev, to_host
from utrip_amd import problems as P

pytestmark = pytest.mark.gpu

F1 = ("ro", "pr", "vx", "vy", "by")
F2 = ("ro", "pr", "vx", "vy", "bx", "by", "az")


def _print_case(*a):
    print("CASE", *a, flush=True)


# ----------------------------------------------------------------- 1D
@pytest.mark.parametrize("ix", [3, 5, 257, 600])
def test_mlw1d_one_call(dev, oracle, ix):
    from utrip_amd import cans
    _print_case("mlw1d one call", ix)
    s = smooth_state_1d(ix, seed=ix)
    x, dx, dxm = stretched_grid(ix, seed=ix)
    ref = {k: v.copy() for k, v in s.items()}
    oracle.mlw_m_1d(ref["ro"], ref["pr"], ref["vx"], ref["vy"], ref["by"], ref["bx"], ref["bxm"],
                    1.3e-3, 3.0, 5.0 / 3.0, dx, dxm)
    t = {k: to_dev(v, dev) for k, v in s.items()}
    cans.mlw_m_1d(t["ro"], t["pr"], t["vx"], t["vy"], t["by"], t["bx"], t["bxm"], 1.3e-3, 3.0, 5.0 / 3.0,
                  to_dev(dx, dev), to_dev(dxm, dev))
    for k in F1:
        assert_bitwise(to_host(t[k]), ref[k], k)


def _loop_1d_oracle(oracle, pb, nsteps):
    f = {k: v.copy() for k, v in pb.fields.items()}
    g, pp = pb.grid, pb.params
    m = pp["margin"]
    dts = []
    for _ in range(nsteps):
        dt, merr, _i = oracle.cfl_m_1d(pp["safety"], pp["dtmin"], pp["gm"], f["bx"], f["ro"], f["pr"], f["vx"],
                                       f["vy"], f["by"], g["dx"])
        assert merr == 0
        oracle.mlw_m_1d(f["ro"], f["pr"], f["vx"], f["vy"], f["by"], f["bx"], f["bxm"], dt, pp["qav"], pp["gm"],
                        g["dx"], g["dxm"])
        for k in F1:
            oracle.bnd_1d(0, 0, m, f[k])
            oracle.bnd_1d(0, 1, m, f[k])
        dts.append(dt)
    return f, dts


def test_mlw1d_shock_tube_dropin_loop(dev, oracle):
    """Brio-Wu (nx=1024, margin 2, bdfrex): 300 steps of the reference loop
    through the drop-in entry points."""
    from utrip_amd import cans
    _print_case("mlw1d shock tube 300 steps")
    pb = P.shock_tube_1d(nx=1024, margin=2)
    ref, dts = _loop_1d_oracle(oracle, pb, 300)
    g, pp = pb.grid, pb.params
    t = {k: to_dev(v, dev) for k, v in pb.fields.items()}
    dx, dxm = to_dev(g["dx"], dev), to_dev(g["dxm"], dev)
    gdts = []
    for _ in range(300):
        dt, merr = cans.cfl_m_1d(pp["safety"], pp["dtmin"], pp["gm"], t["bx"], t["ro"], t["pr"], t["vx"], t["vy"],
                                 t["by"], dx)
        assert merr == 0
        cans.mlw_m_1d(t["ro"], t["pr"], t["vx"], t["vy"], t["by"], t["bx"], t["bxm"], dt, pp["qav"], pp["gm"],
                      dx, dxm)
        for k in F1:
            cans.bnd_1d("fre", 0, 2, t[k])
            cans.bnd_1d("fre", 1, 2, t[k])
        gdts.append(dt)
    assert gdts == dts
    for k in F1:
        assert_bitwise(to_host(t[k]), ref[k], k)


# ----------------------------------------------------------------- 2D
@pytest.mark.parametrize("ix,jx", [(3, 3), (34, 10), (35, 11), (70, 45), (130, 67)])
def test_mlw2d_one_call(dev, oracle, ix, jx):
    from utrip_amd import cans
    _print_case("mlw2d one call", ix, jx)
    s = smooth_state_2d(ix, jx, seed=ix * 100 + jx)
    _, dx, dxm = stretched_grid(ix, seed=ix)
    _, dy, dym = stretched_grid(jx, seed=jx + 7)
    ref = {k: v.copy(order="F") for k, v in s.items()}
    oracle.mlw_m_2d(*[ref[k] for k in F2], 2.1e-3, 3.0, 5.0 / 3.0, dx, dxm, dy, dym)
    t = {k: to_dev(v, dev) for k, v in s.items()}
    cans.mlw_m_2d(*[t[k] for k in F2], 2.1e-3, 3.0, 5.0 / 3.0, to_dev(dx, dev), to_dev(dxm, dev),
                  to_dev(dy, dev), to_dev(dym, dev))
    for k in F2:
        assert_bitwise(to_host(t[k]), ref[k], k)


def _loop_2d_oracle(oracle, pb, nsteps):
    f = {k: v.copy(order="F") for k, v in pb.fields.items()}
    g, pp = pb.grid, pb.params
    m = pp["margin"]
    dts = []
    for _ in range(nsteps):
        dt, merr, _loc = oracle.cfl_m_2d(pp["safety"], pp["dtmin"], pp["gm"], f["ro"], f["pr"], f["vx"], f["vy"],
                                         f["bx"], f["by"], g["dx"], g["dy"])
        assert merr == 0
        oracle.mlw_m_2d(*[f[k] for k in F2], dt, pp["qav"], pp["gm"], g["dx"], g["dxm"], g["dy"], g["dym"])
        for k in F2:
            oracle.bnd_2d(0, 7, m, m, f[k])
        for k in F2:
            oracle.bnd_2d(1, 7, m, m, f[k])
        dts.append(dt)
    return f, dts


def test_mlw2d_ot_dropin_loop(dev, oracle):
    from utrip_amd import cans
    _print_case("mlw2d OT 96^2 drop-in 20 steps")
    pb = P.orszag_tang_2d(n=96, margin=1)
    ref, dts = _loop_2d_oracle(oracle, pb, 20)
    g, pp = pb.grid, pb.params
    t = {k: to_dev(v, dev) for k, v in pb.fields.items()}
    gd = {k: to_dev(v, dev) for k, v in g.items()}
    gdts = []
    for _ in range(20):
        dt, merr = cans.cfl_m_2d(pp["safety"], pp["dtmin"], pp["gm"], *[t[k] for k in F2[:6]], gd["dx"], gd["dy"])
        cans.mlw_m_2d(*[t[k] for k in F2], dt, pp["qav"], pp["gm"], gd["dx"], gd["dxm"], gd["dy"], gd["dym"])
        for k in F2:
            cans.bnd_2d(0, "per", 1, 1, t[k])
        for k in F2:
            cans.bnd_2d(1, "per", 1, 1, t[k])
        gdts.append(dt)
    assert gdts == dts
    for k in F2:
        assert_bitwise(to_host(t[k]), ref[k], k)


@pytest.mark.parametrize("fused", [True, False])
def test_mlw2d_ot_resident(dev, oracle, fused):
    """Resident loop (device clock, ping-pong buffers); fused = periodic
    ghost fill and next-step cfl inside the engine kernel."""
    from utrip_amd import cans
    _print_case("mlw2d OT 80x72 resident fused=", fused)
    pb = P.orszag_tang_2d(n=72, margin=1)
    # make it non-square: 80 x 72 interior
    pb = P.orszag_tang_2d(n=72, margin=1)
    nsteps = 40
    ref, dts = _loop_2d_oracle(oracle, pb, nsteps)
    g, pp = pb.grid, pb.params
    st = [to_dev(pb.fields[k], dev) for k in F2]
    gd = {k: to_dev(v, dev) for k, v in g.items()}
    bc = None if fused else [cans.BD_PER] * 28
    run = cans.MlwRun2D(st, gd["dx"], gd["dxm"], gd["dy"], gd["dym"], pp["qav"], pp["gm"], pp["safety"],
                        margin=1, bc=bc)
    run.reset(dtmin=pp["dtmin"])
    run.steps(17)
    run.steps(nsteps - 17)
    cur, info = run.state()
    assert info["nexec"] == nsteps and info["ns"] == nsteps and info["merr"] == 0
    assert info["dt"] == dts[-1]
    assert info["t"] == sum_sequential(dts)
    for k, tt in zip(F2, cur):
        assert_bitwise(to_host(tt), ref[k], k)


@pytest.mark.parametrize("margin,axis", [(1, "x"), (2, "x"), (1, "y"), (2, "y")])
def test_mlw2d_resident_periodic_ghost_cfl(dev, oracle, margin, axis):
    """Fused periodic run on a stretched grid whose smallest spacings lie in
    ghost cells (dx(1), dx(ix) or dy(1), dy(jx)): the reference's cfl_m takes
    dt from a ghost image, which the fused kernel folds into one term per
    cell."""
    from utrip_amd import cans
    from utrip_amd.problems import Problem
    _print_case("mlw2d resident periodic ghost cfl, margin", margin, "axis", axis)
    base = P.orszag_tang_2d(n=40, margin=margin)
    ix, jx = base.fields["ro"].shape
    _, dx, dxm = stretched_grid(ix, seed=11)
    _, dy, dym = stretched_grid(jx, seed=12)
    if axis == "x":
        dx[0], dx[ix - 1] = 0.3 * dx.min(), 0.35 * dx.min()
    else:
        dy[0], dy[jx - 1] = 0.35 * dy.min(), 0.3 * dy.min()
    grid = dict(base.grid, dx=dx, dxm=dxm, dy=dy, dym=dym)
    pb = Problem(base.name, base.fields, grid, base.params)
    nsteps = 12
    ref, dts = _loop_2d_oracle(oracle, pb, nsteps)
    pp = pb.params
    st = [to_dev(pb.fields[k], dev) for k in F2]
    gd = {k: to_dev(v, dev) for k, v in grid.items()}
    run = cans.MlwRun2D(st, gd["dx"], gd["dxm"], gd["dy"], gd["dym"], pp["qav"], pp["gm"], pp["safety"],
                        margin=margin)
    run.reset(dtmin=pp["dtmin"])
    run.steps(nsteps)
    cur, info = run.state()
    assert info["nexec"] == nsteps and info["merr"] == 0
    assert info["dt"] == dts[-1]
    for k, tt in zip(F2, cur):
        assert_bitwise(to_host(tt), ref[k], k)


def sum_sequential(xs):
    t = 0.0
    for x in xs:
        t = t + x
    return t


def _sides(kinds):
    """Per (axis, side, field) kinds from four per-face entries (one kind, or seven)."""
    return [k for face in kinds for k in (face if isinstance(face, (list, tuple)) else [face] * 7)]


FRE, SPP, SPN, SMP, SMN, CNS, FRD, PER = range(8)
WALL = [SPP, SPP, SPP, SPN, SPN, SPP, SPP]
BOUNDS = {
    "mirror and free": (FRE, FRE, WALL, FRE),
    "mirrors": ([SPP, SPP, SPN, SPP, SPP, SPN, SPN], SMP, SMP, WALL),
    "free and periodic": (FRE, SMP, PER, PER),
    "periodic": (PER, PER, PER, PER),
    # faces with another kind or a mixture: cfl_m, engine and fills one by one
    "mixed": ([FRE, SPP, FRE, FRE, FRE, SPP, FRE], FRE, (SMP, SMP, SMP, SMN, SMP, SMN, SMP), FRE),
    "constant and extrapolated": (FRE, FRD, PER, PER),
}


@pytest.mark.parametrize("bounds", list(BOUNDS))
@pytest.mark.parametrize("nx,ny,margin", [(70, 33, 1), (65, 128, 2), (7, 9, 3), (4, 5, 1)])
def test_mlw2d_resident_bounds(dev, oracle, bounds, nx, ny, margin):
    """Resident runs with every face kind the fused kernel maps (and two that
    it does not), signs per field, on stretched grids whose smallest
    spacings lie in ghost cells; two calls of one run through MlwRun2D and
    through Run, against cfl_m, mlw_m and the bd* of every field one after
    the other.  The initial ghosts are not yet filled."""
    from utrip_amd import cans
    _print_case("mlw2d bounds", bounds, nx, ny, margin)
    bc = _sides(BOUNDS[bounds])
    ix, jx = nx + 2 * margin, ny + 2 * margin
    s = smooth_state_2d(ix, jx, seed=ix + jx)
    _, dx, dxm = stretched_grid(ix, seed=ix)
    _, dy, dym = stretched_grid(jx, seed=jx + 7)
    dx[0], dx[-1], dy[0], dy[-1] = 0.4 * dx.min(), 0.3 * dx.min(), 0.5 * dy.min(), 0.35 * dy.min()
    f = {k: v.copy(order="F") for k, v in s.items()}
    n, dts = 5, []
    for _ in range(n):
        dt, merr, _l = oracle.cfl_m_2d(0.3, 1e-10, 5.0 / 3.0, *[f[k] for k in F2[:6]], dx, dy)
        assert merr == 0
        oracle.mlw_m_2d(*[f[k] for k in F2], dt, 3.0, 5.0 / 3.0, dx, dxm, dy, dym)
        for d in (0, 1):
            for side in (0, 1):
                for q, k in enumerate(F2):
                    kind = bc[(2 * d + side) * 7 + q]
                    if kind == PER:
                        if side == 0:
                            oracle.bnd_2d(d, PER, margin, margin, f[k])
                    else:
                        oracle.bnd_2d(d, kind, side, margin, f[k], 0.0, dxm if d == 0 else dym)
        dts.append(dt)
    gd = dict(dx=to_dev(dx, dev), dxm=to_dev(dxm, dev), dy=to_dev(dy, dev), dym=to_dev(dym, dev))
    for kind in ("MlwRun2D", "Run"):
        st = [to_dev(s[k], dev) for k in F2]
        if kind == "Run":
            run = cans.Run(2, cans.ENGINE_MLW, st, gd, 5.0 / 3.0, 0.3, qav=3.0, margin=margin, bc=bc)
        else:
            run = cans.MlwRun2D(st, gd["dx"], gd["dxm"], gd["dy"], gd["dym"], 3.0, 5.0 / 3.0, 0.3, margin=margin, bc=bc)
        run.reset(dtmin=1e-10)
        run.steps(2)
        run.steps(n - 2)
        cur, info = run.state()
        assert info["nexec"] == n and info["dt"] == dts[-1], (kind, info, dts)
        for k, t in zip(F2, cur):
            assert_bitwise(to_host(t), f[k], f"{kind} {k}")


# cell counts on both sides of each buffer class of the one-launch 1D run
# (coefficients and state in LDS, state in LDS, memory), of its block sizes
# and of its longest tube; every face kind it maps, and two it does not
@pytest.mark.parametrize("faces", [(FRE, FRE), ([SPP, SPP, SPN, SPP, SPN], FRE), (SMP, [SPP, SPP, SPN, SPN, SPP]),
                                   (FRE, SMP), (PER, PER), ([SMP, SMP, SMN, SMP, SMP], FRE), (FRE, CNS)])
@pytest.mark.parametrize("nx,margin", [(5, 1), (248, 1), (249, 3), (497, 2), (1260, 2), (1261, 2), (2028, 2), (2029, 2),
                                       (4798, 1), (4799, 1)])
def test_run_1d_bounds(dev, oracle, faces, nx, margin):
    """Resident 1D MLW runs in three calls (1, 4 and 6 steps): the state, dt
    and the buffer set of the step before, against cfl_m, mlw_m and the bd*
    of every field one after the other; ghost spacings are the smallest."""
    from utrip_amd import cans
    _print_case("run 1d bounds", faces, nx, margin)
    bc = [k for face in faces for k in (face if isinstance(face, list) else [face] * 5)]
    ix = nx + 2 * margin
    s = smooth_state_1d(ix, seed=ix)
    _, dx, dxm = stretched_grid(ix, seed=ix)
    dx[0], dx[-1] = 0.4 * dx.min(), 0.3 * dx.min()
    dx[1], dx[-2] = 0.5 * dx[1:-1].min(), 0.6 * dx[1:-1].min()
    f = {k: s[k].copy() for k in F1}
    n, dts, prev = 11, [], None
    for _ in range(n):
        prev = {k: v.copy() for k, v in f.items()}
        dt, merr, _i = oracle.cfl_m_1d(0.3, 1e-12, 5.0 / 3.0, s["bx"], *[f[k] for k in F1], dx)
        assert merr == 0
        oracle.mlw_m_1d(*[f[k] for k in F1], s["bx"], s["bxm"], dt, 3.0, 5.0 / 3.0, dx, dxm)
        for side in (0, 1):
            for q, k in enumerate(F1):
                kind = bc[side * 5 + q]
                if kind == PER:
                    if side == 0:
                        oracle.bnd_1d(PER, margin, margin, f[k])
                else:
                    oracle.bnd_1d(kind, side, margin, f[k], 0.0, dxm)
        dts.append(dt)
    gd = dict(dx=to_dev(dx, dev), dxm=to_dev(dxm, dev))

    def run_of(**reset):
        r = cans.Run(1, cans.ENGINE_MLW, [to_dev(s[k], dev) for k in F1], gd, 5.0 / 3.0, 0.3, qav=3.0, margin=margin,
                     bc=bc, bx1d=to_dev(s["bx"], dev), bxm1d=to_dev(s["bxm"], dev))
        r.reset(dtmin=1e-12, **reset)
        for k in (1, 4, 6):
            r.steps(k)
        return r

    run = run_of()
    cur, info = run.state()
    t = 0.0
    for d in dts:
        t = t + d
    assert info == dict(t=t, ns=n, nexec=n, merr=0, dt=dts[-1])
    other = run.a if cur is run.b else run.b
    for k, q, r in zip(F1, cur, other):
        assert_bitwise(to_host(q), f[k], k)
        assert_bitwise(to_host(r), prev[k], "step before: " + k)
    # stops on nstop and on tend, in the middle of a call and for good
    info7 = run_of(nstop=7).state()[1]
    assert info7["ns"] == info7["nexec"] == 7 and info7["dt"] == dts[6]
    end = run_of(tend=info7["t"]).state()[1]
    assert end["nexec"] == 7 and end["t"] == info7["t"]
    r = cans.Run(1, cans.ENGINE_MLW, [to_dev(s[k], dev) for k in F1], gd, 5.0 / 3.0, 0.3, qav=3.0, margin=margin,
                 bc=bc, bx1d=to_dev(s["bx"], dev), bxm1d=to_dev(s["bxm"], dev))
    r.reset(dtmin=1.0)
    r.steps(3)
    cur, info = r.state()
    assert info["merr"] == 9001 and info["nexec"] == 0 and info["ns"] == 1
    inner = slice(margin + 1, ix - margin - 1)   # (single fills also run after the stop)
    for k, q in zip(F1, cur):
        assert_bitwise(to_host(q)[inner], s[k][inner], k)


@pytest.mark.parametrize("nx,ny", [(64, 61), (255, 250), (311, 401), (700, 130)])
def test_mlw2d_resident_rows_per_wave(dev, oracle, nx, ny):
    """Resident periodic runs on grids whose strips take 1 to 5 rows per wave
    (one row at 64x61, a ragged last strip at the others): the state and dt
    after 5 steps, bit for bit."""
    from utrip_amd import cans
    _print_case("mlw2d rows per wave", nx, ny)
    pb = P.orszag_tang_box(nx, ny, margin=1)
    ref, dts = _loop_2d_oracle(oracle, pb, 5)
    g, pp = pb.grid, pb.params
    gd = {k: to_dev(v, dev) for k, v in g.items()}
    run = cans.MlwRun2D([to_dev(pb.fields[k], dev) for k in F2], gd["dx"], gd["dxm"], gd["dy"], gd["dym"],
                        pp["qav"], pp["gm"], pp["safety"], margin=1)
    run.reset(dtmin=pp["dtmin"])
    run.steps(5)
    cur, info = run.state()
    assert info["nexec"] == 5 and info["dt"] == dts[-1]
    for k, t in zip(F2, cur):
        assert_bitwise(to_host(t), ref[k], k)


def test_mlw2d_resident_stops_at_tend(dev, oracle):
    """t < tend loop test: steps after the end are no-ops."""
    from utrip_amd import cans
    pb = P.orszag_tang_2d(n=40, margin=1)
    ref, dts = _loop_2d_oracle(oracle, pb, 6)
    tend = sum_sequential(dts[:5]) * (1 + 1e-12)   # reached after step 6
    g, pp = pb.grid, pb.params
    st = [to_dev(pb.fields[k], dev) for k in F2]
    gd = {k: to_dev(v, dev) for k, v in g.items()}
    run = cans.MlwRun2D(st, gd["dx"], gd["dxm"], gd["dy"], gd["dym"], pp["qav"], pp["gm"], pp["safety"])
    run.reset(tend=tend, dtmin=pp["dtmin"])
    run.steps(11)
    cur, info = run.state()
    assert info["nexec"] == 6 and info["ns"] == 6
    for k, tt in zip(F2, cur):
        assert_bitwise(to_host(tt), ref[k], k)


def test_mlw2d_resident_dtmin_stop(dev):
    """dt < dtmin sets merr = 9001 on the device and freezes the state."""
    from utrip_amd import cans
    pb = P.orszag_tang_2d(n=40, margin=1)
    g, pp = pb.grid, pb.params
    st = [to_dev(pb.fields[k], dev) for k in F2]
    orig = [s.clone() for s in st]
    gd = {k: to_dev(v, dev) for k, v in g.items()}
    run = cans.MlwRun2D(st, gd["dx"], gd["dxm"], gd["dy"], gd["dym"], pp["qav"], pp["gm"], pp["safety"])
    run.reset(dtmin=1.0)
    run.steps(4)
    cur, info = run.state()
    assert info["merr"] == 9001 and info["nexec"] == 0 and info["ns"] == 1
    for a, b in zip(cur, orig):
        assert_bitwise(to_host(a), to_host(b))


@pytest.mark.parametrize("dim", [1, 2])
def test_cfl_merr_and_nan(dev, oracle, dim):
    """cfl_m: merr 9001 when dt < dtmin; a NaN cell is skipped by the min
    (cfl_m.f: `if (dtq < dt)` is false for NaN)."""
    from utrip_amd import cans
    if dim == 1:
        s = smooth_state_1d(200, seed=3)
        _, dx, _ = stretched_grid(200)
        s["pr"][57] = np.nan
        dto, merro, _ = oracle.cfl_m_1d(0.4, 1e-10, 1.4, s["bx"], s["ro"], s["pr"], s["vx"], s["vy"], s["by"], dx)
        t = {k: to_dev(v, dev) for k, v in s.items()}
        dtg, merrg = cans.cfl_m_1d(0.4, 1e-10, 1.4, t["bx"], t["ro"], t["pr"], t["vx"], t["vy"], t["by"],
                                   to_dev(dx, dev))
        assert dtg == dto and merrg == merro == 0
        dtg, merrg = cans.cfl_m_1d(0.4, 1.0, 1.4, t["bx"], t["ro"], t["pr"], t["vx"], t["vy"], t["by"],
                                   to_dev(dx, dev))
        assert merrg == 9001 and dtg == dto
    else:
        s = smooth_state_2d(50, 37, seed=4)
        _, dx, _ = stretched_grid(50)
        _, dy, _ = stretched_grid(37, seed=5)
        s["ro"][10, 20] = np.nan
        dto, merro, _ = oracle.cfl_m_2d(0.4, 1e-10, 1.4, s["ro"], s["pr"], s["vx"], s["vy"], s["bx"], s["by"],
                                        dx, dy)
        t = {k: to_dev(v, dev) for k, v in s.items()}
        dtg, merrg = cans.cfl_m_2d(0.4, 1e-10, 1.4, t["ro"], t["pr"], t["vx"], t["vy"], t["bx"], t["by"],
                                   to_dev(dx, dev), to_dev(dy, dev))
        assert dtg == dto and merrg == merro == 0


@pytest.mark.parametrize("kind", range(8))
def test_bnd_kinds(dev, oracle, kind):
    from utrip_amd import cans
    rng = np.random.default_rng(kind)
    for margin in (1, 2, 3):
        q = np.asfortranarray(rng.standard_normal(23))
        _, _, dxm = stretched_grid(23)
        sides = [(margin, margin)] if kind == 7 else [(0, margin), (1, margin)]
        for mbnd, mg in sides:
            r = q.copy()
            oracle.bnd_1d(kind, mbnd, mg, r, 0.37, dxm)
            t = to_dev(q, dev)
            cans.bnd_1d(kind, mbnd, mg, t, 0.37, to_dev(dxm, dev))
            assert_bitwise(to_host(t), r, f"1d kind {kind} side {mbnd} margin {margin}")
        q2 = np.asfortranarray(rng.standard_normal((13, 11)))
        for d in (0, 1):
            _, _, dm = stretched_grid(13 if d == 0 else 11)
            for mbnd, mg in sides:
                r = q2.copy(order="F")
                oracle.bnd_2d(d, kind, mbnd, mg, r, 0.37, dm)
                t = to_dev(q2, dev)
                cans.bnd_2d(d, kind, mbnd, mg, t, 0.37, to_dev(dm, dev))
                assert_bitwise(to_host(t), r, f"2d dir {d} kind {kind} side {mbnd} margin {margin}")
