"""A flow's V-cycle and what it is built from on the GPU: the single-workgroup tail (k_mg_tail_fast
and its general form), the fused up-leg of a level (k_up), the lean passes of large 3D levels
(k_lean_*), bit for bit against the oracle at the sizes where their tiles and thread maps end; the
measured fields (k_measure) and the levels' coefficients (k_restrictL, k_restrictL_chain)."""
import itertools
import os

import numpy as np
import pytest

import wl_oracle as O
from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def wl():
    m = load_package()
    m.load_library()
    return m


CASES = [
    # the smallest hierarchy: the tail is level 1 on
    ((8, 8), {}), ((8, 8, 8), {}),
    # around one and two tiles of k_up (54 x 22 and 24 x 8 x 8 cells), ragged coarsening
    ((52, 20), {}), ((56, 24), {}), ((108, 44), {}), ((24, 8, 8), {}), ((26, 10, 12), {}),
    # odd extents: directions that never coarsen, half_rangek short of the last plane
    ((64, 33), {}), ((33, 64), {}), ((32, 16, 17), {}), ((17, 32, 16), {}),
    # levels with more x pairs than the tail has threads; a tail of a single level
    ((264, 136), {}), ((268, 140), {}), ((96, 64, 40), {}),
    # periodic in one or every direction, exit
    ((64, 48), dict(perdir=(2,))), ((40, 32, 24), dict(perdir=(1, 2, 3))), ((48, 32, 24), dict(perdir=(3,))),
    ((72, 40), dict(exit_bc=True)), ((48, 24, 32), dict(exit_bc=True)),
    # the lean passes on one level, on two; rows of less and more than a wave's pairs; with exit
    ((128, 40, 40), dict(lean=True)), ((144, 96, 80), dict(lean=True)), ((264, 56, 56), dict(lean=True)),
    ((96, 88, 56), dict(lean=True, exit_bc=True)),
]


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("n,kw", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "".join(v))
def test_flow_steps_bitwise(wl, n, kw, T, monkeypatch):
    if kw.get("lean"):
        monkeypatch.setenv("WL_LEAN", "2")  # at every size
    if T is np.float64 and kw.get("exit_bc"):
        pytest.skip("the exit plane's sums are Float64 on both sides, in orders of their own: Float64 shows it")
    print("case: coarse levels", n, kw, T.__name__, flush=True)
    D, R = len(n), min(n) / 5
    c = tuple(v / 2 - 0.3 for v in n)
    U = (1,) + (0,) * (D - 1)
    sim = wl.Simulation(n, U, 2 * R, ν=R / 50, body=wl.Sphere(c, R), T=T, perdir=kw.get("perdir", ()),
                        exitBC=kw.get("exit_bc", False))
    o = O.OSimulation(n, U, 2 * R, nu=R / 50, bodies=[{"kind": 1, "center": c, "radius": R}],
                      dtype=O.WL_F64 if T is np.float64 else O.WL_F32, perdir=kw.get("perdir", ()),
                      exit_bc=kw.get("exit_bc", False))
    for name in ("mu0", "mu1", "V"):
        sim.flow.set(name, o.flow.get(name))
    sim.pois.update()
    for k in range(3):
        wl.sim_step(sim, remeasure=False)
        o.step(remeasure=False)
        assert sim.pois.n == o.n, k
        for name in ("u", "p"):
            assert np.array_equal(sim.flow.get(name), o.flow.get(name)), (k, name)


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("how", ["body moves", "no body", "g and itmx 2", "profile"])
def test_lean_equals_plain(wl, how, T, monkeypatch):
    """The lean passes against the general ones (WL_LEAN=0) on the same flow: the coefficients' flags
    and 1/D follow a body that moves along and across the segments' ends, a flow without one has no
    row that reads them, and a projection cut after two V-cycles leaves the same p and u."""
    print("case: lean and plain", how, T.__name__, flush=True)
    n, got = (272, 56, 48), {}
    for mode in ("0", "2"):
        monkeypatch.setenv("WL_LEAN", mode)
        body = None if how == "no body" else wl.Sphere((60.3, 26.0, 24.0), 9)
        sim = wl.Simulation(n, (1, 0, 0), 18, ν=0.02, body=body, T=T, exitBC=how == "profile",
                            g=(lambda i, x, t: 0.1 * t) if how == "g and itmx 2" else None)
        if how == "g and itmx 2":
            sim.pois.set_solver(itmx=2)
        sim.flow.profile(how == "profile")
        got[mode] = []
        for k in range(4):
            if how == "body moves":  # its edge passes the end of the first 128 cells
                sim.body = wl.Sphere((100.0 + 7.5 * k, 12.0 + 4 * k, 40.0 - 6 * k), 9)
            wl.sim_step(sim, remeasure=how == "body moves")
            got[mode] += [sim.flow.get("u"), sim.flow.get("p"), list(sim.pois.n)]
    for a, b in zip(got["0"], got["2"]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("n", [(72, 40), (64, 33), (32, 24, 16), (128, 40, 40)], ids=lambda v: "x".join(map(str, v)))
def test_launches_ahead_of_the_read(wl, n, T, monkeypatch):
    """The launches issued before the host has read Σr² (guessed from the last solve's V-cycles) against
    a run that issues none (a profiled flow), while the tolerance and the limit make the guess wrong
    both ways: the same V-cycles, u and p."""
    print("case: launches ahead", n, T.__name__, flush=True)
    monkeypatch.setenv("WL_LEAN", "2" if n[0] == 128 else "1")
    D, R, got = len(n), min(n) / 5, []
    for profiled in (True, False):
        sim = wl.Simulation(n, (1,) + (0,) * (D - 1), 2 * R, ν=R / 50, body=wl.Sphere(tuple(v / 2 for v in n), R), T=T)
        sim.flow.profile(profiled)
        out = []
        for kw in ({}, dict(tol=1e-7), dict(tol=1e-7), dict(itmx=1), dict(tol=1e-7, itmx=2), dict(tol=1e-1), {}):
            sim.pois.set_solver(**kw)
            wl.sim_step(sim, remeasure=False)
            out += [sim.flow.get("u"), sim.flow.get("p")]
        got.append((list(sim.pois.n), out))
    assert got[0][0] == got[1][0] and len(set(got[0][0])) > 2
    for a, b in zip(got[0][1], got[1][1]):
        assert np.array_equal(a, b)


def bc_fill(a, perdir, value=0):
    """BC!(a, value) (src/core.jl:200-219) of a vector field without exit, in the reference's loops."""
    D = a.ndim - 1
    for i in range(D):
        v = a[..., i]
        for j in range(D):
            def at(k):
                return tuple(k if q == j else slice(None) for q in range(D))
            N = a.shape[j]
            if j + 1 in perdir:
                v[at(0)], v[at(N - 1)] = v[at(N - 2)], v[at(1)]
            elif i == j:
                v[at(0)] = v[at(1)] = v[at(N - 1)] = value
            else:
                v[at(0)], v[at(N - 1)] = v[at(1)], v[at(N - 2)]


def restrict_l(fine, perdir):
    """restrictL (src/MultiLevelPoisson.jl:20-26,42-48) with its BC!, sums in the reference's order."""
    D = fine.ndim - 1
    cm = [N % 2 == 0 and N > 4 for N in fine.shape[:D]]
    Nc = [1 + N // 2 if c else N for N, c in zip(fine.shape[:D], cm)]
    out = np.zeros(Nc + [D], dtype=fine.dtype)
    inner = tuple(slice(1, -1) for _ in range(D))
    for i in range(D):
        f = fine[inner + (i,)]
        steps = [(0,) if j == i or not cm[j] else (0, 1) for j in range(D)]
        parts = [p[::-1] for p in itertools.product(*steps[::-1])]  # z slowest, x fastest
        s = np.zeros([N - 2 for N in Nc], dtype=fine.dtype)
        for p in parts:
            s = s + f[tuple(slice(p[j], None, 2 if cm[j] else None) for j in range(D))]
        out[inner + (i,)] = s / fine.dtype.type(2) if cm[i] else s
    bc_fill(out, perdir)
    return out


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("n,perdir", [((64, 48), ()), ((136, 72), (2,)), ((64, 33), ()), ((40, 32, 24), ()),
                                      ((48, 40, 32), (1, 3)), ((32, 16, 17), ())],
                         ids=lambda v: "x".join(map(str, v)) or "-")
def test_measured_fields_and_levels(wl, n, perdir, T):
    """measure! in one pass: its ghosts are BC!'s bit for bit, μ₁ and V 0 there, and the step uses the
    same row flags as after an upload of the same fields; update!: every level's L is restrictL's with
    its BC!.  The body reaches the walls."""
    print("case: measured fields and levels", n, perdir, T.__name__, flush=True)
    D, R = len(n), min(n) / 4
    U = (1,) + (0,) * (D - 1)
    body = wl.Sphere((3.3,) + tuple(v - 4.4 for v in n[1:]), R)
    a, b = (wl.Simulation(n, U, 2 * R, ν=0.05, body=body, T=T, perdir=perdir) for _ in range(2))
    mu0, mu1, V = (a.flow.get(k) for k in ("mu0", "mu1", "V"))
    ref = mu0.copy()
    bc_fill(ref, perdir)
    assert np.array_equal(mu0, ref)
    ghost = np.ones(mu0.shape[:-1], bool)
    ghost[tuple(slice(1, -1) for _ in range(D))] = False
    assert not mu1[ghost].any() and not V.any()
    for name in ("mu0", "mu1", "V"):
        b.flow.set(name, b.flow.get(name))
    b.pois.update()
    for s in (a, b):
        wl.sim_step(s, remeasure=False)
    for name in ("u", "p"):
        assert np.array_equal(a.flow.get(name), b.flow.get(name)), name
    ml = wl.MultiLevelPoisson(np.zeros(mu0.shape[:-1], T), mu0, np.zeros(mu0.shape[:-1], T), perdir=perdir)
    L, l = mu0, 0
    while l + 1 < len(ml.levels):
        L, l = restrict_l(L, perdir), l + 1
        assert np.array_equal(ml.get("L", l), L), l


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("how", ["upload", "measure"])
def test_lean_follows_mu0_without_update(wl, how, T, monkeypatch):
    """μ₀ changed without update!: the lean passes' 1/D is that of the L they read, as in the passes
    that form it, with the row flags and without (WL_LROWS=0)."""
    print("case: lean after a change of mu0 alone", how, T.__name__, flush=True)
    n, got = (144, 56, 48), []
    moved = wl.Sphere((60.5, 26.1, 23.9), 9.1)  # (the coarse levels keep the other body's)
    mu0 = wl.Simulation(n, (1, 0, 0), 18, ν=0.02, body=moved, T=T).flow.get("mu0")
    for lean, rows in (("0", "1"), ("0", "0"), ("2", "1"), ("2", "0")):
        monkeypatch.setenv("WL_LEAN", lean)
        monkeypatch.setenv("WL_LROWS", rows)
        sim = wl.Simulation(n, (1, 0, 0), 18, ν=0.02, body=wl.Sphere((60.3, 26.0, 24.0), 9), T=T)
        wl.sim_step(sim, remeasure=False)
        if how == "upload":
            sim.flow.set("mu0", mu0)
        else:
            wl.measure_flow(sim.flow, moved)
        for _ in range(2):
            wl.sim_step(sim, remeasure=False)
        got.append([sim.flow.get("u"), sim.flow.get("p"), list(sim.pois.n)])
    for g in got[1:]:
        for a, b in zip(got[0], g):
            assert np.array_equal(a, b)


def launches(flow, run):
    """The profiled (name, level, bytes) of what `run` launches."""
    flow.profile(True)
    run()
    got = {(k["name"], k["level"], k["bytes_per_launch"]) for k in flow.profile_read()}
    flow.profile(False)
    return got


@pytest.mark.parametrize("mode", ["plain", "mixed"])
@pytest.mark.parametrize("lean", ["0", "2"])
def test_autotune_times_the_flows_own_launches(wl, lean, mode, monkeypatch):
    """The tile autotuner of a 3D flow times launches that its steps make, and with the lean passes on
    the finest level none of that level, which take no target."""
    print("case: autotune", lean, mode, flush=True)
    monkeypatch.setenv("WL_LEAN", lean)
    sim = wl.Simulation((272, 56, 48), (1, 0, 0), 18, ν=0.02, body=wl.Sphere((60.3, 26.0, 24.0), 9))
    sim.pois.set_solver(mode=wl.WL_SOLVER_MIXED if mode == "mixed" else wl.WL_SOLVER_PLAIN)
    for _ in range(2):
        wl.sim_step(sim, remeasure=False)
    u, p = sim.flow.u, sim.flow.p
    timed = launches(sim.flow, lambda: sim.flow.autotune(1))
    assert np.array_equal(sim.flow.u, u) and np.array_equal(sim.flow.p, p)
    stepped = launches(sim.flow, lambda: wl.sim_step(sim, remeasure=False))
    assert timed and timed <= stepped, timed - stepped
    assert (min(k[1] for k in timed) == 0) == (lean == "0" or mode == "mixed")


@pytest.mark.parametrize("n,perdir", [((72, 40), ()), ((64, 33), ()), ((40, 32, 24), ()), ((136, 72), (2,)),
                                      ((48, 32, 24), (3,)), ("batch", ())],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else v)
def test_up_cells_is_read_per_handle(wl, n, perdir, monkeypatch):
    """WL_UP_CELLS=0 (every level by its separate passes) beside the default, one process: the same
    V-cycles, u and p; k_up runs in the second alone."""
    print("case: WL_UP_CELLS", n, perdir, flush=True)
    shapes = [(72, 40), (128, 64)] if n == "batch" else [n]
    got = []
    for cells in ("0", None, "0"):
        if cells is None:
            monkeypatch.delenv("WL_UP_CELLS", raising=False)
        else:
            monkeypatch.setenv("WL_UP_CELLS", cells)
        sims = [wl.Simulation(s, (1,) + (0,) * (len(s) - 1), min(s) / 3, ν=0.02, perdir=perdir,
                              body=wl.Sphere(tuple(v / 2 - 0.3 for v in s), min(s) / 6)) for s in shapes]
        keys = set()
        if n == "batch":
            b = wl.Batch(sims)
            for _ in range(3):
                b.step()
        else:
            for _ in range(3):
                keys |= {k[0] for k in launches(sims[0].flow, lambda: wl.sim_step(sims[0], remeasure=False))}
            assert bool(keys & {"up", "up_fin"}) == (cells is None), keys
        got.append([v for s in sims for v in (s.flow.get("u"), s.flow.get("p"), list(s.pois.n))])
    for a, b, c in zip(*got):
        assert np.array_equal(a, b) and np.array_equal(a, c)


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("n,perdir", [((8, 8), ()), ((32, 32), ()), ((64, 64), ()), ((72, 56), ()), ((34, 68), ()),
                                      ((64, 33), ()), ((64, 48), (1,)), ((8, 8, 8), ()), ((40, 24, 20), ()),
                                      ((32, 16, 17), ()), ((32, 24, 40), (2, 3))],
                         ids=lambda v: "x".join(map(str, v)) or "-")
def test_standalone_multigrid_levels(wl, n, perdir, T):
    """A MultiLevelPoisson of its own keeps every level's state (k_mg_tail_lds, whose passes take a cell
    or a pair per thread): x and r of each level after two V-cycles, bit for bit.  The source is
    antisymmetric, so no order of its sum removes a mean."""
    print("case: standalone multigrid", n, perdir, T.__name__, flush=True)
    rng, Ng, D = np.random.default_rng(11), tuple(v + 2 for v in n), len(n)
    inner = (slice(1, -1),) * D
    L = np.ones(Ng + (D,), T, order="F")
    L[inner] = rng.uniform(0.1, 1.0, size=n + (D,))
    bc_fill(L, perdir)
    z = np.zeros(Ng, T, order="F")
    v = rng.normal(size=n).astype(T)
    z[inner] = v - np.flip(v)
    x = np.zeros(Ng, T, order="F")
    g, o = wl.MultiLevelPoisson(x, L, z, perdir=perdir), O.OPois(L, perdir=perdir, dtype=O.WL_F64 if T is np.float64 else O.WL_F32)
    o.set("z", z)
    wl.solver(g, tol=0, itmx=2)
    o.solve(tol=0, itmx=2)
    assert g.n == o.n and g.nlevels == o.nlevels
    for l in range(g.nlevels):
        for name in ("x", "r"):
            assert np.array_equal(g.get(name, l), o.get(name, l)), (l, name)


@pytest.mark.parametrize("n,levels", [((128, 40, 40), 1), ((144, 96, 80), 2), ((264, 56, 56), 2), ((96, 88, 56), 1),
                                      ((272, 56, 48), 2), ((144, 56, 48), 1), ((256, 208, 208), 1), ((96, 64, 64), 0)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_lean_levels(wl, n, levels, monkeypatch):
    """Which levels the lean passes run, by the bytes of their restriction (a fifth to a quarter of the
    plain one's): at WL_LEAN=2 those of the tests above, without it those of at least 40 and 16 MB."""
    print("case: lean levels", n, levels, flush=True)
    got = []
    for mode in ("0", None if n[0] == 256 or n == (96, 64, 64) else "2"):
        monkeypatch.delenv("WL_LEAN", raising=False) if mode is None else monkeypatch.setenv("WL_LEAN", mode)
        sim = wl.Simulation(n, (1, 0, 0), 8, ν=0.02, body=wl.Sphere(tuple(v / 2 for v in n), 8))
        got.append({k[1]: k[2] for k in launches(sim.flow, lambda: wl.sim_step(sim, remeasure=False))
                    if k[0] == "inc_restrict"})
    assert sorted(got[0]) == sorted(got[1])
    assert [l for l in sorted(got[0]) if 3 * got[1][l] < got[0][l]] == list(range(levels))


@pytest.mark.parametrize("n", [(72, 40), (48, 24, 32), (48, 56, 40), (40, 48, 44)], ids=lambda v: "x".join(map(str, v)))
def test_exit_f64(wl, n):
    """exitBC! in Float64, in one workgroup and (over 2048 exit cells) gathered, against the oracle.  The
    exit plane's two sums over its `cnt` cells are Float64 on both sides in orders of their own: at most
    cnt·2⁻⁵³ apart each, relative to U = 1.  A step's projections spread that over u with at most a
    factor of the box's length, and over p with that once more over Δt."""
    print("case: exit in Float64", n, flush=True)
    D, R, steps = len(n), min(n) / 5, 3
    c, U = tuple(v / 2 - 0.3 for v in n), (1,) + (0,) * (D - 1)
    sim = wl.Simulation(n, U, 2 * R, ν=R / 50, body=wl.Sphere(c, R), T=np.float64, exitBC=True)
    o = O.OSimulation(n, U, 2 * R, nu=R / 50, bodies=[{"kind": 1, "center": c, "radius": R}], dtype=O.WL_F64,
                      exit_bc=True)
    for name in ("mu0", "mu1", "V"):
        sim.flow.set(name, o.flow.get(name))
    sim.pois.update()
    tol = 2 * steps * int(np.prod(n[1:])) * 2.0 ** -53 * n[0]
    for k in range(steps):
        wl.sim_step(sim, remeasure=False)
        o.step(remeasure=False)
        assert sim.pois.n == o.n, k
        eu, ep = (float(np.abs(sim.flow.get(f) - o.flow.get(f)).max()) for f in ("u", "p"))
        print(f"  step {k}: u {eu:.2e} of {tol:.2e}, p {ep:.2e}", flush=True)
        assert eu <= tol and ep <= tol * n[0] / min(sim.flow.Δt)


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("n,wide", [((64, 64, 56), 1), ((88, 88, 88), 2), ((104, 104, 96), 3)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "-")
def test_up_levels(wl, n, wide, T, monkeypatch):
    """k_up takes a 3D level whose field has at most 400 KB: level 1 of 64x64x56 (34 680 cells) in both
    types, of 88x88x88 (97 336) in Float32, of 104x104x96 (145 800) in neither; the same u and p as with
    none."""
    print("case: levels of k_up", n, T.__name__, flush=True)
    got, first = [], 1 if wide == 1 or (wide == 2 and T is np.float32) else 2
    for cells in (None, "0"):
        monkeypatch.delenv("WL_UP_CELLS", raising=False) if cells is None else monkeypatch.setenv("WL_UP_CELLS", cells)
        sim = wl.Simulation(n, (1, 0, 0), 12, ν=0.02, body=wl.Sphere(tuple(v / 2 for v in n), 12), T=T)
        keys = launches(sim.flow, lambda: wl.sim_step(sim, remeasure=False))
        assert min((k[1] for k in keys if k[0] == "up"), default=None) == (first if cells is None else None)
        wl.sim_step(sim, remeasure=False)
        got.append([sim.flow.get("u"), sim.flow.get("p"), list(sim.pois.n)])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
