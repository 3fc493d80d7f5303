"""The coarse levels of a flow's V-cycle on the GPU: the single-workgroup tail (k_mg_tail_fast and
its general form) and the fused up-leg of a level (k_up), bit for bit against the oracle at the
sizes where their tiles and thread maps end."""
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
]


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("n,kw", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "".join(v))
def test_flow_steps_bitwise(wl, n, kw, T):
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
