"""Skin-list orders kept from step to step against the oracle's cell walk, bit
for bit, where agents change cells often and seldom: fast drifts across cells,
lists at capacity beside short ones, every list ordered after a build, several
simulations, one-stage (Euler) and two-stage (Heun) steps, and graph replays."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


def contexts(m, sims, pos):
    g = Context(m, sims)
    os_ = []
    for q, s in enumerate(sims):
        o = O.Oracle(m, s)
        for a in range(m.dims):
            o.set(a, pos[q][a])
            g.upload(a, pos[q][a], sim=q)
        assert o.init() == 0
        os_.append(o)
    g.neighbors()
    return g, os_


def check(g, os_, dims, what):
    for q, o in enumerate(os_):
        for a in range(dims):
            assert np.array_equal(g.download(a, o.n, sim=q), o.get(a)), (what, q, a)


# drift moves every agent by up to drift * L * dt per step: a cell in about 30
# steps, in about 3, or hardly any
@pytest.mark.parametrize("integ", [A.EULER, A.HEUN])
@pytest.mark.parametrize("dims,periodic", [(2, 0), (2, 1), (3, 0), (3, 1)])
@pytest.mark.parametrize("drift", [0.0, 0.1, 1.0])
def test_kept_orders_follow_the_cells(gpu_available, integ, dims, periodic, drift):
    rng = np.random.default_rng(dims + 10 * periodic)
    L = 60.0 if dims == 2 else 20.0
    n = 1301 if dims == 2 else 900
    box = [[-L / 3, 2 * L / 3]] * dims
    pos = [rng.uniform(-L / 3, 2 * L / 3, n) for _ in range(dims)]
    for a in range(dims):     # 70 agents whose lists overflow
        pos[a][:70] = 0.3 + rng.uniform(-0.4, 0.4, 70)
    m = model(dims, integrator=integ, neighbors=A.CELL_LINKED, law=A.LAW_REP_ADH, dt=0.01, periodic=periodic,
              cell_edge=2.4, drift=drift)
    sims = [sim(n, box, [1.0, 1.0, 0.1, 2.4]), sim(200, box, [0.7, 1.0, 0.05, 2.4])]
    g, os_ = contexts(m, sims, [pos, [p[70:270] for p in pos]])
    for k in (1, 2, 7, 20, 15):
        for o in os_:
            o.step(k)
        g.step(k)
        check(g, os_, dims, k)
    if drift != 1.0:          # builds decided on the device, orders kept across the replays
        g.step_graph(4, 3)
        for o in os_:
            o.step(12)
        check(g, os_, dims, "graph")
        g.step(9)
        for o in os_:
            o.step(9)
        check(g, os_, dims, "after")
