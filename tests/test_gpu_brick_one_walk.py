"""Bricks walked once with one lane per agent, where a few agents have more in
reach than a queue holds (tight clumps in an ordinary box): those walk a
second time for the rest, and the sums and the stage-2 lists keep the order.
Bit for bit against the oracle; blocks that hold a little more or less than
whole wavefronts of agents."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


# agents per unit volume such that a brick holds about 250, 290 or 200 agents
@pytest.mark.parametrize("dims,n,L,periodic", [(2, 100001, 500.0, 0), (2, 100001, 500.0, 1), (2, 110001, 480.0, 1),
                                               (3, 70001, 99.0, 0), (3, 120001, 118.0, 1)])
@pytest.mark.parametrize("integrator", [A.EULER, A.HEUN, A.RK4])
def test_clumps_walk_twice(gpu_available, dims, n, L, periodic, integrator):
    rng = np.random.default_rng(n + dims)
    pos = rng.uniform(0.0, L, (dims, n))
    # clumps of 2 to 40 agents within a fifth of the reach
    k = 0
    for c in range(60):
        m = 2 + c * 38 // 59
        pos[:, k:k + m] = rng.uniform(3.0, L - 3.0, (dims, 1)) + rng.uniform(-0.25, 0.25, (dims, m))
        k += m
    md = model(dims, integrator=integrator, neighbors=A.CELL_LINKED, law=A.LAW_REP_ADH, dt=1e-3, periodic=periodic,
               cell_edge=2.4)
    md.walk = 1
    s = sim(n, [[0.0, L]] * dims, [1.0, 1.0, 0.1, 2.4])
    o, g = O.Oracle(md, s), Context(md, [s])
    for a in range(dims):
        o.set(a, pos[a])
        g.upload(a, pos[a])
    assert o.init() == 0
    g.neighbors()
    for q in (1, 2):
        o.step(q)
        g.step(q)
        for a in range(dims):
            assert np.array_equal(g.download(a, n), o.get(a)), (q, a)
    g.close()


# the other laws, boxes and dimensions on the same walk (one agent per cell and
# a half, so a lane per agent), a clump of 30 among them
@pytest.mark.parametrize("dims,n,L,law,p,edge,periodic", [
    (1, 100001, 150000.0, A.LAW_LINEAR, [1.0, 2.0], 2.0, 0),
    (1, 100001, 150000.0, A.LAW_LINEAR, [1.0, 2.0], 2.0, 1),
    (2, 100001, 500.0, A.LAW_LINEAR, [1.0, 2.0], 2.0, 0),
    (2, 100001, 500.0, A.LAW_LINEAR, [1.0, 2.0], 2.0, 1),
    (3, 100001, 112.0, A.LAW_LINEAR, [1.0, 2.0], 2.0, 0),
    (3, 100001, 112.0, A.LAW_LINEAR, [1.0, 2.0], 2.0, 1),
    (2, 100001, 316.0, A.LAW_AGGREGATION, [0.8, 1.0, 1.0, 1.0, 1.0], 1.0, 0),
    (2, 100001, 640.0, A.LAW_SOFT_SPHERES, [0.5, 1.4, 2.0, 1.0, 0.5, 3.0], 3.4, 0),
    (2, 100001, 640.0, A.LAW_SOFT_SPHERES, [0.5, 1.4, 2.0, 1.0, 0.5, 3.0], 3.4, 1)])
def test_every_law_walks_once(gpu_available, dims, n, L, law, p, edge, periodic):
    rng = np.random.default_rng(dims * 7 + law)
    pos = rng.uniform(0.0, L, (dims, n))
    pos[:, :30] = rng.uniform(3.0, L - 3.0, (dims, 1)) + rng.uniform(-0.2, 0.2, (dims, 30))
    soft = law == A.LAW_SOFT_SPHERES
    md = model(dims, integrator=A.HEUN if soft else A.EULER, neighbors=A.CELL_LINKED, law=law, dt=1e-4 if soft else 1e-3,
               periodic=periodic, cell_edge=edge, lagged=1 if law == A.LAW_AGGREGATION else 0)
    md.walk = 1
    s = sim(n, [[0.0, L]] * dims, p)
    o, g = O.Oracle(md, s), Context(md, [s])
    fields = [(a, pos[a]) for a in range(dims)]
    if soft:
        fields += [(A.F_RADIUS, rng.uniform(0.8, 1.2, n)), (A.F_FATE, rng.integers(1, 3, n).astype(np.int64))]
    for f, v in fields:
        o.set(f, v)
        g.upload(f, v)
    assert o.init() == 0
    g.neighbors()
    for q in (1, 2):
        o.step(q)
        g.step(q)
        for a in range(dims):
            assert np.array_equal(g.download(a, n), o.get(a)), (q, a)
    g.close()
