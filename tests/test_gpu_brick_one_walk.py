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
