"""The brick walk with one and with four lanes per agent (chosen at set-up by
the agents per brick) against the oracle, bit for bit: queues of kept
candidates that fill and drain several times, bricks whose agents leave a
wavefront partly filled, and open boxes whose outer cells are empty (the tile
is sized for the density of the box, so none overflows)."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


def run_both(m, s, fields, dims, steps):
    o = O.Oracle(m, s)
    g = Context(m, [s])
    for f, v in fields:
        o.set(f, v)
        g.upload(f, v)
    assert o.init() == 0
    g.neighbors()
    for k in steps:
        o.step(k)
        g.step(k)
        for a in range(dims):
            assert np.array_equal(g.download(a, o.n), o.get(a)), (k, a)
    return g


# 17 to 27 agents in reach of each other everywhere, more than a queue of one
# (14) or four lanes (24) holds; the larger boxes are walked with one lane per
# agent, the smaller ones with four
@pytest.mark.parametrize("dims,n,L,periodic", [(2, 90001, 245.0, 0), (2, 90001, 245.0, 1), (3, 300007, 100.0, 1),
                                               (2, 2049, 37.0, 0), (3, 2049, 17.0, 0), (3, 2049, 17.0, 1),
                                               (1, 777, 140.0, 1)])
@pytest.mark.parametrize("law,p,edge", [(A.LAW_REP_ADH, [1.0, 1.0, 0.1, 2.4], 2.4),
                                        (A.LAW_AGGREGATION, [0.8, 1.0, 2.3, 0.5, 1.0], 2.4)])
def test_walk_drains_queues_in_order(gpu_available, dims, n, L, periodic, law, p, edge):
    rng = np.random.default_rng(n + dims)
    pos = [rng.uniform(0.0, L, n) for _ in range(dims)]
    m = model(dims, integrator=A.EULER, neighbors=A.CELL_LINKED, law=law, dt=1e-3, periodic=periodic, cell_edge=edge)
    m.walk = 1
    g = run_both(m, sim(n, [[0.0, L]] * dims, p), [(a, pos[a]) for a in range(dims)], dims, (1, 2))
    assert g.bricks()["overflows"] == 0


@pytest.mark.parametrize("dims,side", [(3, 20), (2, 90)])
def test_open_lattice_stays_on_bricks(gpu_available, dims, side):
    n = side ** dims
    rng = np.random.default_rng(side)
    k = np.arange(n)
    pos = []
    for _ in range(dims):
        pos.append((k % side + 0.5 + rng.uniform(-0.1, 0.1, n)) * 2.0)
        k = k // side
    fields = [(a, pos[a]) for a in range(dims)] + [(A.F_VX + a, rng.normal(0, 0.3, n)) for a in range(dims)]
    fields += [(A.F_RADIUS, rng.uniform(0.8, 1.2, n)), (A.F_MASS, rng.uniform(0.5, 2.0, n)),
               (A.F_FATE, rng.integers(1, 3, n).astype(np.int64))]
    m = model(dims, integrator=A.HEUN, neighbors=A.CELL_LINKED, law=A.LAW_SOFT_SPHERES, dt=0.01, cell_edge=3.4)
    g = run_both(m, sim(n, [[0.0, 2.0 * side]] * dims, [0.5, 1.4, 2.0, 1.0, 0.5, 3.0]), fields, dims, (1, 4))
    assert g.bricks()["overflows"] == 0
