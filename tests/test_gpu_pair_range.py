"""The short root and quotient of the pair laws against the library's, through
whole steps: in-range pairs, pairs out of range (agents 1e-40 apart, law
constants of 1e-40, coincident agents) beside ordinary ones in one wavefront,
bit for bit against the oracle."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,walk", [(A.VERLET_DISPLACEMENT, 0), (A.CELL_LINKED, 0), (A.CELL_LINKED, 1), (A.FULL, 0)])
@pytest.mark.parametrize("law,p", [(A.LAW_REP_ADH, [1.0, 1.0, 0.1, 2.4]), (A.LAW_REP_ADH, [1.0, 1.0, 0.0, 2.4]),
                                   (A.LAW_REP_ADH, [1e-40, 1.0, 1e-40, 2.4]), (A.LAW_LINEAR, [0.7, 2.3]),
                                   (A.LAW_LINEAR, [1e-40, 2.3]), (A.LAW_SOFT_SPHERES, [0.5, 1.2, 2.0, 1.0, 0.5, 3.0]),
                                   (A.LAW_SOFT_SPHERES, [0.5, 1.2, 1e-40, 1.0, 0.5, 3.0])])
def test_in_and_out_of_range_pairs(gpu_available, nb, walk, law, p):
    n, L = 500, 24.0
    rng = np.random.default_rng(3)
    pos = [rng.uniform(0.0, L, n) for _ in range(2)]
    for a in range(2):       # a tight pair beside the origin, a coincident pair, a pair on one axis
        pos[a][1] = pos[a][0] = 1e-30
        pos[a][3] = pos[a][2]
    pos[0][1] += 3e-40
    pos[1][5] = pos[1][4]
    soft = law == A.LAW_SOFT_SPHERES
    if soft:                 # overlapping spheres at 1e-40 would leave float64's range
        pos[0][1] = 2.0
    kw = {"skin": 3.2, "max_neighbors": 64} if nb == A.VERLET_DISPLACEMENT else {"cell_edge": 3.2}
    m = model(2, integrator=A.HEUN, neighbors=nb, law=law, dt=1e-3, **(kw if nb != A.FULL else {}))
    m.walk = walk
    s = sim(n, [[0.0, L]] * 2, p)
    o, g = O.Oracle(m, s), Context(m, [s])
    fields = [(a, pos[a]) for a in range(2)]
    if soft:
        fields += [(A.F_RADIUS, rng.uniform(0.8, 1.2, n)), (A.F_FATE, rng.integers(1, 3, n).astype(np.int64))]
    for f, v in fields:
        o.set(f, v)
        g.upload(f, v)
    assert o.init() == 0
    g.neighbors()
    for k in (1, 3):
        o.step(k)
        g.step(k)
        for a in range(2):
            assert np.array_equal(g.download(a, n), o.get(a)), (k, a)
