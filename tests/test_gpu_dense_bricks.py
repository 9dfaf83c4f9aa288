"""Dense boxes keep their bricks: the smallest tile takes the whole LDS budget
of a block before the row-parallel kernel takes its rows.  Bit for bit against
the oracle, with no brick over its capacity."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


def lattice(dims, per_axis, edge, seed):
    """per_axis agents per cell edge along each axis, evenly, a little jittered."""
    h = edge / per_axis
    m = int(round(9 * per_axis))
    n = m ** dims
    k = np.arange(n)
    rng = np.random.default_rng(seed)
    pos = []
    for _ in range(dims):
        pos.append((k % m + 0.5 + rng.uniform(-0.2, 0.2, n)) * h)
        k = k // m
    return n, 9 * edge, pos


# agents per 3-D cell: 8, 19 (44 KiB for points, 64 for spheres, which stage
# radius and fate too), 27 (64 KiB)
@pytest.mark.parametrize("soft,per_axis", [(False, 2.0), (False, 24.0 / 9.0), (False, 3.0), (True, 2.0),
                                           (True, 24.0 / 9.0)])
def test_dense_box_stays_on_bricks(gpu_available, per_axis, soft):
    edge = 2.0
    n, L, pos = lattice(3, per_axis, edge, 4)
    law, p = (A.LAW_SOFT_SPHERES, [0.5, 1.2, 2.0, 1.0, 0.5, 3.0]) if soft else (A.LAW_LINEAR, [1.0, 0.9])
    m = model(3, integrator=A.EULER, neighbors=A.CELL_LINKED, law=law, dt=1e-3, periodic=1, cell_edge=edge)
    m.walk = 1
    s = sim(n, [[0.0, L]] * 3, p)
    o, g = O.Oracle(m, s), Context(m, [s])
    fields = [(a, pos[a]) for a in range(3)]
    if soft:
        fields += [(A.F_RADIUS, np.full(n, 0.4))]
    for f, v in fields:
        o.set(f, v)
        g.upload(f, v)
    assert o.init() == 0
    g.neighbors()
    for k in (1, 2):
        o.step(k)
        g.step(k)
        for a in range(3):
            assert np.array_equal(g.download(a, n), o.get(a)), (k, a)
    assert g.bricks()["overflows"] == 0
    g.close()
