"""The cell sort (runs of equal cells counted once per wavefront, the scan's
two tile sizes, the slot ranks) against the oracle, bit for bit: cell tables
around one scan tile (4096 counts), around the line between the tile sizes
(524288) and past it, with agents spread out of order and with cells that
hold more agents than a wavefront, and with agents removed while they are
sorted."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [3, 4093, 4094, 4095, 8190, 524286, 524287, 1100003])
@pytest.mark.parametrize("n", [1, 63, 65, 2561])
@pytest.mark.parametrize("crowd", [0, 1])
@pytest.mark.parametrize("rule", [A.RULE_NONE, A.RULE_DEATH])
def test_sorted_cells_keep_slot_order(gpu_available, cells, n, crowd, rule):
    rng = np.random.default_rng(cells + n)
    x = rng.uniform(0.0, cells, n)
    if crowd:
        near = rng.permutation(n)[: 2 * n // 3]
        x[near] = np.floor(cells / 2) + rng.uniform(0.0, 1.0, near.size)
    m = model(1, integrator=A.EULER, neighbors=A.CELL_LINKED, law=A.LAW_REP_ADH, dt=1e-3, periodic=0, cell_edge=1.0,
              rule=rule, seed=11)
    if rule:
        m.rule_p[0] = 150.0
    m.walk = 1
    s = sim(n, [[0.0, float(cells)]], [1.0, 0.4, 0.05, 2.4], n_max=n + 5)
    o = O.Oracle(m, s)
    g = Context(m, [s])
    for c in (o.set, g.upload):
        c(A.F_X, x)
    assert o.init() == 0
    g.neighbors()
    for k in (1, 3):
        o.step(k)
        g.step(k)
        assert g.n() == o.n
        if o.n:
            assert np.array_equal(g.download(A.F_ID, o.n), o.get(A.F_ID))
            assert np.array_equal(g.download(A.F_X, o.n), o.get(A.F_X))
