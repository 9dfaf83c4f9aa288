"""Pair distances whose significand is all ones (53 of them, or the leading
ones) under a power-of-two numerator: the quotients nearest to a rounding
boundary that doubles have.  Bit for bit against the oracle, whose division
is the processor's.

With d = 1 - 2^-53, c = 1 and k = 2^50 the linear law has s = 2^-3 and
s/d = 2^-3 (1 + 2^-53 + 2^-106): just above the middle of two doubles, where
a reciprocal rounded to 1 gives the lower one."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu

NB = [(A.FULL, 0), (A.VERLET_DISPLACEMENT, 0), (A.CELL_LINKED, 0), (A.CELL_LINKED, 1)]


def both(m, s, fields):
    o, g = O.Oracle(m, s), Context(m, [s])
    for f, v in fields:
        o.set(f, v)
        g.upload(f, v)
    assert o.init() == 0
    g.neighbors()
    o.step(1)
    g.step(1)
    return o, g


@pytest.mark.parametrize("nb,walk", NB)
@pytest.mark.parametrize("scale", [-3, 0, 1])
@pytest.mark.parametrize("ones", [53, 52, 40, 33, 20, 19])
def test_quotients_at_rounding_boundaries(gpu_available, nb, walk, scale, ones):
    d = (2.0 - 2.0 ** (1 - ones)) * 2.0 ** (scale - 1)
    c = 2.0 ** scale
    m = model(1, neighbors=nb, law=A.LAW_LINEAR, dt=1.0, cell_edge=4.0, skin=3.0, max_neighbors=8, rebuild_disp=0.1)
    m.walk = walk
    s = sim(2, [[-20.0, 20.0]], [2.0 ** (ones - 3), c])
    o, g = both(m, s, [(0, np.array([0.0, d]))])
    assert np.array_equal(g.download(0, 2), o.get(0))
    # s = k (c - d) = 2^(scale - 3), so the agents part
    assert o.get(0)[0] < 0.0


@pytest.mark.parametrize("nb,walk", NB)
@pytest.mark.parametrize("ones", [53, 40, 33])
def test_soft_spheres_at_rounding_boundaries(gpu_available, nb, walk, ones):
    d = 1.0 - 2.0 ** -ones
    m = model(2, neighbors=nb, law=A.LAW_SOFT_SPHERES, dt=1.0, cell_edge=4.0, skin=3.0, max_neighbors=8,
              rebuild_disp=0.1)
    m.walk = walk
    s = sim(2, [[-20.0, 20.0]] * 2, [0.5, 1.5, 2.0, 1.0, 0.5, 3.0])
    fields = [(0, np.array([0.0, d])), (1, np.zeros(2)), (A.F_RADIUS, np.array([0.5, 0.5]))]
    o, g = both(m, s, fields)
    for f in (0, 1, A.F_VX, A.F_VY):
        assert np.array_equal(g.download(f, 2), o.get(f)), f
