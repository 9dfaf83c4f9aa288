"""A user law on brick tiles with one and with four lanes per agent (the
rule of the built-in laws) against the oracle's restated law, bit for bit."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import model, sim, uniform_positions

pytestmark = pytest.mark.gpu

LINEAR_BODY = """
struct UserLaw {
  static constexpr bool active = true, per_axis_division = false, walls = false;
  double k, c;
  __device__ explicit UserLaw(const double* p) : k(p[0]), c(p[1]) {}
  __device__ bool operator()(double d, double& s) const {
    s = k * (c - d);
    return d > 0.0 && d < c;
  }
};
"""


# the large plane is walked with one lane per agent, the others with four
@pytest.mark.parametrize("dims,n,L", [(1, 301, 90.0), (2, 2049, 60.0), (2, 120001, 480.0), (3, 4099, 34.0)])
@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("integrator", [A.EULER, A.HEUN])
def test_user_law_walks_in_order(gpu_available, dims, n, L, periodic, integrator):
    box = [[0.0, L]] * dims
    pos = uniform_positions(n, box, n)
    base = dict(integrator=integrator, neighbors=A.CELL_LINKED, dt=0.01, periodic=periodic, cell_edge=2.8)
    s = sim(n, box, [1.0, 2.8])
    g = Context(model(dims, law=A.LAW_CUSTOM, **base), [s])
    g.compile(LINEAR_BODY)
    o = O.Oracle(model(dims, law=A.LAW_LINEAR, **base), s)
    for a in range(dims):
        g.upload(a, pos[a])
        o.set(a, pos[a])
    g.neighbors()
    o.init()
    for k in (1, 3):
        g.step(k)
        o.step(k)
        for a in range(dims):
            assert np.array_equal(g.download(a, n), o.get(a))
    g.close()
