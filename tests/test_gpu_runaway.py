"""An agent that runs off to infinity is no neighbor of the others, so they
move as they do without it, bit for bit: brick tiles that stage it, walked
with one or four lanes per agent, must not let it into their sums (lanes past
an agent's last candidate read some staged place)."""
import numpy as np
import pytest

import cbm._abi as A
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu

# agents below the cut (the runaway alone) are pushed to -infinity
BODY = """
struct UserLaw {
  static constexpr bool active = true, per_axis_division = false, walls = false;
  double k, c, cut;
  __device__ explicit UserLaw(const double* p) : k(p[0]), c(p[1]), cut(p[2]) {}
  __device__ bool operator()(double d, double& s) const {
    s = k * (c - d);
    return d > 0.0 && d < c;
  }
  __device__ void self(const double* x, double* f) const {
    f[0] = x[1] < cut ? -__builtin_inf() : 0.0;
  }
};
"""


def run(dims, L, pos, steps):
    n = pos.shape[1]
    m = model(dims, integrator=A.EULER, neighbors=A.CELL_LINKED, law=A.LAW_CUSTOM, dt=0.01, cell_edge=2.0)
    g = Context(m, [sim(n, [[0.0, L]] * dims, [1.0, 2.0, 0.5])])
    g.compile_model(BODY)
    for a in range(dims):
        g.upload(a, pos[a])
    g.neighbors()
    g.step(steps)
    out = np.stack([g.download(a, n) for a in range(dims)])
    b = g.bricks()
    g.close()
    assert 10 * b["overflows"] < steps * b["nbricks"]      # the row kernel has few of them
    return out


# the runaway's cell is the first of the tile at the origin; the others stay
# two cells away from it
@pytest.mark.parametrize("dims,n,L", [(2, 1801, 36.0), (2, 90001, 280.0), (3, 60001, 90.0)])
def test_runaway_touches_nobody(gpu_available, dims, n, L):
    rng = np.random.default_rng(n)
    pos = rng.uniform(4.5, L, (dims, n))
    far = np.full((dims, 1), 0.25)
    with_it = run(dims, L, np.concatenate([pos, far], axis=1), 6)
    without = run(dims, L, pos, 6)
    assert with_it[0, n] == -np.inf
    assert np.isfinite(without).all()
    assert np.array_equal(with_it[:, :n], without)
