"""A user's law is called with the distances of neighbor candidates (and 0) and
no others, whatever the lanes of a brick do: a body may look its magnitude up
in a table that ends where the neighbor cells end."""
import numpy as np
import pytest

import cbm._abi as A
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu

BODY = """
__device__ int far_calls = 0;
struct UserLaw {
  static constexpr bool active = true, per_axis_division = false, walls = false;
  double k, c, most;
  __device__ explicit UserLaw(const double* p) : k(p[0]), c(p[1]), most(p[2]) {}
  __device__ bool operator()(double d, double& s) const {
    if (!(d <= most)) far_calls = 1;
    s = k * (c - d);
    return d > 0.0 && d < c;
  }
  __device__ void self(const double* x, double* f) const { f[0] = far_calls ? 100.0 : 0.0; }
};
"""


def run(dims, n, L, pos, most, integrator):
    m = model(dims, integrator=integrator, neighbors=A.CELL_LINKED, law=A.LAW_CUSTOM, dt=1e-3, cell_edge=2.0)
    g = Context(m, [sim(n, [[0.0, L]] * dims, [1.0, 2.0, most])])
    g.compile_model(BODY)
    for a in range(dims):
        g.upload(a, pos[a])
    g.neighbors()
    g.step(4)
    out = np.stack([g.download(a, n) for a in range(dims)])
    g.close()
    return out


# small systems (four lanes per agent) and a large one (one lane)
@pytest.mark.parametrize("dims,n,L", [(1, 301, 90.0), (2, 2049, 60.0), (2, 120001, 480.0), (3, 4099, 34.0)])
@pytest.mark.parametrize("integrator", [A.EULER, A.RK4])
def test_no_call_past_the_neighbor_cells(gpu_available, dims, n, L, integrator):
    pos = np.random.default_rng(n).uniform(0.0, L, (dims, n))
    most = 2.0 * 2.0 * np.sqrt(dims) + 0.5      # two cell edges along every axis, and what a stage moves
    noted = run(dims, n, L, pos, most, integrator)
    never = run(dims, n, L, pos, 1e300, integrator)
    assert np.array_equal(noted, never)
