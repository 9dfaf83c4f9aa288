"""A compiled law holds the stages of its context's integrator alone (noisy or
not): steps, the block tuner before them and a second compile run on those,
and a linear law restated moves as the built-in one, bit for bit."""
import numpy as np
import pytest

import cbm._abi as A
from cbm import autotune
from cbm.api import Context
from helpers import model, sim, uniform_positions

pytestmark = pytest.mark.gpu

BODY = """
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


@pytest.mark.parametrize("integrator", [A.EULER, A.HEUN, A.RK4, A.EM, A.EULER_HEUN])
@pytest.mark.parametrize("neigh", [A.FULL, A.CELL_LINKED, A.VERLET_DISPLACEMENT])
def test_each_integrator_has_its_stages(gpu_available, integrator, neigh):
    n, L = 700, 30.0
    box = [[0.0, L]] * 2
    pos = uniform_positions(n, box, 8)
    noisy = integrator in (A.EM, A.EULER_HEUN)
    out = []
    for law in (A.LAW_LINEAR, A.LAW_CUSTOM):
        m = model(2, integrator=integrator, neighbors=neigh, law=law, dt=0.01, cell_edge=2.0, skin=2.4,
                  max_neighbors=64, rebuild_disp=0.2, noise=0.1 if noisy else 0.0, seed=5)
        m.walk = 1
        g = Context(m, [sim(n, box, [1.0, 2.0])])
        if law == A.LAW_CUSTOM:
            with pytest.raises(A.CBMError):
                g.step(1)
            g.compile(BODY)
        for a in range(2):
            g.upload(a, pos[a])
        g.neighbors()
        assert autotune.tune_block(g) in (64, 128, 256)
        g.step(5)
        if law == A.LAW_CUSTOM:
            g.compile(BODY)
        g.step(5)
        out.append([g.download(a, n) for a in range(2)])
        g.close()
    for a in range(2):
        assert np.array_equal(out[0][a], out[1][a])
    assert not np.array_equal(out[0][0], pos[0])
