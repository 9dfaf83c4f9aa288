"""The rod stage with several lanes per rod at the sizes around a round of them
(16 candidates on cells and in the full loop, 8 in lists): a lone rod, and
crowds of one round less, exactly and more, against the oracle within the
bound of the rods' own conditioning (test_gpu_rods)."""
import pytest

import cbm._abi as A
from helpers import model, sim
from test_gpu_rods import P, assert_close, both, nudged, rods

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [A.FULL, A.CELL_LINKED, A.VERLET_DISPLACEMENT])
@pytest.mark.parametrize("n", [1, 2, 8, 9, 10, 16, 17, 18, 33, 257])
def test_rods_around_a_round_of_lanes(gpu_available, nb, n):
    L = 9.0 if n < 100 else 26.0
    kw = {"cell_edge": 4.5} if nb == A.CELL_LINKED else {"skin": 5.5, "max_neighbors": 256}
    m = model(2, integrator=A.HEUN, neighbors=nb, law=A.LAW_RODS, dt=0.002, **(kw if nb != A.FULL else {}))
    s = sim(n, [[0.0, L]] * 2, P)
    ag = rods(n, L, 40 + n)
    o, g = both(m, s, ag)
    for more, steps in ((1, 1), (4, 5)):
        o.step(more)
        g.step(more)
        assert_close(o, g, nudged(m, s, ag, steps), (nb, n, steps))
