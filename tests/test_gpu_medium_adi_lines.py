"""DGADI sweeps staged in LDS at the sizes where they can go wrong, bit for bit
against the oracle's line-by-line sweeps: the shortest axis, lengths around the
register chunks of the two passes, line counts that leave a block partly
filled, the longest line that fits in LDS and the first that does not."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import sim, uniform_positions
from test_gpu_medium_adi import field
from test_oracle_medium_adi import adi_model

pytestmark = pytest.mark.gpu

# lines of n nodes take (3n + 32) doubles of LDS alone in a block of 64 KiB
LONGEST = 2719


@pytest.mark.parametrize("n", [(4,), (5,), (LONGEST,), (LONGEST + 1,), (4, 4), (4, 37), (21, 4), (12, 19), (36, 35),
                               (67, 130), (LONGEST, 6), (5, LONGEST + 1), (4, 5, 18), (11, 20, 28), (34, 4, 13)])
def test_adi_line_lengths(gpu_available, n):
    dims = len(n)
    box = [[0.0, float(q)] for q in n]
    m = adi_model(dims, n, 1.7, 0.1, 0.25)
    N = 20
    s = sim(N, box)
    pos = uniform_positions(N, box, 7 + sum(n))
    c0 = np.random.default_rng(sum(n)).uniform(0.5, 1.5, int(np.prod(n)))
    o = O.Oracle(m, s)
    g = Context(m, [s])
    for a, v in enumerate(pos):
        o.set(a, v)
        g.upload(a, v)
    o.set_medium(c0)
    A.check(g.lib.cbm_upload_medium(g.h, c0.ctypes.data, c0.size), g.h)
    assert o.init() == 0
    g.neighbors()
    o.step(3)
    g.step(3)
    assert np.array_equal(field(g, c0.size), o.medium(c0.size))
