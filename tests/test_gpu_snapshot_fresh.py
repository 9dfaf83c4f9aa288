"""A snapshot taken right after its configuration: the fill of the fresh
buffers must not land on it."""
import numpy as np
import pytest

import cbm._abi as A
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


def test_first_snapshot_of_a_fresh_configuration(gpu_available):
    n = 70001
    x = np.random.default_rng(0).uniform(0.0, 500.0, n)
    m = model(1, integrator=A.EULER, neighbors=A.CELL_LINKED, law=A.LAW_LINEAR, dt=0.01, cell_edge=2.0)
    ctx = Context(m, [sim(n, [[0.0, 500.0]], [1.0, 1.0])])
    ctx.upload(A.F_X, x)
    ctx.neighbors()
    for _ in range(40):
        ctx.snapshot_config([A.F_X], 3)
        ctx.snapshot_take()
        v, got, _ = ctx.snapshot(0, A.F_X)
        assert got == n and np.array_equal(v, x)
    ctx.close()
