"""Reads of agent values around the size up to which a context keeps host
memory for them (131072 values): every value comes back at its slot from rows
the cell sort has moved, from each simulation of a batch, whole and in part,
now and out of a snapshot, and errors of the status words still surface."""
import numpy as np
import pytest

import cbm._abi as A
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 131071, 131072, 131073, 200001])
@pytest.mark.parametrize("other", [3, 140000])
def test_reads_return_every_slot(gpu_available, n, other):
    rng = np.random.default_rng(n)
    sizes = (n, other)
    m = model(2, integrator=A.EULER, neighbors=A.CELL_LINKED, law=A.LAW_LINEAR, dt=0.01, cell_edge=2.0)
    edge = [4.0 + 2.0 * float(np.sqrt(k)) for k in sizes]
    ctx = Context(m, [sim(k, [[0.0, L]] * 2, [1.0, 1.0], n_max=k + 2) for k, L in zip(sizes, edge)])
    pos = [[rng.uniform(0.0, L, k) for _ in range(2)] for k, L in zip(sizes, edge)]
    for q in range(2):
        for a in range(2):
            ctx.upload(a, pos[q][a], sim=q)
    ctx.neighbors()
    ctx.snapshot_config([A.F_X, A.F_Y, A.F_ID], 1)
    ctx.snapshot_take()
    for q, k in enumerate(sizes):
        assert ctx.n(q) == k and ctx.id_max(q) == k
        for a in range(2):
            assert np.array_equal(ctx.download(a, k, sim=q), pos[q][a])
            v, got, t = ctx.snapshot(0, a, sim=q)
            assert got == k and t == 0.0 and np.array_equal(v, pos[q][a])
        assert np.array_equal(ctx.download(A.F_X, (k + 1) // 2, sim=q), pos[q][0][: (k + 1) // 2])
        assert np.array_equal(ctx.download(A.F_ID, k, sim=q), np.arange(1, k + 1))
        assert ctx.download(A.F_X, 0, sim=q).size == 0
    ctx.close()


@pytest.mark.parametrize("n", [500, 131073])
def test_a_full_list_surfaces_on_a_read(gpu_available, n):
    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 1.0, 2 * n).reshape(2, n) * np.sqrt(n) / 8
    m = model(2, integrator=A.EULER, neighbors=A.VERLET_DISPLACEMENT, law=A.LAW_LINEAR, dt=0.01, skin=2.5,
              max_neighbors=4, rebuild_disp=0.2)
    ctx = Context(m, [sim(n, [[0.0, float(np.sqrt(n) / 8)]] * 2, [1.0, 1.0])])
    for a in range(2):
        ctx.upload(a, x[a])
    ctx.neighbors()
    with pytest.raises(Exception, match="overflow"):
        ctx.download(A.F_X, n)
    with pytest.raises(Exception, match="overflow"):
        ctx.sync()
    ctx.close()
