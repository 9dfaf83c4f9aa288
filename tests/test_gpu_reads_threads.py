"""Host threads that read one context at the same time each get their own
answers: counts, ids and snapshots of simulations of different sizes."""
import threading

import numpy as np
import pytest

import cbm._abi as A
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


def test_threads_read_their_own_simulation(gpu_available):
    sizes = [30, 500, 41, 900]
    m = model(2, integrator=A.EULER, neighbors=A.FULL, law=A.LAW_LINEAR, dt=0.01)
    ctx = Context(m, [sim(k, [[0.0, 20.0]] * 2, [1.0, 1.0]) for k in sizes])
    pos = [np.random.default_rng(k).uniform(0.0, 20.0, k) for k in sizes]
    for q in range(len(sizes)):
        ctx.upload(A.F_X, pos[q], sim=q)
    ctx.neighbors()
    ctx.snapshot_config([A.F_X], 1)
    ctx.snapshot_take()
    wrong = []

    def read(q):
        for _ in range(300):
            n = ctx.n(q)
            i = ctx.id_max(q)
            v, k, _ = ctx.snapshot(0, A.F_X, sim=q)
            if n != sizes[q] or i != sizes[q] or k != sizes[q] or not np.array_equal(v, pos[q]):
                wrong.append((q, n, i, k))
                return

    threads = [threading.Thread(target=read, args=(q,)) for q in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong
    ctx.close()
