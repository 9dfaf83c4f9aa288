"""The adjoint's list builds on brick tiles, with the rows left in place,
against the oracle's dual numbers: builds in the middle of the pass, lists
longer than a lane's queue, bricks too crowded for LDS (their rows take the
row kernel), several simulations and one, two and three axes."""
import numpy as np
import pytest

import cbm._abi as A
import oracle as O
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,n,ball", [(1, 401, 0), (2, 1201, 0), (3, 1501, 0), (2, 1201, 60), (3, 2300, 1400)])
def test_builds_in_place_match_dual_numbers(gpu_available, dims, n, ball):
    rng = np.random.default_rng(n + ball)
    L = float((n - ball) / 0.3) ** (1.0 / dims) * 1.5
    x = rng.uniform(0.0, L, (dims, n))
    if ball:
        x[:, rng.permutation(n)[:ball]] = L / 2 + rng.uniform(-0.9, 0.9, (dims, ball))
    m = model(dims, integrator=A.EULER, neighbors=A.VERLET_DISPLACEMENT, law=A.LAW_REP_ADH, dt=0.002,
              skin=2.8, max_neighbors=max(64, ball + 64), rebuild_disp=0.02)
    thetas = [np.array([1.0, 1.0, 0.05]), np.array([1.2, 0.95, 0.06])]
    s = [sim(n, [[0.0, L]] * dims, list(t) + [2.4]) for t in thetas]
    g = Context(m, s)
    steps, saves = 6, np.array([3, 6])
    tgt = np.stack([x + 0.01 * rng.normal(0.0, 1.0, x.shape) for _ in saves])
    for q in range(2):
        for a in range(dims):
            g.upload(a, x[a], sim=q)
    g.neighbors()
    before, over = g.rebuilds(), g.bricks()["overflows"]
    loss, grad = g.adjoint(steps, 2, saves, [tgt] * 2)
    assert g.rebuilds() > before
    assert (g.bricks()["overflows"] > over) == (ball > 1000)
    for q, t in enumerate(thetas):
        o = O.Oracle(m, s[q])
        for a in range(dims):
            o.set(a, x[a])
        o.init()
        rl, rg = o.traj_grad_dual(t, steps, saves, tgt.ravel())
        assert abs(loss[q] - rl) <= 1e-12 * abs(rl)
        assert np.allclose(grad[q], rg, rtol=1e-9, atol=1e-14 * np.abs(rg).max())
    g.close()
