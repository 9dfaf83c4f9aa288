"""Performance cases of the agent step engine: what is timed, on which inputs,
and what the outputs are in plain float64 arithmetic.

Every case is one pass of work that a program of this package has it do
through its public entry points (Community / Context): a run of steps on a
loaded community and the agents brought back, as `evolve!` does it.  The
families:

  pairs    overdamped agents under a pair law: 2-D and 3-D, periodic or open
           boxes, cell-linked grids or Verlet lists, Euler / Heun / RK4 /
           Euler-Maruyama, built-in laws and a user body
  soft     inertial soft spheres with mixed radii, masses and fates
  rods     the 2-D rod model
  colony   a dense growing and dividing colony on a nutrient field
  field    agents feeding on a field solved by FTCS or Douglas-Gunn ADI
  sweep    many independent simulations in one context (parameter sweeps)
  adjoint  the gradient of a trajectory loss for a batch of parameter sets

The state of a pass is what the pass before left, as in a program that runs
on; the adjoint leaves its community where it was.
"""
import itertools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cellbasedmodels.jl_amd"))

import cbm._abi as A  # noqa: E402
from cbm.api import (ABM, CBMIntegrators, CBMModels, CBMNeighbors, CBMRules, Community, Context,  # noqa: E402
                     bringFromPlatform_, evolve_, loadToPlatform_, step_)

# a user's interaction body: Morse-like repulsion and attraction, cut off
MORSE = """
struct UserLaw {
  static constexpr bool active = true, per_axis_division = false, walls = false;
  double D, al, r0, c;
  __device__ explicit UserLaw(const double* p) : D(p[0]), al(p[1]), r0(p[2]), c(p[3]) {}
  __device__ bool operator()(double d, double& s) const {
    const double e = exp(-al * (d - r0));
    s = 2.0 * D * al * (e * e - e);
    return d > 0.0 && d < c;
  }
};
"""

# law -> (parameters, reach)
LAWS = {
    "linear": ([1.0, 2.0], 2.0),
    "rep_adh": ([1.0, 1.0, 0.1, 2.4], 2.4),
    "aggregation": ([0.8, 1.0, 1.0, 1.0, 1.0], 1.0),
    "morse": ([0.3, 1.0, 2.0, 2.8], 2.8),
}
SOFT_P = [0.5, 1.4, 2.0, 1.0, 0.5, 3.0]
ROD_P = [60.0, 3.0, 4.0, 0.4, 0.0, 0.8, 1.5]
SIGMA = math.sqrt(2 * 0.01)


def _density(case):
    """Agents per unit of area or volume: a packing fraction near 1 in the plane
    and 0.3 in space for agents of radius 1, and one agent per unit square for
    the shorter-ranged aggregation law."""
    if case["law"] == "aggregation":
        return 1.0
    return 0.4 if case["dims"] == 2 else 0.3 / (4.0 / 3.0 * math.pi)


def listed():
    def pairs(name, **k):
        return dict({"name": name, "family": "pairs", "save_each": 0}, **k)

    return [
        # the smallest calls: a thousand agents in a periodic plane, launch-bound
        pairs("small_plane", dims=2, n=1000, law="linear", integrator="euler", neighbors="cells", periodic=True,
              steps=100),
        # the documentation's aggregation benchmark: its largest population (1,960), noise, forces of the step
        # before (its declared fx, fy), the community saved along the run
        pairs("aggregation_saves", dims=2, n=1960, law="aggregation", integrator="em", neighbors="cells",
              periodic=False, steps=100, save_each=20),
        # the headline workload: a million cells in space, Heun on Verlet lists
        pairs("tissue_verlet", dims=3, n=1048576, law="rep_adh", integrator="heun", neighbors="verlet",
              periodic=False, steps=400),
        # the same tissue as a cell-linked model
        pairs("tissue_cells", dims=3, n=1048576, law="rep_adh", integrator="heun", neighbors="cells",
              periodic=False, steps=400),
        # noisy tissue of an ordinary, odd size
        pairs("noisy_tissue", dims=3, n=262147, law="rep_adh", integrator="em", neighbors="verlet", periodic=False,
              steps=200),
        # a user's own interaction body, compiled at load time
        pairs("user_body", dims=3, n=100003, law="morse", integrator="rk4", neighbors="verlet", periodic=True,
              steps=100),
        # inertial spheres of mixed sizes on the cell grid
        {"name": "soft_spheres", "family": "soft", "dims": 3, "n": 120001, "integrator": "heun", "steps": 100},
        # bacteria-like rods
        {"name": "rods", "family": "rods", "n": 20011, "integrator": "heun", "steps": 40},
        # a dense dividing colony on its nutrient
        {"name": "colony", "family": "colony", "n": 150001, "nodes": 1024, "steps": 100},
        # agents on a field with an implicit solver
        {"name": "field_adi", "family": "field", "dims": 2, "n": 20011, "nodes": 768, "alg": "DGADI", "steps": 50},
        # a parameter sweep: simulations of uneven sizes in one context
        {"name": "sweep", "family": "sweep", "sims": 128, "n_min": 500, "n_max": 50000, "neighbors": "verlet",
         "steps": 200},
        # fitting by gradients: parameter sets around a guess
        {"name": "adjoint", "family": "adjoint", "n": 65536, "sets": 8, "steps": 100, "every": 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["pairs"] * 5 + ["soft", "rods", "colony", "field", "sweep", "adjoint"])
    if family == "pairs":
        dims = rng.choice([2, 3])
        law = rng.choice(["linear", "rep_adh", "morse"] + (["aggregation"] if dims == 2 else []))
        n = _log(rng, 700, 700000) | 1
        steps = max(20, min(200, 60_000_000 // n))
        return {"family": family, "dims": dims, "n": n, "law": law, "steps": steps,
                "integrator": rng.choice(["euler", "heun", "rk4", "em"]),
                "neighbors": rng.choice(["cells", "verlet"]),
                "periodic": rng.random() < 0.5 and law != "aggregation",
                "save_each": rng.choice([0, 0, steps // 4])}
    if family == "soft":
        return {"family": family, "dims": rng.choice([2, 3]), "n": _log(rng, 1000, 150000) | 1,
                "integrator": rng.choice(["euler", "heun", "rk4"]), "steps": rng.randrange(20, 101)}
    if family == "rods":
        return {"family": family, "n": _log(rng, 500, 40000) | 1, "integrator": rng.choice(["euler", "heun"]),
                "steps": rng.randrange(10, 41)}
    if family == "colony":
        return {"family": family, "n": _log(rng, 2000, 200000) | 1, "nodes": rng.randrange(600, 1200),
                "steps": rng.randrange(20, 101)}
    if family == "field":
        dims = rng.choice([2, 3])
        return {"family": family, "dims": dims, "n": _log(rng, 2000, 40000) | 1,
                "nodes": rng.randrange(200, 1000) if dims == 2 else rng.randrange(30, 100),
                "alg": rng.choice(["FTCS", "DGADI"]), "steps": rng.randrange(10, 51)}
    if family == "sweep":
        return {"family": family, "sims": rng.randrange(8, 129), "n_min": rng.randrange(300, 900),
                "n_max": rng.randrange(5000, 40001), "neighbors": rng.choice(["cells", "verlet"]),
                "steps": rng.randrange(50, 201)}
    return {"family": family, "n": _log(rng, 4000, 65000), "sets": rng.randrange(1, 9),
            "steps": rng.randrange(20, 101), "every": rng.choice([10, 20])}


# ------------------------------------------------------------------ inputs
def _lattice(rng, n, dims, spacing, jitter):
    """n jittered points of a square lattice and the box edge they fill."""
    m = math.ceil(n ** (1.0 / dims))
    at = rng.permutation(m ** dims)[:n]
    pos = []
    for _ in range(dims):
        pos.append((at % m + 0.5 + rng.uniform(-jitter, jitter, n)) * spacing)
        at = at // m
    return pos, m * spacing


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    f = case["family"]
    v = {"seed": int(seed) % (1 << 31)}
    n = case.get("n")
    if f == "pairs":
        v["L"] = float((n / _density(case)) ** (1.0 / case["dims"]))
        v["x"] = [rng.uniform(0.0, v["L"], n) for _ in range(case["dims"])]
        v["dt"] = 0.1 if case["law"] == "aggregation" else (0.01 if case["dims"] == 2 else 0.005)
    elif f == "soft":
        d = case["dims"]
        v["x"], v["L"] = _lattice(rng, n, d, 2.0, 0.1)
        v["v"] = [rng.normal(0.0, 0.3, n) for _ in range(d)]
        v["r"] = rng.uniform(0.8, 1.2, n)
        v["m"] = rng.uniform(0.5, 2.0, n)
        v["fate"] = rng.integers(1, 3, n).astype(np.int64)
        v["dt"] = 0.01
    elif f == "rods":
        L = v["L"] = float(math.sqrt(n * 2.0 / 0.5))
        v["x"] = [rng.uniform(1.0, L - 1.0, n) for _ in range(2)]
        v["v"] = [rng.normal(0.0, 0.3, n) for _ in range(2)]
        v["theta"] = rng.uniform(-np.pi, np.pi, n)
        v["omega"] = rng.normal(0.0, 0.5, n)
        v["l"] = rng.uniform(1.0, 3.0, n)
        v["m"] = rng.uniform(0.5, 2.0, n)
        v["dt"] = 0.002
    elif f == "colony":
        # a disc of 2 agents per unit area (radius 1 each: compressed) on a
        # field of unit spacing; slow growth against the mechanics
        L = v["L"] = float(case["nodes"])
        r = np.sqrt(n / (2.0 * math.pi)) * np.sqrt(rng.uniform(0.0, 1.0, n))
        th = rng.uniform(0.0, 2.0 * math.pi, n)
        v["x"] = [L / 2 + r * np.cos(th), L / 2 + r * np.sin(th)]
        v["vol"] = rng.uniform(1.0, 2.0, n)
        v["growth"] = 2e-4 * rng.uniform(0.9, 1.1, n)
        v["dt"] = 0.05
    elif f == "field":
        d = case["dims"]
        L = v["L"] = float((n / (0.4 if d == 2 else 0.07)) ** (1.0 / d))
        v["x"] = [rng.uniform(0.0, L, n) for _ in range(d)]
        v["dt"] = 0.01
        v["D"] = 200.0 * (L / case["nodes"]) ** 2 if case["alg"] == "DGADI" else 0.1 * (L / case["nodes"]) ** 2 / 0.01
    elif f == "sweep":
        sizes = np.random.default_rng(case["sims"])     # the same sizes for every seed
        ns = np.round(np.exp(sizes.uniform(np.log(case["n_min"]), np.log(case["n_max"]), case["sims"]))).astype(int)
        v["n"], v["Ls"], v["p"], v["xs"] = [int(q) for q in ns], [], [], []
        for q in v["n"]:
            L = float(np.sqrt(q * np.pi / rng.uniform(0.2, 0.5)))
            v["Ls"].append(L)
            v["p"].append([rng.uniform(0.5, 2.0), 1.0, rng.uniform(0.0, 0.2), 2.4])
            v["xs"].append([rng.uniform(0.0, L, q) for _ in range(2)])
        v["dt"] = 0.01
    else:   # adjoint: one community under several parameter sets, observed at four times
        L = v["L"] = float((n * 4.0 / 3.0 * math.pi / 0.3) ** (1.0 / 3.0))
        v["x"] = [rng.uniform(0.0, L, n) for _ in range(3)]
        v["theta"] = [np.array([1.0, 1.0, 0.05]) * rng.uniform(0.9, 1.1, 3) for _ in range(case["sets"])]
        v["saves"] = [max(1, case["steps"] * q // 4) for q in (1, 2, 3, 4)]
        x0 = np.stack(v["x"])
        v["target"] = np.stack([x0 + rng.normal(0.0, 0.05 * (1 + q), (3, n)) for q in range(4)])
        v["dt"] = 0.01
    return v


INTEGRATORS = {"euler": CBMIntegrators.Euler, "heun": CBMIntegrators.Heun, "rk4": CBMIntegrators.RungeKutta4,
               "em": CBMIntegrators.EM}


def _neighbors(kind, reach, dims):
    if kind == "cells":
        return CBMNeighbors.CellLinked(cellEdge=reach)
    return CBMNeighbors.VerletDisplacement(skin=reach + 0.3, nMaxNeighbors=48 if dims == 2 else 32,
                                           rebuildDisplacement=0.15)


def _law(name):
    p = LAWS[name][0]
    if name == "linear":
        return CBMModels.linearRepulsion(*p)
    if name == "rep_adh":
        return CBMModels.repulsionAdhesion(*p)
    if name == "aggregation":
        return CBMModels.aggregation(p[0], p[1], p[2], p[3], walls=True)
    return CBMModels.custom(MORSE, p)


def prepare(case, seed):
    v = _inputs(case, seed)
    f = case["family"]
    s = {"case": case}
    if f == "sweep":
        m = A.ModelDesc()
        m.dims, m.integrator, m.law, m.periodic, m.dt = 2, A.EULER, A.LAW_REP_ADH, 1, v["dt"]
        if case["neighbors"] == "cells":
            m.neighbors, m.cell_edge = A.CELL_LINKED, 2.4
        else:
            m.neighbors, m.skin, m.max_neighbors, m.rebuild_disp = A.VERLET_DISPLACEMENT, 3.0, 48, 0.3
        sims = []
        for q, n in enumerate(v["n"]):
            d = A.SimDesc()
            d.n = d.n_max = n
            d.box_hi[0] = d.box_hi[1] = v["Ls"][q]
            for k, p in enumerate(v["p"][q]):
                d.p[k] = p
            sims.append(d)
        ctx = s["ctx"] = Context(m, sims)
        for q in range(len(sims)):
            for a in range(2):
                ctx.upload(a, v["xs"][q][a], sim=q)
        ctx.neighbors()
        ctx.sync()
        s["n"] = v["n"]
        return s
    if f == "adjoint":
        m = A.ModelDesc()
        m.dims, m.integrator, m.law, m.dt = 3, A.EULER, A.LAW_REP_ADH, v["dt"]
        m.neighbors, m.skin, m.max_neighbors, m.rebuild_disp = A.VERLET_DISPLACEMENT, 3.0, 48, 0.15
        sims = []
        for th in v["theta"]:
            d = A.SimDesc()
            d.n = d.n_max = case["n"]
            for a in range(3):
                d.box_hi[a] = v["L"]
            for k, p in enumerate(list(th) + [2.4]):
                d.p[k] = p
            sims.append(d)
        ctx = s["ctx"] = Context(m, sims)
        for q in range(len(sims)):
            for a in range(3):
                ctx.upload(a, v["x"][a], sim=q)
        ctx.neighbors()
        ctx.sync()
        s["saves"] = v["saves"]
        s["target"] = [v["target"]] * len(sims)
        return s
    dims = case.get("dims", 2)
    extra, capacity = {}, 0
    if f == "pairs":
        reach = LAWS[case["law"]][1]
        abm = ABM(dims, agentODE=_law(case["law"]), agentSDE=SIGMA if case["integrator"] == "em" else 0.0,
                  neighborsAlg=_neighbors(case["neighbors"], reach, dims), periodic=case["periodic"],
                  agentAlg=INTEGRATORS[case["integrator"]](), seed=v["seed"], lagged=case["law"] == "aggregation")
    elif f == "soft":
        abm = ABM(dims, agentODE=CBMModels.softSpheres(SOFT_P[0], SOFT_P[1], [SOFT_P[2:4], SOFT_P[4:6]]),
                  neighborsAlg=CBMNeighbors.CellLinked(cellEdge=3.4), agentAlg=INTEGRATORS[case["integrator"]]())
        extra = {"r": v["r"], "m": v["m"], "cellFate": v["fate"]}
        extra.update({k: v["v"][a] for a, k in enumerate(("vx", "vy", "vz")[:dims])})
    elif f == "rods":
        abm = ABM(2, agentODE=CBMModels.rods2D(*ROD_P), neighborsAlg=CBMNeighbors.CellLinked(cellEdge=4.0),
                  agentAlg=INTEGRATORS[case["integrator"]]())
        extra = {"vx": v["v"][0], "vy": v["v"][1], "theta": v["theta"], "ω": v["omega"], "l": v["l"], "m": v["m"]}
    elif f == "colony":
        abm = ABM(2, agentODE=CBMModels.linearRepulsion(1.0, 2.0), neighborsAlg=CBMNeighbors.CellLinked(cellEdge=2.0),
                  agentAlg=CBMIntegrators.Euler(), seed=v["seed"],
                  agentRule=CBMRules.growthDivision(2e-4, 0.1, 0.5, 2.0),
                  medium={"NMedium": [case["nodes"]] * 2, "D": 1.0, "consume": 0.1, "c0": 1.0})
        extra = {"vol": v["vol"], "vbirth": 1.0, "growth": v["growth"]}
        capacity = case["n"]
    else:   # field
        reach = LAWS["linear"][1]
        abm = ABM(dims, agentODE=_law("linear"), neighborsAlg=CBMNeighbors.CellLinked(cellEdge=reach),
                  agentAlg=CBMIntegrators.Euler(),
                  medium={"NMedium": [case["nodes"]] * dims, "D": v["D"], "consume": 0.1, "c0": 1.0,
                          "mediumAlg": case["alg"]})
    com = Community(abm, N=case["n"], dt=v["dt"], simBox=[[0.0, v["L"]]] * dims,
                    **{k: v["x"][a] for a, k in enumerate(("x", "y", "z")[:dims])}, **extra)
    loadToPlatform_(com, preallocateAgents=capacity)
    com.ctx.sync()
    s["com"] = com
    return s


def run(state):
    case = state["case"]
    f = case["family"]
    if f == "sweep":
        ctx = state["ctx"]
        ctx.step(case["steps"])
        return {k: np.concatenate([ctx.download(a, n, sim=q) for q, n in enumerate(state["n"])])
                for a, k in enumerate(("x", "y"))}
    if f == "adjoint":
        # the observations go to the device with the first call of a fit
        loss, grad = state["ctx"].adjoint(case["steps"], case["every"], state["saves"], state.pop("target", None))
        return {"loss": loss, "grad": grad}
    com = state["com"]
    if case.get("save_each"):
        com.pastTimes.clear()
        evolve_(com, case["steps"], saveEach=case["save_each"])
        saved = [{k: snap[k] for k in com.params} for snap in com.pastTimes]
        return {"now": dict(com.params), "saved": saved}
    step_(com, case["steps"])
    bringFromPlatform_(com)
    out = dict(com.params)
    if f == "colony":      # the population varies: every agent's values in arrays of the capacity
        out = {k: np.concatenate([a, np.zeros(2 * case["n"] - com.N, a.dtype)]) for k, a in out.items()}
        out["N"] = com.N
    if f in ("colony", "field"):
        nodes = case["nodes"] ** case.get("dims", 2)
        med = np.empty(nodes)
        A.check(com.ctx.lib.cbm_download_medium(com.ctx.h, med.ctypes.data, nodes), com.ctx.h)
        out["medium"] = med
    return out


def work(case):
    """Per agent and stage: the state read and the new state written once, and
    the pair arithmetic of the mean number of neighbors in reach; a field adds
    its read, its write and its stencil per node and step."""
    f, steps = case["family"], case["steps"]
    d = case.get("dims", 3 if f == "adjoint" else 2)
    stages = {"heun": 2, "rk4": 4}.get(case.get("integrator"), 1)
    nodes = 0
    if f == "pairs":
        n, nvar = case["n"], d
        reach = LAWS[case["law"]][1]
        near = _density(case) * (math.pi * reach ** 2 if d == 2 else 4.0 / 3.0 * math.pi * reach ** 3)
    elif f == "soft":
        n, nvar, near = case["n"], 2 * d + 2, 12.0 if d == 3 else 6.0
    elif f == "rods":
        n, nvar, near = case["n"], 8, 6.0
    elif f == "colony":
        n, nvar, near, nodes = case["n"], 4, 25.0, case["nodes"] ** 2
    elif f == "field":
        n, nvar, near, nodes = case["n"], d, 5.0, case["nodes"] ** d
    elif f == "sweep":
        lo, hi = case["n_min"], case["n_max"]
        n, nvar, near = case["sims"] * (hi - lo) / math.log(hi / lo), 2, 2.0
    else:   # forward, recomputation and the adjoint step with its own state
        n, nvar, near, stages = case["n"] * case["sets"], 3, 4.1, 4
    return {"bytes": steps * (16.0 * nvar * stages * n + 16.0 * nodes),
            "flops": steps * (stages * n * near * (3 * d + 14.0) + 10.0 * nodes)}


# ------------------------------------------------- plain float64 reference
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_dev())


def _wrap(d, L):
    return torch.where(d > 0.5 * L, d - L, torch.where(d < -0.5 * L, d + L, d))


def _pairs_within(x, L, sim, R, periodic):
    """All ordered pairs (i, j) of one simulation closer than R; L per simulation."""
    g = torch.clamp(torch.floor(L / R), min=1).long()
    edge = (L / g)[sim]
    gs, D = g[sim], len(x)
    c = [torch.minimum(torch.clamp(torch.floor(q / edge).long(), min=0), gs - 1) for q in x]
    cells = g ** D
    off = (torch.cumsum(cells, 0) - cells)[sim]

    def lin(q):
        r = q[-1]
        for a in range(D - 2, -1, -1):
            r = q[a] + gs * r
        return off + r

    own = lin(c)
    order = torch.argsort(own)
    start = torch.searchsorted(own[order], torch.arange(int(cells.sum()) + 1, device=own.device))
    got_i, got_j = [], []
    for o in itertools.product((-1, 0, 1), repeat=D):
        q = [c[a] + o[a] for a in range(D)]
        ok = torch.ones_like(own, dtype=torch.bool)
        for a in range(D):
            if periodic:
                q[a] = q[a] % gs
            else:
                ok &= (q[a] >= 0) & (q[a] < gs)
                q[a] = torch.minimum(torch.clamp(q[a], min=0), gs - 1)
        t = lin(q)
        s = start[t]
        cnt = torch.where(ok, start[t + 1] - s, torch.zeros_like(s))
        for k in range(int(cnt.max()) if cnt.numel() else 0):
            i = torch.nonzero(cnt > k).squeeze(1)
            j = order[s[i] + k]
            d2 = torch.zeros(i.numel(), dtype=torch.float64, device=i.device)
            for a in range(D):
                dx = x[a][i] - x[a][j]
                if periodic:
                    dx = _wrap(dx, L[sim[i]])
                d2 += dx * dx
            keep = (d2 < R * R) & (i != j)
            got_i.append(i[keep])
            got_j.append(j[keep])
    return torch.cat(got_i), torch.cat(got_j)


class _Neighbors:
    """Pairs in reach of moving agents: a list with a margin, renewed before
    any agent has moved half of it; cell grids admit only pairs whose cells
    at the start of the step touch."""

    def __init__(self, L, sim, reach, periodic, edge=None):
        self.L, self.sim, self.reach, self.periodic, self.edge = L, sim, reach, periodic, edge
        self.margin = 0.25 * reach
        self.ref = None

    def at(self, x):
        if self.ref is not None:
            far = torch.zeros_like(x[0])
            for a, q in enumerate(x):
                d = q.detach() - self.ref[a]
                if self.periodic:
                    d = _wrap(d, self.L[self.sim])
                far += d * d
            if float(far.max()) >= (0.49 * self.margin) ** 2:
                self.ref = None
        if self.ref is None:
            self.ref = [q.detach().clone() for q in x]
            self.i, self.j = _pairs_within(self.ref, self.L, self.sim, self.reach + self.margin, self.periodic)
            self.mask = None
        if self.edge is not None and self.mask is None:
            self.mask = self._touching()
        return self.i, self.j, self.mask

    def step_start(self, x):
        self.start = [q.clone() for q in x]
        self.mask = None

    def _touching(self):
        L = self.L[self.sim]
        ok = torch.ones_like(self.i, dtype=torch.bool)
        for q in self.start:
            if self.periodic:
                n = torch.floor(L / self.edge)
                c = torch.minimum(torch.clamp(torch.floor(q / (L / n)), min=0), n - 1)
            else:
                n = torch.ceil(L / self.edge + 2.0)
                c = torch.floor(q / self.edge) + 1
                c = torch.where(q > L, n - 1, torch.where(q < 0, torch.zeros_like(c), c))
            d = (c[self.i] - c[self.j]).abs()
            if self.periodic:
                d = torch.minimum(d, n[self.i] - d)
            ok &= d <= 1
        return ok


def _magnitude(law, d, p):
    """s(d) and whether the pair interacts; p: one tensor or number per parameter."""
    if law == "linear":
        return p[0] * (p[1] - d), d < p[1]
    if law == "rep_adh":
        c, dc = 2.0 * p[1], p[3] * p[1]
        a4 = 4.0 * p[2] / ((dc - c) * (dc - c))
        return torch.where(d < c, p[0] * (c - d), -a4 * (d - c) * (dc - d)), d < dc
    if law == "aggregation":
        return torch.where(d < p[0], p[1] * (p[0] - d), -p[3] * (p[2] - d)), d < max(p[0], p[2])
    e = torch.exp(-p[1] * (d - p[2]))
    return 2.0 * p[0] * p[1] * (e * e - e), d < p[3]


def _pair_force(nb, x, magnitude):
    """Sum over pairs of s(d) (x_i - x_j) / d."""
    i, j, mask = nb.at(x)
    dx = [q[i] - q[j] for q in x]
    if nb.periodic:
        L = nb.L[nb.sim[i]]
        dx = [_wrap(q, L) for q in dx]
    d = torch.sqrt(sum(q * q for q in dx))
    s, on = magnitude(d, i, j)
    on = on & (d > 0)
    if mask is not None:
        on = on & mask
    s = torch.where(on, s / torch.where(d > 0, d, torch.ones_like(d)), torch.zeros_like(d))
    return [torch.zeros_like(x[0]).index_add_(0, i, s * q) for q in dx]


def _step(u, deriv, how, dt, noise=None):
    """One step of the integrator on the list of variables u."""
    k1 = deriv(u)
    if how == "euler":
        return [q + k * dt for q, k in zip(u, k1)]
    if how == "em":
        return [(q + k * dt) + z * math.sqrt(dt) for q, k, z in zip(u, k1, noise)]
    if how == "heun":
        h = [q + k * dt for q, k in zip(u, k1)]
        return [(a + (q + k * dt)) / 2 for a, q, k in zip(h, u, deriv(h))]
    k2 = deriv([q + k * dt / 2 for q, k in zip(u, k1)])
    k3 = deriv([q + k * dt / 2 for q, k in zip(u, k2)])
    k4 = deriv([q + k * dt for q, k in zip(u, k3)])
    return [q + (a + 2 * b + 2 * c + d) * dt / 6 for q, a, b, c, d in zip(u, k1, k2, k3, k4)]


def _philox(step, ids, purpose, seed, sim=0):
    """Philox4x32-10 (Salmon et al., 2011) of the counter (step, id, sim, purpose)."""
    M = 0xFFFFFFFF
    c0, c2, c3 = (torch.full_like(ids, q) for q in (int(step), int(sim), int(purpose)))
    c1 = ids & M
    k0, k1 = int(seed) & M, (int(seed) >> 32) & M
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
        a, b = c0 * 0xD2511F53, c2 * 0xCD9E8D57     # the low 64 bits hold the whole product
        c0, c1, c2, c3 = ((b >> 32) & M) ^ c1 ^ k0, b & M, ((a >> 32) & M) ^ c3 ^ k1, a & M
    return c0, c1, c2, c3


def _u53(a, b):
    return ((a >> 5).double() * 67108864.0 + (b >> 6).double()) / 9007199254740992.0


def _normals(step, ids, purpose, seed):
    r = _philox(step, ids, purpose, seed)
    rad = torch.sqrt(-2.0 * torch.log(1.0 - _u53(r[0], r[1])))
    th = 6.283185307179586 * _u53(r[2], r[3])
    return rad * torch.cos(th), rad * torch.sin(th)


def _one_box(v):
    return _t([v["L"]]), torch.zeros(len(v["x"][0]), dtype=torch.long, device=_dev())


def _named(x, more=None):
    out = dict(zip(("x", "y", "z"), (q.cpu().numpy() for q in x)))
    out["id"] = None
    out.update(more or {})
    return out


def _exact_pairs(case, v):
    law, dims, L = case["law"], case["dims"], v["L"]
    p, reach = LAWS[law]
    box, sim = _one_box(v)
    nb = _Neighbors(box, sim, reach, case["periodic"], reach if case["neighbors"] == "cells" else None)
    x = [_t(q) for q in v["x"]]
    ids = torch.arange(1, case["n"] + 1, dtype=torch.long, device=_dev())

    force = {"old": [torch.zeros_like(q) for q in x]}

    def deriv(u):
        f = _pair_force(nb, u, lambda d, i, j: _magnitude(law, d, p))
        if law == "aggregation":    # with the push of the walls; the step moves by the force of the one before
            force["new"] = [a + torch.where(q < p[0] / 2, p[1], 0.0) - torch.where(q > L - p[0] / 2, p[1], 0.0)
                            for a, q in zip(f, u)]
            return force["old"]
        return f

    def named():
        more = {}
        if law == "aggregation":
            more = {"fx": force["old"][0].cpu().numpy(), "fy": force["old"][1].cpu().numpy()}
        return _named(x, more)

    saved = []
    for k in range(case["steps"]):
        nb.step_start(x)
        z = None
        if case["integrator"] == "em":
            z = list(_normals(k, ids, 0x100, v["seed"]))
            if dims == 3:
                z.append(_normals(k, ids, 0x101, v["seed"])[0])
            z = [SIGMA * q for q in z[:dims]]
        x = _step(x, deriv, case["integrator"], v["dt"], z)
        if case["periodic"]:
            x = [torch.where(q >= L, q - L, torch.where(q < 0, q + L, q)) for q in x]
        force["old"] = force.get("new", force["old"])
        if case.get("save_each") and (k + 1) % case["save_each"] == 0:
            saved.append(named())
    return {"now": named(), "saved": saved} if case.get("save_each") else named()


def _exact_soft(case, v):
    d = case["dims"]
    b, mu, f0 = SOFT_P[0], SOFT_P[1], _t(SOFT_P[2:])
    box, sim = _one_box(v)
    nb = _Neighbors(box, sim, mu * 2.4, False, 3.4)
    r, m = _t(v["r"]), _t(v["m"])
    fate = torch.as_tensor(v["fate"], device=_dev()) - 1

    def magnitude(dist, i, j):
        rij = r[i] + r[j]
        return f0[2 * fate[i] + fate[j]] * (rij / dist - 1) * (mu * rij / dist - 1), dist < mu * rij

    def deriv(u):
        f = _pair_force(nb, u[:d], magnitude)
        return list(u[d:]) + [-b * q / m + a / m for q, a in zip(u[d:], f)]

    u = [_t(q) for q in v["x"]] + [_t(q) for q in v["v"]]
    for _ in range(case["steps"]):
        nb.step_start(u[:d])
        u = _step(u, deriv, case["integrator"], v["dt"])
    host = [q.cpu().numpy() for q in u]
    return _named(u[:d], dict({k: host[d + a] for a, k in enumerate(("vx", "vy", "vz")[:d])},
                              r=v["r"], m=v["m"], cellFate=None))


def _exact_rods(case, v):
    kn, gn, gt, mucc, _, beta, bw = ROD_P
    l, m = _t(v["l"]), _t(v["m"])
    dia = torch.ones_like(l)
    edge, L = 4.0, v["L"]
    got = {}

    def candidates(x):
        """Ordered pairs in touching cells of the grid at the step start."""
        n = int(math.ceil(L / edge + 2.0))
        c = []
        for q in x:
            k = torch.floor(q / edge) + 1
            c.append(torch.where(q > L, torch.full_like(k, n - 1), torch.where(q < 0, torch.zeros_like(k), k)).long())
        lin = c[0] + n * c[1]
        order = torch.argsort(lin)
        start = torch.searchsorted(lin[order], torch.arange(n * n + 1, device=lin.device))
        pi, pj = [], []
        for ox, oy in itertools.product((-1, 0, 1), repeat=2):
            qx, qy = c[0] + ox, c[1] + oy
            ok = (qx >= 0) & (qx < n) & (qy >= 0) & (qy < n)
            t = torch.where(ok, qx + n * qy, 0)
            s = start[t]
            cnt = torch.where(ok, start[t + 1] - s, 0)
            for k in range(int(cnt.max())):
                i = torch.nonzero(cnt > k).squeeze(1)
                j = order[s[i] + k]
                pi.append(i[i != j])
                pj.append(j[i != j])
        return torch.cat(pi), torch.cat(pj)

    def project(ax, ay, q):
        k = q["s"] * (q["x"] - ax) - q["c"] * (q["y"] - ay)
        return k * q["s"] + ax, -k * q["c"] + ay

    def clamp(q, ax, ay):
        ex, ey = q["x"] - ax, q["y"] - ay
        di = torch.clamp(torch.sqrt(ex * ex + ey * ey), min=1e-8)
        r = 0.99 * torch.minimum(di, q["l"] / 2)
        return r * ((ax - q["x"]) / di) + q["x"], r * ((ay - q["y"]) / di) + q["y"]

    def pick(on, a, b):
        return torch.where(on, a[0], b[0]), torch.where(on, a[1], b[1])

    def dist(q, a):
        return torch.sqrt((q["x"] - a[0]) ** 2 + (q["y"] - a[1]) ** 2)

    def closest(p, q):
        cx, cy = p["x"] - q["x"], p["y"] - q["y"]
        nrm = p["c"] * q["s"] - p["s"] * q["c"]
        k = (-q["s"] * cx + q["c"] * cy) / torch.where(nrm.abs() > 1e-7, nrm, torch.ones_like(nrm))
        meet = pick(nrm.abs() > 1e-7, (k * p["c"] + p["x"], k * p["s"] + p["y"]),
                    ((p["x"] + q["x"]) / 2, (p["y"] + q["y"]) / 2))
        di, dj = dist(p, meet), dist(q, meet)
        flat = clamp(p, *project(*meet, p)), clamp(q, *project(*meet, q))
        cp, cq = clamp(p, *meet), clamp(q, *meet)
        pq = project(*cq, p)          # q's end on p's line, and the reverse
        qp = project(*cp, q)
        in_i, in_j = di <= p["l"] / 2, dj <= q["l"] / 2
        beyond = dist(p, pq) > p["l"] / 2
        far_a = pick(beyond, cp, pq)
        far_b = pick(beyond & (dist(q, qp) < q["l"] / 2), qp, cq)
        a = pick(in_i & in_j, cp, pick(in_i, pq, pick(in_j, cp, far_a)))
        b = pick(in_i & in_j, cq, pick(in_i, cq, pick(in_j, qp, far_b)))
        par = nrm.abs() < 1e-6
        return pick(par, flat[0], a), pick(par, flat[1], b)

    def deriv(u):
        x, y, vx, vy, th, om = u
        i, j = got["pairs"]
        sn, cs = torch.sin(th), torch.cos(th)

        def axis(k):
            return {"x": x[k], "y": y[k], "l": l[k], "c": cs[k], "s": sn[k]}

        p, q = axis(i), axis(j)
        a, b = closest(p, q)
        rij = torch.sqrt((a[0] - b[0]) ** 2 + (a[1] - b[1]) ** 2)
        on = (rij > 0) & (rij < (dia[i] + dia[j]) / 2)
        i, j, rij = i[on], j[on], rij[on]
        ax, ay, bx, by = (w[on] for w in (*a, *b))
        de, me = dia[i] - rij, m[i] / 2
        nx, ny = (ax - bx) / rij, (ay - by) / rij
        wx, wy = vx[i] - vx[j], vy[i] - vy[j]
        vn = nx * wx + ny * wy
        fn = kn * de ** 1.5 - gn * me * de * vn
        ft = -torch.minimum(gt * me * torch.sqrt(de), mucc * fn)
        fx, fy = fn * nx + ft * (wx - vn * nx), fn * ny + ft * (wy - vn * ny)
        w = (ax - x[i]) * fy - (ay - y[i]) * fx
        tot = [torch.zeros_like(x).index_add_(0, i, q) for q in (fx, fy, w, torch.sqrt(fx * fx + fy * fy))]
        got["out"] = tot
        inertia = m * (dia + l) ** 2 / 12 + m * dia ** 2
        return [vx, vy, -beta * vx + tot[0] / m, -beta * vy + tot[1] / m, om, tot[2] / inertia - bw * om]

    u = [_t(q) for q in (*v["x"], *v["v"], v["theta"], v["omega"])]
    for _ in range(case["steps"]):
        got["pairs"] = candidates(u[:2])
        u = _step(u, deriv, case["integrator"], v["dt"])
    h = [q.cpu().numpy() for q in u]
    o = [q.cpu().numpy() for q in got["out"]]
    return _named(u[:2], {"vx": h[2], "vy": h[3], "theta": h[4], "ω": h[5], "fx": o[0], "fy": o[1], "W": o[2],
                          "pressure": o[3], "d": np.ones(case["n"]), "l": v["l"], "m": v["m"]})


def _count_nodes(x, L, nodes):
    """Agents per node of the field, x fastest."""
    t = torch.zeros_like(x[0], dtype=torch.long)
    for a in range(len(x) - 1, -1, -1):
        t = t * nodes + torch.clamp(torch.floor(x[a] / (L / nodes)).long(), 0, nodes - 1)
    return torch.bincount(t, minlength=nodes ** len(x)).double().reshape([nodes] * len(x))


def _laplacian(c, dx):
    lap = torch.zeros_like(c)
    for a in range(c.dim()):
        up = torch.cat([c.narrow(a, 1, c.shape[a] - 1), c.narrow(a, c.shape[a] - 1, 1)], a)
        dn = torch.cat([c.narrow(a, 0, 1), c.narrow(a, 0, c.shape[a] - 1)], a)
        lap += ((up - 2 * c) + dn) / (dx * dx)
    return lap


def _exact_colony(case, v):
    L, dt, nodes, seed = v["L"], v["dt"], case["nodes"], v["seed"]
    x = [_t(q) for q in v["x"]]
    vol, gr = _t(v["vol"]), _t(v["growth"])
    vb = torch.ones_like(vol)
    ids = torch.arange(1, case["n"] + 1, dtype=torch.long, device=_dev())
    c = torch.ones(nodes, nodes, dtype=torch.float64, device=_dev())
    box = _t([L])
    for k in range(case["steps"]):
        n = vol.numel()
        nb = _Neighbors(box, torch.zeros(n, dtype=torch.long, device=_dev()), 2.0, False, 2.0)
        nb.step_start(x)    # the cells date from before the divisions
        w = torch.nonzero(vol >= 2.0 * vb).squeeze(1)
        ra, rg = _philox(k, ids[w], 0x200, seed), _philox(k, ids[w], 0x300, seed)
        th = 6.283185307179586 * _u53(ra[0], ra[1])
        ax = [0.5 * torch.cos(th), 0.5 * torch.sin(th)]
        born = [x[a][w] + ax[a] for a in range(2)]
        x = [q.index_add(0, w, -s) for q, s in zip(x, ax)]
        half = vol[w] / 2
        vol = vol.index_copy(0, w, half)
        g1, g2 = (2e-4 * (1.0 + 0.1 * (2.0 * _u53(*r) - 1.0)) for r in (rg[:2], rg[2:]))
        f = _pair_force(nb, x, lambda d, i, j: _magnitude("linear", d, [1.0, 2.0]))
        x = [q + a * dt for q, a in zip(x, f)]
        vol = vol + gr * vol * dt
        cnt = _count_nodes(x, L, nodes)
        c = c + dt * (_laplacian(c, L / nodes) - 0.1 * c * cnt)
        x = [torch.cat([q, b]) for q, b in zip(x, born)]
        vol = torch.cat([vol, half])
        vb = torch.cat([vb.index_copy(0, w, half), half])
        gr = torch.cat([gr.index_copy(0, w, g1), g2])
        ids = torch.cat([ids, int(ids.max()) + 1 + torch.arange(w.numel(), device=_dev())])
    out = {k: np.concatenate([q.cpu().numpy(), np.zeros(2 * case["n"] - q.numel())])
           for k, q in (("x", x[0]), ("y", x[1]), ("vol", vol), ("vbirth", vb), ("growth", gr))}
    return dict(out, id=None, N=None, medium=c.reshape(-1).cpu().numpy())


def _exact_field(case, v):
    L, dt, nodes, d = v["L"], v["dt"], case["nodes"], case["dims"]
    box, sim = _one_box(v)
    nb = _Neighbors(box, sim, 2.0, False, 2.0)
    x = [_t(q) for q in v["x"]]
    c = torch.ones([nodes] * d, dtype=torch.float64, device=_dev())
    init, dx = c.clone(), L / nodes
    r = dt / (d * dx * dx)
    A_ = torch.zeros(nodes - 2, nodes - 2, dtype=torch.float64)
    A_.diagonal().fill_(1 + 2 * v["D"] * r)
    A_.diagonal(1).fill_(-v["D"] * r)
    A_.diagonal(-1).fill_(-v["D"] * r)
    inv = torch.linalg.inv(A_).to(_dev())
    inside = tuple(slice(1, -1) for _ in range(d))

    def sweep(s, axis):
        """Every interior line along the array axis solved, the border held."""
        s = s.transpose(axis, -1)
        b = s[inside].clone()
        rest = tuple(slice(1, -1) for _ in range(d - 1))
        b[..., 0] += v["D"] * r * s[rest + (0,)]
        b[..., -1] += v["D"] * r * s[rest + (-1,)]
        out = init.transpose(axis, -1).clone()
        out[inside] = b @ inv.T
        return out.transpose(axis, -1).contiguous()

    for _ in range(case["steps"]):
        nb.step_start(x)
        f = _pair_force(nb, x, lambda q, i, j: _magnitude("linear", q, [1.0, 2.0]))
        x = [q + a * dt for q, a in zip(x, f)]
        eat = -0.1 * c * _count_nodes(x, L, nodes)
        if case["alg"] == "FTCS":
            c = c + dt * (v["D"] * _laplacian(c, dx) + eat)
        else:
            c = c + dt * eat
            for a in range(d):     # x is the last array axis
                c = sweep(c, d - 1 - a)
    return _named(x, {"medium": c.reshape(-1).cpu().numpy()})


def _exact_sweep(case, v):
    box = _t(v["Ls"])
    sim = torch.repeat_interleave(torch.arange(len(v["n"]), device=_dev()), torch.as_tensor(v["n"], device=_dev()))
    nb = _Neighbors(box, sim, 2.4, True, 2.4 if case["neighbors"] == "cells" else None)
    x = [_t(np.concatenate([q[a] for q in v["xs"]])) for a in range(2)]
    p = _t(np.array(v["p"])).T[:, sim]
    L = box[sim]
    for _ in range(case["steps"]):
        nb.step_start(x)
        f = _pair_force(nb, x, lambda d, i, j: _magnitude("rep_adh", d, [q[i] for q in p]))
        x = [q + a * v["dt"] for q, a in zip(x, f)]
        x = [torch.where(q >= L, q - L, torch.where(q < 0, q + L, q)) for q in x]
    return {"x": x[0].cpu().numpy(), "y": x[1].cpu().numpy()}


def _exact_adjoint(case, v):
    loss, grad = [], []
    n, saves = case["n"], v["saves"]
    box, sim = _one_box(v)
    target = _t(v["target"])
    for th in v["theta"]:
        nb = _Neighbors(box, sim, 2.4 * float(th[1]), False)

        def step(x, t):
            f = _pair_force(nb, x, lambda d, i, j: _magnitude("rep_adh", d, [t[0], t[1], t[2], 2.4]))
            return [q + a * v["dt"] for q, a in zip(x, f)]

        theta = _t(th)
        path = [[_t(q) for q in v["x"]]]
        with torch.no_grad():
            for _ in range(case["steps"]):
                path.append(step(path[-1], theta))
        w = 1.0 / (len(saves) * n)
        off = {}
        for q, s in enumerate(saves):    # saves that coincide cannot occur: steps >= 20
            off[s] = [a - b for a, b in zip(path[s], target[q])]
        loss.append(w * sum(float((a * a).sum()) for d in off.values() for a in d))
        lam = [2 * w * a for a in off[case["steps"]]]
        g = torch.zeros(3, dtype=torch.float64, device=_dev())
        for t in range(case["steps"] - 1, -1, -1):
            x = [q.clone().requires_grad_(True) for q in path[t]]
            tt = theta.clone().requires_grad_(True)
            back = torch.autograd.grad(step(x, tt), x + [tt], lam)
            lam = [b.detach() for b in back[:3]]
            g += back[3]
            if t in off:
                lam = [a + 2 * w * b for a, b in zip(lam, off[t])]
        grad.append(g.cpu().numpy())
    return {"loss": np.array(loss), "grad": np.stack(grad)}


def exact(case, seed):
    v = _inputs(case, seed)
    return {"pairs": _exact_pairs, "soft": _exact_soft, "rods": _exact_rods, "colony": _exact_colony,
            "field": _exact_field, "sweep": _exact_sweep, "adjoint": _exact_adjoint}[case["family"]](case, v)
