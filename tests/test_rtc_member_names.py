"""A user's interaction body may give its members any name that the library
does not document (active, per_axis_division, walls, self, de, pair, ode,
sums): the kernels take the built-in laws' short cuts by type.  Bodies with
members of the built-in laws' own names compile, and their functions of
those names, deleted here, are not called.  Runs in a child process, as
test_rtc_bodies.py does, with either hipRTC."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

HEAD = """
struct UserLaw {
  static constexpr bool active = true, per_axis_division = false, walls = false;
  double k, c;
  __device__ explicit UserLaw(const double* p) : k(p[0]), c(p[1]) {}
  __device__ bool operator()(double d, double& s) const { s = k * (c - d); return d > 0.0 && d < c; }
"""
MEMBERS = {
    "near_value": "  double near = 0.5;\n",
    "near_function": "  __device__ double near(double d) const = delete;\n",
    "near_and_plain": "  __device__ bool plain() const = delete;\n"
                      "  __device__ bool near(double d, double& s) const = delete;\n",
    "reach_value": "  double reach = 2.0;\n",
    "reach_function": "  __device__ double reach() const = delete;\n",
    "span_and_mu": "  double span = 1.0, mu = 1.0, f0 = 2.0;\n",
}

CHILD = """
import sys
sys.path[:0] = {paths!r}
if {torch!r}:
    import torch
import ctypes as C
import cbm._abi as A
from helpers import model
bad = 0
for label, body in {bodies!r}.items():
    for dims, neigh in ((2, A.CELL_LINKED), (3, A.CELL_LINKED), (3, A.VERLET_DISPLACEMENT), (2, A.FULL)):
        m = model(dims, neighbors=neigh, law=A.LAW_CUSTOM, cell_edge=2.0, skin=2.3, max_neighbors=32)
        log = C.create_string_buffer(1 << 16)
        print(label, dims, neigh, flush=True)
        if A.lib().cbm_compile_check(C.byref(m), body.encode(), None, None, None, log, len(log)) != A.OK:
            bad += 1
            print(log.value.decode(errors="replace")[:600], flush=True)
sys.exit(1 if bad else 0)
"""


@pytest.mark.parametrize("torch_first", [False, True], ids=["rocm", "torch-bundled"])
def test_members_with_the_library_laws_names(torch_first):
    root = os.path.dirname(HERE)
    code = CHILD.format(paths=[HERE, root, os.path.join(root, "cellbasedmodels.jl_amd")], torch=torch_first,
                        bodies={k: HEAD + v + "};\n" for k, v in MEMBERS.items()})
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout[-4000:]}\n{r.stderr[-2000:]}"
