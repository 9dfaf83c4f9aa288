"""Every complete user body that a test file or the performance cases hold as a
module-level string goes through hipRTC on the CPU, in the one-lane and the
four-lane form of the brick kernels (cbm_compile_check builds both).  Found by
reading the files, so a new test's bodies are in it without a list.  Runs in a
child process, with either hipRTC, as test_rtc_bodies.py does."""
import ast
import glob
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

CHILD = """
import sys
sys.path[:0] = {paths!r}
if {torch!r}:
    import torch
import cbm._abi as A
from rtc_bodies_check import check
ok = [check(A, label, body) for label, body in {bodies!r}]
sys.exit(0 if all(ok) and ok else 1)
"""


def bodies():
    """(file:line, text) of every string constant that is a whole body of its own."""
    out = []
    files = sorted(glob.glob(os.path.join(HERE, "*.py"))) + [os.path.join(ROOT, "perf", "cases.py")]
    for path in files:
        with open(path) as f:
            tree = ast.parse(f.read())
        for node in tree.body:
            text = node.value.value if isinstance(node, ast.Assign) and isinstance(node.value, ast.Constant) else None
            t = text.strip() if isinstance(text, str) else ""
            whole = t.startswith("struct User") and t.endswith("};") and t.count("{") == t.count("}")
            if whole and "%s" not in t:
                out.append((f"{os.path.basename(path)}:{node.lineno}", text))
    return out


def test_the_search_finds_the_bodies():
    found = {label.split(":")[0] for label, _ in bodies()}
    assert {"cases.py", "test_gpu_user_lanes.py", "test_gpu_custom_law.py", "test_gpu_runaway.py"} <= found


@pytest.mark.parametrize("torch_first", [False, True], ids=["rocm", "torch-bundled"])
def test_every_body_compiles(torch_first):
    code = CHILD.format(paths=[HERE, ROOT, os.path.join(ROOT, "cellbasedmodels.jl_amd")], torch=torch_first,
                        bodies=bodies())
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout[-4000:]}\n{r.stderr[-2000:]}"
