"""The message of a body that does not compile begins with its first errors
and stays short, however long the compiler's log is."""
import pytest

import cbm._abi as A
from cbm.api import Context
from helpers import model, sim

pytestmark = pytest.mark.gpu

BODY = """
struct UserLaw {
  static constexpr bool active = true, per_axis_division = false, walls = false;
  double k;
  __device__ explicit UserLaw(const double* p) : k(p[0]) {}
  __device__ bool operator()(double d, double& s) const {
    %s
    return d > 0.0;
  }
};
"""


def test_first_errors_are_kept(gpu_available):
    lines = "\n    ".join(f"s = no_such_name_{k}(d) + {'another_missing_name' * 5}_{k};" for k in range(60))
    g = Context(model(2, neighbors=A.FULL, law=A.LAW_CUSTOM, dt=0.01), [sim(4, [[0.0, 8.0]] * 2, [1.0])])
    with pytest.raises(A.CBMError) as e:
        g.compile(BODY % lines)
    text = str(e.value)
    assert "no_such_name_0" in text and "no_such_name_1" in text
    assert len(text) < 3500
    assert "changed in memory" not in text
    g.close()
