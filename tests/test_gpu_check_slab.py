"""check_field of the fault slab reads the slab's seven planes and no more."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

dyn = pytest.importorskip("dynfd3dcuda_amd")


def test_check_of_the_fault_slab():
    case = cases.sw_case()
    s = dyn.Solver(case["params"])
    cases.apply_to_solver(case, s)
    s.setup()
    d = s.dims()
    x = np.zeros((7, 9, d["nz"], d["ny"]), np.float32)
    x[:, :, 3:-3, 3:-3] = np.random.default_rng(5).standard_normal((7, 9, d["nz"] - 6, d["ny"] - 6), dtype=np.float32)
    x[0, 0, 3, 3], x[6, 8, -4, -4] = 30.0, -40.0  # the first and the last word of the interior
    s.put("slabH", x.reshape(s.get("slabH").shape))
    assert s.check_field("slabH") == {"nonfinite": 0, "ghost_nonzero": 0, "maxabs": 40.0}
    x[6, 8, -4, -4], x[0, 0, 3, 3] = np.nan, np.inf
    x[3, 4, 0, 0], x[6, 8, -1, -1] = 50.0, 60.0  # ghost layers along y and z
    s.put("slabH", x.reshape(s.get("slabH").shape))
    c = s.check_field("slabH")
    y = np.abs(x[:, :, 3:-3, 3:-3])
    assert c == {"nonfinite": 2, "ghost_nonzero": 2, "maxabs": y[np.isfinite(y)].max()}
    c = s.check_field("W")
    assert c["nonfinite"] == 0 and c["ghost_nonzero"] == 0
    s.close()
