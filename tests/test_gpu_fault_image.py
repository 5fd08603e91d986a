"""The odd image of the split nodes' tractions above the free surface in the
friction trial (trial_slipweakening.cu:215-260): the top three rows each
mirror another set of words, so each row of the trial's traction is compared
with the oracle's, from split nodes whose dip tractions carry signal there
(in a rupture they vanish towards the surface and hide the mirrored words).
Tolerance: the trial is a sum of about twenty FP32 terms of the row's size,
so 2e-5 of the row's largest value; a mirrored word left out is 4e-2 of it."""
import numpy as np
import pytest

import cases
from oracle.binding import Oracle

pytestmark = pytest.mark.gpu

dyn = pytest.importorskip("dynfd3dcuda_amd")


@pytest.mark.parametrize("it", [0, 1])  # with irk, both directions of the operator along dip
@pytest.mark.parametrize("irk", [0, 1])
def test_trial_rows_under_the_surface(it, irk):
    case = cases.sw_case(curved=True)
    case["stress"]["Ty"] = -60e6 * np.ones_like(case["stress"]["Ty"])  # no node slides: the trial traction stays
    case["stress"]["mu_s"] = np.full_like(case["stress"]["Ty"], 10.0)
    s, o = dyn.Solver(case["params"]), Oracle(case["params"])
    cases.apply_to_solver(case, s)
    cases.apply_to_oracle(case, o)
    s.setup()
    o.setup()
    d = s.dims()
    fw = np.zeros((9, 2, d["nz"], d["ny"]), np.float32)
    rng = np.random.default_rng(7)
    fw[3:, :, 3:-3, 3:-3] = 1e5 * rng.standard_normal((6, 2, d["nk"], d["nj"]))
    s.put("FW", fw)
    o.put("FW", fw)
    f = s.stage_flags_lib(it, irk)
    s.fault_trial(it, irk)
    o.fault_trial(it, irk, *f)
    assert not np.any(s.get("flag_rup")), "locked"
    shape = (7, d["nz"], d["ny"])
    for n in ("T11", "T12", "T13"):
        a, b = s.get(n).reshape(shape)[3].astype(np.float64), o.get(n).reshape(shape)[3]
        for row in range(d["nk"] - 6, d["nk"]):
            e = np.abs(a[row + 3] - b[row + 3]).max() / np.abs(b[row + 3]).max()
            assert e < 2e-5, (n, d["nk"] - row, e)
