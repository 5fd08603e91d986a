"""Absorbing layers that meet or overlap (2 PML_N above an axis's length, as
the default 20 layers do on a grid 30 points wide): the general stage kernel
adds both faces of an axis to a point.  Three RK4 steps against the oracle,
with the tolerance of the other absorbing cases (1e-5 per component)."""
import numpy as np
import pytest

import cases
from test_gpu_parity import dyn, interior, make_pair, relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opts", [dict(NX=20, PML_N=11), dict(NX=30, NY=33, PML_N=20), dict(NX=19, NY=25, NZ=21, PML_N=14, FreeSurface=0),
                                  dict(NX=22, NY=20, PML_N=12, useCerjan=1), dict(NX=20, NY=70, PML_N=11, WaveInteriorKernel=0)],
                         ids=["x", "x_y", "all", "x_y_sponge", "general_interior"])
def test_overlapping_bands_match_oracle(opts):
    case = cases.volume_case(curved=True, **opts)
    s, o = make_pair(case)
    d = o.dims()
    W = cases.random_wavefield(d["nx"], d["ny"], d["nz"], seed=6)
    s.put("W", W)
    o.put("W", W)
    for it in range(3):
        s.step(it)
        o.step(it)
    x, y = interior(s.get("W"), d, 9), interior(o.get("W"), d, 9)
    for c in range(9):
        assert relerr(x[c], y[c]) < 1e-5, c
    for f in ["PMLx1", "PMLx2", "PMLy1", "PMLy2", "PMLz1"] + ([] if case["params"]["FreeSurface"] else ["PMLz2"]):
        assert np.abs(o.get(f)).max() > 0 and relerr(s.get(f), o.get(f)) < 1e-5, f


def test_layer_wider_than_an_axis():
    """20 layers along an axis of 18 points: what a face's arrays hold beside
    the grid is never advanced, and the solution stays finite."""
    case = cases.volume_case(curved=True, NX=18, NY=40, NZ=24, PML_N=20)
    s = dyn.Solver(case["params"])
    cases.apply_to_solver(case, s)
    s.setup()
    d = s.dims()
    s.put("W", cases.random_wavefield(d["nx"], d["ny"], d["nz"], seed=6))
    s.run(0, 3)
    assert s.check_field("W")["nonfinite"] == 0
    for f, beside in (("PMLx1", slice(18, 20)), ("PMLx2", slice(0, 2))):
        x = s.get(f).reshape(9, 20, d["nk"], d["nj"])
        assert np.isfinite(x).all() and np.abs(x).max() > 0 and not x[:, beside].any(), f
