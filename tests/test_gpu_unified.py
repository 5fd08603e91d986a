"""One launch of tiles of any kind per stage (WaveUnified 1, the default on
small grids) against one launch per kind (0): the same arithmetic at every
point, so every field is the same bit for bit, over the flag cycle and at
sizes that leave partial tiles along j, k and the plane chunks."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

dyn = pytest.importorskip("dynfd3dcuda_amd")

GRIDS = {
    "two_tiles": dict(NX=20, NY=64, NZ=20),           # whole tiles, bands meet in the middle
    "one_lane_over": dict(NX=17, NY=129, NZ=21),      # a tile of one column and one row
    "narrow": dict(NX=19, NY=17, NZ=23),              # both y bands in one tile
    "tall": dict(NX=33, NY=71, NZ=66),
}


@pytest.mark.parametrize("grid", GRIDS, ids=list(GRIDS))
@pytest.mark.parametrize("opts", [{}, {"FreeSurface": 0}, {"useCerjan": 1}, {"usePML": 0}, {"usePML": 0, "useCerjan": 1},
                                  {"MetricBF16": 1}, {"MetricBF16": 2}, {"WaveBandIChunk": 3}],
                         ids=["pml", "no_free_surface", "pml_and_sponge", "plain", "sponge", "bf16", "bf16_deviations", "chunk_3"])
def test_unified_launch_same_result(grid, opts):
    case = cases.volume_case(curved=True, PML_N=8, **GRIDS[grid], **opts)
    a = dyn.Solver(dict(case["params"], WaveUnified=1))
    b = dyn.Solver(dict(case["params"], WaveUnified=0))
    for s in (a, b):
        cases.apply_to_solver(case, s)
        s.setup()
        d = s.dims()
        s.put("W", cases.random_wavefield(d["nx"], d["ny"], d["nz"], seed=5))
        s.run(0, 8)
    names = ["W"]
    if case["params"]["usePML"]:
        names += ["PMLx1", "PMLx2", "PMLy1", "PMLy2", "PMLz1"] + ([] if case["params"]["FreeSurface"] else ["PMLz2"])
        aux = a.profile_aux()
        assert aux["stage_band"][0] == aux["stage_band"][1] and aux["pml_aux"] == (0, 0)
    for n in names:
        x = a.get(n)
        assert np.abs(x).max() > 0, n
        np.testing.assert_array_equal(x, b.get(n), err_msg=n)
    a.wave_rhs(1, -1, 1)
    b.wave_rhs(1, -1, 1)
    np.testing.assert_array_equal(a.get("hW"), b.get("hW"))


@pytest.mark.parametrize("kind", ["sw", "rs"])
def test_unified_launch_same_rupture(kind):
    case = cases.sw_case(curved=True, FaultSmooth=1) if kind == "sw" else cases.rs_case(curved=True)
    a = dyn.Solver(dict(case["params"], WaveUnified=1))
    b = dyn.Solver(dict(case["params"], WaveUnified=0))
    for s in (a, b):
        cases.apply_to_solver(case, s)
        s.setup()
        s.run(0, 10)
    assert np.abs(a.get("Vs1")).max() > 0
    for n in ("W", "FW", "Vs1", "Vs2", "Ts1", "Ts2", "Tn", "slip", "State", "slabH", "rup_sensor"):
        np.testing.assert_array_equal(a.get(n), b.get(n), err_msg=n)
