"""The ADE-PML auxiliary fields keep the caller's layout [9][planes][k][j]
through put, get and check although the faces of an axis share one device
array (along y and z their planes alternate)."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

dyn = pytest.importorskip("dynfd3dcuda_amd")


@pytest.mark.parametrize("free", [1, 0])
def test_aux_fields_round_trip(free):
    s = dyn.Solver(cases.volume_case(curved=False, NX=23, NY=31, NZ=27, PML_N=8, FreeSurface=free)["params"])
    s.setup()
    names = ["PMLx1", "PMLx2", "PMLy1", "PMLy2", "PMLz1"] + ([] if free else ["PMLz2"])
    rng = np.random.default_rng(3)
    v = {n: rng.standard_normal(s.field_info(n)[0]).astype(np.float32) for n in names}
    for n in names:
        s.put(n, v[n])
    for n in names:  # each face on its own: no face's words reach another's
        assert np.array_equal(s.get(n), v[n]), n
        c = s.check_field(n)
        assert c["nonfinite"] == 0 and c["maxabs"] == np.abs(v[n]).max(), n
    bad = v["PMLy2"].copy()
    bad[-1] = np.nan
    s.put("PMLy2", bad)
    assert s.check_field("PMLy2")["nonfinite"] == 1 and s.check_field("PMLy1")["nonfinite"] == 0
