"""The words of an output record, gathered on the device: every field and
slice of the files equals what cgfdm_get_field returns for the same state, at
sizes that are no multiple of anything and with slices at the grid's edges."""
import numpy as np
import pytest
from scipy.io import netcdf_file

import cases

pytestmark = pytest.mark.gpu

dyn = pytest.importorskip("dynfd3dcuda_amd")


def last(path, name):
    with netcdf_file(str(path), "r", mmap=False) as f:
        v = f.variables[name]
        return np.array(v[-1] if v.isrec else v[:])


@pytest.mark.parametrize("kind", ["sw", "tp", "wave"])
@pytest.mark.parametrize("slices", [(0, 0, 0), (10**6, 10**6, 10**6), (13, 31, 17)], ids=["low", "high", "inside"])
def test_record_equals_fields(tmp_path, kind, slices):
    if kind == "wave":
        case = cases.volume_case(NX=23, NY=41, NZ=29, PML_N=8)
    elif kind == "sw":
        case = cases.sw_case(NX=29, NY=83, NZ=47)
    else:
        case = cases.rs_case(NX=29, NY=83, NZ=47, Friction_type=3, TP_n=5, RS_L=0.4)
        case["stress"]["TP_hy"] = np.full_like(case["stress"]["L"], 2.0 ** -11)
    case["params"].update(OUT=str(tmp_path), EXPORT_TIME_SKIP=2, EXPORT_WAVE_SLICE_X=slices[0],
                          EXPORT_WAVE_SLICE_Y=slices[1], EXPORT_WAVE_SLICE_Z=slices[2])
    s = dyn.Solver(case["params"])
    cases.apply_to_solver(case, s)
    s.setup()
    d = s.dims()
    s.put("W", cases.random_wavefield(d["nx"], d["ny"], d["nz"], seed=2) * 0.01)
    s.run(0, 4, write_outputs=True)
    s.write_outputs(4)  # the third record holds the present state
    W = s.get("W").reshape(9, d["nx"], d["nz"], d["ny"])[:3, 3:-3, 3:-3, 3:-3]
    i, j, k = (min(max(v, 0), n - 1) for v, n in zip(slices, (d["ni"], d["nj"], d["nk"])))
    for plane, a in (("xy", W[:, :, k, :]), ("xz", W[:, :, :, j]), ("yz", W[:, i])):
        for c, n in enumerate(("Vx", "Vy", "Vz")):
            assert np.abs(a[c]).max() > 0
            np.testing.assert_array_equal(last(tmp_path / f"wave_{plane}_mpi000000.nc", n), a[c], err_msg=plane + n)
    if kind == "wave":
        return
    f = tmp_path / "fault_mpi000000.nc"
    for n, field in {"Vs1": "Vs1", "Vs2": "Vs2", "tn": "Tn", "ts1": "Ts1", "ts2": "Ts2", "Us0": "slip", "State": "State",
                     "rup_index_y": "rup_index_y", "rup_index_z": "rup_index_z", "rup_sensor": "rup_sensor",
                     "init_t0": "init_t0", "TP_T": "TP_T", "TP_P": "TP_P"}.items():
        got = last(f, n).ravel()
        if n.startswith("TP_") and kind != "tp":
            assert not got.any()
            continue
        want = s.get(field)[:got.size]  # of the TP levels the one on the fault
        np.testing.assert_array_equal(got, want.astype(got.dtype.newbyteorder("=")), err_msg=n)
