"""The interior box beside the launch of tiles of any kind (WaveUnified 2, the
default from 4 to 200 million points) in both of the kernels that run it
(WaveInteriorKernel 1 and 3), with every metric form and with a rupture whose
fault planes cross the box: the same arithmetic at every point as one launch
per kind, so every field is the same bit for bit."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

dyn = pytest.importorskip("dynfd3dcuda_amd")


def pair(case, kernel, other, prepare=lambda s: None, steps=8):
    a = dyn.Solver(dict(case["params"], WaveUnified=2, WaveInteriorKernel=kernel))
    b = dyn.Solver(dict(case["params"], **other))
    for s in (a, b):
        cases.apply_to_solver(case, s)
        s.setup()
        prepare(s)
        s.run(0, steps)
    a.profile(True)
    for s in (a, b):
        s.run(steps, 1)
    report = a.profile_report()
    assert report["stage_interior"][1] > 0 and report["stage_surface"][1] == 0
    return a, b


@pytest.mark.parametrize("kernel", [1, 3], ids=["ring_64x8", "64x4"])
@pytest.mark.parametrize("metric", [0, 1, 2])
@pytest.mark.parametrize("dims", [(20, 112, 24), (37, 241, 45)], ids=["one_tile", "several"])
def test_box_same_as_general_kernels(dims, metric, kernel):
    case = cases.volume_case(curved=True, NX=dims[0], NY=dims[1], NZ=dims[2], PML_N=8, MetricBF16=metric)

    def prepare(s):
        d = s.dims()
        s.put("W", cases.random_wavefield(d["nx"], d["ny"], d["nz"], seed=13))

    a, b = pair(case, kernel, dict(WaveUnified=0, WaveInteriorKernel=0, WaveBandKernel=0, WaveSurfaceKernel=0, PmlAuxFused=0), prepare)
    for n in ("W", "PMLx1", "PMLx2", "PMLy1", "PMLy2", "PMLz1"):
        assert np.abs(a.get(n)).max() > 0, n
        np.testing.assert_array_equal(a.get(n), b.get(n), err_msg=n)


@pytest.mark.parametrize("kernel", [1, 3], ids=["ring_64x8", "64x4"])
@pytest.mark.parametrize("metric", [0, 2])
@pytest.mark.parametrize("kind", ["sw", "rs"])
def test_box_same_rupture(kind, metric, kernel):
    """The six planes of split-node stencils and the fault plane lie in the
    box and in the tiles around it."""
    make = cases.sw_case if kind == "sw" else cases.rs_case
    case = make(curved=True, NY=140, MetricBF16=metric, **({"FaultSmooth": 1} if kind == "sw" else {}))
    a, b = pair(case, kernel, dict(WaveUnified=0), steps=10)
    assert np.abs(a.get("Vs1")).max() > 0
    for n in ("W", "FW", "Vs1", "Vs2", "Ts1", "Ts2", "Tn", "slip", "State", "slabH", "rup_sensor", "PMLx1", "PMLx2", "PMLy1",
              "PMLy2", "PMLz1"):
        np.testing.assert_array_equal(a.get(n), b.get(n), err_msg=n)


@pytest.mark.parametrize("opts,used", [
    ({}, 1), ({"WaveUnified": 2}, 1), ({"WaveUnified": 2, "NY": 112}, 2), ({"WaveUnified": 2, "NY": 112, "WaveInteriorKernel": 3}, 2),
    ({"WaveUnified": 0}, 0), ({"WaveUnified": 1, "WaveInteriorKernel": 3}, 0), ({"WaveUnified": 1, "StageStreams": 1}, 0),
    ({"WaveUnified": 2, "WaveTopIChunk": 4}, 0), ({"WaveUnified": 1, "PML_N": 11}, 0), ({"WaveUnified": 1, "WaveBandIChunk": 5}, 1)],
    ids=["default", "no_box", "box", "box_64x4", "off", "other_kernel", "streams", "surface_chunk", "bands_overlap", "chunk"])
def test_setup_reports_the_layout_in_use(opts, used):
    """A WaveUnified that cannot be honoured reads back as what runs."""
    case = cases.volume_case(curved=False, **dict(dict(NX=20, NY=40, NZ=24, PML_N=8), **opts))
    s = dyn.Solver(case["params"])
    assert s.get_param("WaveUnified") == opts.get("WaveUnified", -1)
    s.setup()
    assert s.get_param("WaveUnified") == used
    s.run(0, 1)
    s.close()
