"""The pipelined stage kernels, which advance the auxiliary fields of all faces
of a point in its tile and compute the surface rows beside other rows, against
the general kernels with the auxiliary kernel of its own: the same arithmetic
at every point, so every field is the same bit for bit.  The sizes leave
wavefronts without a point, tiles of one row or column, and surface rows at
every place of a tile."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

dyn = pytest.importorskip("dynfd3dcuda_amd")

GENERAL = dict(WaveUnified=0, WaveInteriorKernel=0, WaveBandKernel=0, WaveSurfaceKernel=0, PmlAuxFused=0)


@pytest.mark.parametrize("nz", [16, 17, 18, 21, 23])
@pytest.mark.parametrize("opts", [{"WaveUnified": 1}, {"WaveUnified": 0}, {"WaveUnified": 0, "WaveBandKernel": 2},
                                  {"WaveUnified": 1, "useCerjan": 1}, {"WaveUnified": 1, "FreeSurface": 0}],
                         ids=["unified", "per_kind", "per_kind_64x4", "unified_sponge", "unified_no_surface"])
def test_same_as_general_kernels(opts, nz):
    case = cases.volume_case(curved=True, NX=19, NY=33 if nz % 2 else 70, NZ=nz, PML_N=8,
                             **{k: v for k, v in opts.items() if not k.startswith("Wave")})
    a = dyn.Solver(dict(case["params"], **opts))
    b = dyn.Solver(dict(case["params"], **GENERAL))
    for s in (a, b):
        cases.apply_to_solver(case, s)
        s.setup()
        d = s.dims()
        s.put("W", cases.random_wavefield(d["nx"], d["ny"], d["nz"], seed=11))
        s.run(0, 8)
    assert a.profile_aux()["pml_aux"] == (0, 0) and b.profile_aux()["pml_aux"][1] > 0
    for n in ["W", "PMLx1", "PMLx2", "PMLy1", "PMLy2", "PMLz1"] + ([] if case["params"]["FreeSurface"] else ["PMLz2"]):
        x = a.get(n)
        assert np.abs(x).max() > 0, n
        np.testing.assert_array_equal(x, b.get(n), err_msg=n)


@pytest.mark.parametrize("dims", [(20, 112, 24), (41, 113, 27), (37, 241, 45), (19, 96, 40)])
@pytest.mark.parametrize("opts", [{}, {"useCerjan": 1}, {"FreeSurface": 0}, {"MetricBF16": 1}, {"usePML": 0}],
                         ids=["pml", "sponge", "no_surface", "bf16", "plain"])
def test_interior_box_beside_unified_tiles(opts, dims):
    """The interior kernel on the whole 64 x 8 tiles of the interior, one
    launch of 32 x 8 tiles around them: boxes of one tile, of several, and
    none at all (the last size)."""
    case = cases.volume_case(curved=True, NX=dims[0], NY=dims[1], NZ=dims[2], PML_N=8, **opts)
    a = dyn.Solver(dict(case["params"], WaveUnified=2))
    b = dyn.Solver(dict(case["params"], **GENERAL))
    for s in (a, b):
        cases.apply_to_solver(case, s)
        s.setup()
        d = s.dims()
        s.put("W", cases.random_wavefield(d["nx"], d["ny"], d["nz"], seed=12))
        s.run(0, 8)
    a.profile(True)
    a.run(8, 1)
    b.run(8, 1)
    edge = case["params"]["PML_N"] if opts.get("usePML", 1) else 0
    lo = (edge + 31) // 32 * 32
    assert (a.profile_report()["stage_interior"][1] > 0) == ((dims[1] - edge - lo) // 64 >= 1)
    for n in ["W"] + (["PMLx1", "PMLx2", "PMLy1", "PMLy2", "PMLz1"] if case["params"]["usePML"] else []):
        assert np.abs(a.get(n)).max() > 0, n
        np.testing.assert_array_equal(a.get(n), b.get(n), err_msg=n)
