"""put, get and check of the ADE-PML auxiliary fields where a field is larger
than the piece that one copy takes (16 MB), and at odd sizes."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

dyn = pytest.importorskip("dynfd3dcuda_amd")


@pytest.fixture(scope="module", params=[(501, 449, 45), (19, 37, 23)], ids=["pieces", "small"])
def faces(request):
    nx, ny, nz = request.param
    s = dyn.Solver(cases.volume_case(curved=False, NX=nx, NY=ny, NZ=nz, PML_N=20 if nz > 40 else 8, FreeSurface=0)["params"])
    s.setup()
    rng = np.random.default_rng(7)
    v = {}
    for n in ("PMLx1", "PMLx2", "PMLy1", "PMLy2", "PMLz1", "PMLz2"):
        v[n] = rng.standard_normal(s.field_info(n)[0], dtype=np.float32)
        s.put(n, v[n])
    yield s, v
    s.close()


def test_round_trip(faces):
    s, v = faces
    for n in v:
        assert np.array_equal(s.get(n), v[n]), n
    s.put("PMLz1", -v["PMLz1"])
    s.put("PMLy2", 2.0 * v["PMLy2"])
    assert np.array_equal(s.get("PMLz1"), -v["PMLz1"]) and np.array_equal(s.get("PMLz2"), v["PMLz2"])
    assert np.array_equal(s.get("PMLy2"), 2.0 * v["PMLy2"]) and np.array_equal(s.get("PMLy1"), v["PMLy1"])
    s.put("PMLz1", v["PMLz1"])
    s.put("PMLy2", v["PMLy2"])


def test_check_sees_its_own_face_only(faces):
    """One face's planes lie between the other's: non-finite words and the
    largest magnitude at the first, a middle and the last word of a face are
    found there and not in its neighbour."""
    s, v = faces
    for n, other in (("PMLx2", "PMLx1"), ("PMLy1", "PMLy2"), ("PMLz2", "PMLz1")):
        x = v[n].reshape(-1).copy()
        x[[0, x.size // 2, -1]] = 40.0, np.nan, -50.0
        s.put(n, x.reshape(v[n].shape))
        c = s.check_field(n)
        assert c["nonfinite"] == 1 and c["maxabs"] == 50.0, n
        x[[0, -1]] = np.inf, 30.0
        s.put(n, x.reshape(v[n].shape))
        c = s.check_field(n)
        assert c["nonfinite"] == 2 and c["maxabs"] == 30.0, n
        c = s.check_field(other)
        assert c["nonfinite"] == 0 and c["maxabs"] == np.abs(v[other]).max(), other
        s.put(n, v[n])


def test_wavefield_round_trip(faces):
    """Pieces end in the middle of rows; the check reads the device's own layout."""
    s, _ = faces
    d = s.dims()
    W = np.random.default_rng(9).standard_normal(s.field_info("W")[0], dtype=np.float32).reshape(9, d["nx"], d["nz"], d["ny"])
    W[4, 2, 5, 7] = np.nan  # a ghost plane
    s.put("W", W)
    assert np.array_equal(s.get("W").reshape(W.shape), W, equal_nan=True)
    inner = W[:, 3:-3, 3:-3, 3:-3]
    c = s.check_field("W")
    assert c == {"nonfinite": 1, "ghost_nonzero": np.count_nonzero(W) - np.count_nonzero(inner), "maxabs": np.abs(inner).max()}
    s.put("W", np.zeros_like(W))
    assert s.check_field("W") == {"nonfinite": 0, "ghost_nonzero": 0, "maxabs": 0.0}
