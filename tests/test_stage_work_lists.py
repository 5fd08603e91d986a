"""The stage kernels' work lists as setup builds them (csrc/wave_stage.hip),
checked on the host: no GPU needed."""
import os
import subprocess

import numpy as np
import pytest

dyn = pytest.importorskip("dynfd3dcuda_amd")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "dynfd3dcuda_amd")


@pytest.fixture(scope="module")
def tool(tmp_path_factory):
    dyn.load_library()
    exe = str(tmp_path_factory.mktemp("work") / "stage_work_tool")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(PKG, "csrc"),
                           "-I", "/opt/rocm/include", os.path.join(ROOT, "tests", "stage_work_tool.cpp"), "-o", exe,
                           "-L", PKG, "-lcgfdm", "-L", "/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + PKG,
                           "-Wl,-rpath,/opt/rocm/lib", "-Wl,--allow-shlib-undefined"])
    return exe


def work(tool, cus=256, **params):
    out = subprocess.check_output([tool, str(cus)] + [f"{k}={v}" for k, v in params.items()], text=True)
    r = {"item": [], "box": []}
    for line in out.splitlines():
        what, *v = line.split()
        v = [int(x) for x in v]
        if what in r:
            r[what].append(v)
        else:
            r[what] = v if what in ("points", "read", "update", "column") else v[0]
    return r


def lanes(r, item):
    """Columns and rows of the block's tile."""
    if item[0] == 0:
        return 64, r["tki"]
    if r["unified"]:
        return 32, 8
    return {1: (64, r["band_tk"]), 2: (r["tjn"], 12 if r["tjn"] == 20 else 8), 3: (64, 8)}[item[0]]


@pytest.mark.parametrize("layer,opts", [(8, {"WaveUnified": 0}), (20, {"WaveUnified": 0}), (20, {"WaveBandKernel": 1}),
                                        (20, {"WaveUnified": 0, "useCerjan": 1, "DAMP_N": 27}), (20, {"WaveUnified": 1}),
                                        (20, {"NX": 400, "NY": 1000, "NZ": 504})],
                         ids=["layer_8", "layer_20", "band_64x8", "sponge_27", "unified", "default_above_200M"])
def test_lanes_beside_the_grid_read_profiles_inside_them(tool, layer, opts):
    """A lane of the free-surface tiles that lies beside the grid reads the
    y profile at the nearest point's index: tiles of one launch per kind start
    below column 0."""
    p = dict(dict(NX=44, NY=150, NZ=52, PML_N=layer), **opts)
    r = work(tool, **p)
    kind = 1 if r["unified"] else 3
    low = 0
    for it in r["item"]:
        if it[0] == kind and it[2] + it[6] > p["NZ"] - 3:
            tj = lanes(r, it)[0]
            read = np.array(r["column"][it[1] + 64:it[1] + tj + 64])
            assert read.min() >= 0 and read.max() < p["NY"]
            own = np.arange(it[1] + it[7], it[1] + it[5])
            assert np.array_equal(read[it[7]:it[5]], own)
            low = min(low, it[1])
    edge = max(layer, p.get("DAMP_N", 0) if p.get("useCerjan") else 0)
    assert low == (0 if r["unified"] else edge - 32 * ((edge + 31) // 32))


LAYOUTS = [{"WaveUnified": 0}, {"WaveUnified": 0, "WaveInteriorKernel": 3}, {"WaveUnified": 0, "WaveSurfaceKernel": 0},
           {"WaveUnified": 0, "WaveSurfaceTiles": 0}, {"WaveUnified": 0, "PmlAuxFused": 0}, {"WaveUnified": 0, "WaveBandRound": 1},
           {"WaveUnified": 1}, {"WaveUnified": 1, "WaveBandIChunk": 3}, {"WaveUnified": 2}]


@pytest.mark.parametrize("dims", [(44, 150, 52), (41, 181, 61), (45, 240, 47)], ids=["44x150x52", "41x181x61", "45x240x47"])
@pytest.mark.parametrize("free", [1, 0], ids=["surface", "no_surface"])
@pytest.mark.parametrize("layout", LAYOUTS, ids=lambda v: "-".join(f"{k}{x}" for k, x in v.items()))
def test_every_point_and_face_once(tool, layout, free, dims):
    """Every point is in one block's tile, every (point, absorbing face) pair
    is read by one block and advanced by one block or box, no interior block
    holds an absorbing point or a surface row, and the counts that the solver
    reports are those of the blocks in the list."""
    N = 12
    r = work(tool, **dict(dict(zip(("NX", "NY", "NZ"), dims), PML_N=N, FreeSurface=free), **layout))
    ni, nj, nk = dims
    faces = np.zeros(dims, int)  # absorbing faces of each point
    for ax, n in enumerate(dims):
        edge = np.zeros(n, int)
        edge[:N] += 1
        if ax < 2 or not free:
            edge[n - N:] += 1
        faces += edge.reshape([-1 if a == ax else 1 for a in range(3)])
    seen, updated = np.zeros(dims, int), np.zeros(dims, int)
    points, read, update = [0, 0, 0], [0, 0, 0, 0], [0, 0, 0, 0]
    for kind, j, k, i0, i1, jn, kn, jo, ko in r["item"]:
        w, h = lanes(r, (kind,))
        assert 0 <= jo < jn <= w and 0 <= ko < kn <= h and i0 < i1
        at = (slice(i0, i1), slice(j + jo, j + jn), slice(k + ko, k + kn))
        assert i0 >= 0 and i1 <= ni and at[1].start >= 0 and at[1].stop <= nj and at[2].start >= 0 and at[2].stop <= nk
        seen[at] += 1
        group = 0 if kind == 0 else 2 if kind == 3 else 1
        pairs = int(faces[at].sum())
        points[group] += seen[at].size
        read[group] += pairs
        if group == 0:
            assert pairs == 0 and not (free and at[2].stop > nk - 3)
        elif r["fused"] and (group == 1 or r["surf_pipe"]):
            update[group] += pairs
            updated[at] += faces[at]
    for f, j, nj_, k, nk_, i, ni_, _ in r["box"]:
        off = [0, 0, 0]  # the face's first point
        if f & 1:
            off[f // 2] = dims[f // 2] - N
        at = tuple(slice(o + x, o + x + n) for o, x, n in zip(off, (i, j, k), (ni_, nj_, nk_)))
        updated[at] += 1
        update[3] += ni_ * nj_ * nk_
    assert (seen == 1).all() and np.array_equal(updated, faces)
    assert r["points"] == points and r["read"] == read and r["update"] == update
    if layout["WaveUnified"] == 2:
        assert points[0] > 0


@pytest.mark.parametrize("opts,rows", [(dict(NX=600, NY=640, NZ=500), 4), (dict(NX=400, NY=300, NZ=200), 8),
                                       (dict(NX=44, NY=150, NZ=52, WaveUnified=2, WaveInteriorKernel=3), 4),
                                       (dict(NX=600, NY=640, NZ=500, WaveUnified=2, WaveInteriorKernel=1), 8)],
                         ids=["automatic_large", "automatic", "64x4", "64x8_ring"])
def test_kernel_of_the_interior_box(tool, opts, rows):
    """The box beside the tiles of any kind runs in 64 x 4 tiles when it holds
    many of them or when asked to, else in the ring kernel's 64 x 8 tiles."""
    r = work(tool, **opts)
    assert r["unified"] and r["points"][0] > 0
    assert {it[6] for it in r["item"] if it[0] == 0} == {rows} and r["ring"] == (rows == 8)


@pytest.mark.parametrize("free", [1, 0], ids=["surface", "no_surface"])
@pytest.mark.parametrize("dims", [(18, 40, 24), (30, 17, 24), (18, 19, 15), (40, 44, 16)], ids=lambda d: "x".join(map(str, d)))
def test_layers_wider_than_the_grid_stay_inside_it(tool, dims, free):
    """A layer of 20 points along an axis of fewer: the boxes of the
    auxiliary kernel hold the grid's points and none beside it, each
    (point, face) pair once."""
    N = 20
    r = work(tool, **dict(zip(("NX", "NY", "NZ"), dims)), PML_N=N, FreeSurface=free)
    faces, updated = np.zeros(dims, int), np.zeros(dims, int)
    for f in range(5 if free else 6):
        ax, n = f // 2, dims[f // 2]
        band = np.zeros(n, int)
        band[max(n - N, 0):] = 1 if f & 1 else band[max(n - N, 0):]
        if not f & 1:
            band[:N] = 1
        faces += band.reshape([-1 if a == ax else 1 for a in range(3)])
    for f, j, nj, k, nk, i, ni, _ in r["box"]:
        first = [i, j, k]
        first[f // 2] += dims[f // 2] - N if f & 1 else 0
        for a, n in enumerate((ni, nj, nk)):
            assert first[a] >= 0 and first[a] + n <= dims[a], (f, first)
        updated[tuple(slice(x, x + n) for x, n in zip(first, (ni, nj, nk)))] += 1
    assert bool(r["box"]) != bool(r["fused"])  # without overlap the tiles advance them all
    if r["box"]:
        assert np.array_equal(updated, faces)
    assert sum(r["read"]) == sum(r["update"]) == faces.sum()
