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
