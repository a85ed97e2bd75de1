"""Host side of a context (no GPU): tests/context_host_check.cpp, compiled with
g++ and linked against libpiks3d.so, creates one under each combination of the
settings that choose the sweep.  Exactly one sweep is on, with the storage
order and records it reads: tiles where they are asked for and serve the
context (whatever PIKS_SWEEP_FLOW says), else rows of cells unless a setting
asks for the hyperplane launches.  A context whose padded slots do not fit the memory there
is takes the hyperplane launches' layout if that fits."""
import os
import shutil
import subprocess

import pytest

import piks3d_amd
from piks3d_amd import images

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(REPO, "piks3d_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
SHAPE = (15, 14, 17)  # nz, ny, nx


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no g++ or HIP headers")
    d = tmp_path_factory.mktemp("context_host")
    out = str(d / "context_host_check")
    lib = os.path.dirname(piks3d_amd.LIB_PATH)
    subprocess.run([gxx, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
                    "-I" + CSRC, "-I" + os.path.join(REPO, "include"), "-o", out,
                    os.path.join(HERE, "context_host_check.cpp"), "-L" + lib, "-lpiks3d", "-Wl,-rpath," + lib,
                    "-L" + os.path.join(ROCM, "lib"), "-lamdhip64", "-Wl,-rpath," + os.path.join(ROCM, "lib")],
                   check=True)
    raw = str(d / "image.raw")
    images.write_raw(raw, images.box_blocks(SHAPE, 10, 2, 4, 3))
    return out, raw


def _host(checker, env, nc, precision, sweep, *extra):
    exe, raw = checker
    e = {k: v for k, v in os.environ.items() if not k.startswith("PIKS_")}
    e.update(env)
    nz, ny, nx = SHAPE
    r = subprocess.run([exe, raw, str(nx), str(ny), str(nz), "2", "2", str(nc), str(precision), str(sweep), *extra],
                       capture_output=True, text=True, timeout=120, env=e)
    assert r.returncode == 0, (env, nc, precision, sweep, r.returncode, r.stderr)
    words = r.stdout.split()
    return {k: int(v) for k, v in zip(words[::2], words[1::2])}


@pytest.mark.parametrize("nc", [3, 4, 6])            # 27, 64, 216 velocities per octant
@pytest.mark.parametrize("precision", [0, 1])        # FP64, refined
@pytest.mark.parametrize("tiles_env", [None, "0", "1"])
@pytest.mark.parametrize("flow", [None, "0", "1"])
def test_settings_choose_one_sweep(checker, flow, tiles_env, precision, nc):
    env = {k: v for k, v in (("PIKS_SWEEP_FLOW", flow), ("PIKS_SWEEP_TILES", tiles_env)) if v is not None}
    for sweep in (0, 1, 2):
        got = _host(checker, env, nc, precision, sweep)
        assert got["rc"] == 0
        tiles = (sweep == 2 or sweep == 0 and tiles_env == "1") and precision == 0 and nc ** 3 <= 64
        rows = not tiles and (flow == "1" or flow is None and sweep == 0 and tiles_env is None)
        assert (got["tiles"], got["rows"]) == (int(tiles), int(rows)), (env, sweep)
        # the storage order and the records of that sweep
        assert got["raster"] == int(rows)
        assert (got["row_words"] > 0) == rows
        assert (got["tile_words"] > 0) == tiles
        assert (got["hyper_words"] > 0) == (not rows)
        assert rows or got["vs"] == got["nc8"]


def test_generic_kernel_setting_takes_no_tiles(checker):
    # PIKS_SWEEP_GENERIC forces the generic kernel of the hyperplane launches
    got = _host(checker, {"PIKS_SWEEP_GENERIC": "1", "PIKS_SWEEP_TILES": "1"}, 4, 0, 0)
    assert (got["rc"], got["tiles"], got["rows"]) == (0, 0, 0)


# FP64 and refined contexts whose slots the rows pad (8, 27) or whose partial
# moments they keep per 64 velocities (216)
@pytest.mark.parametrize("nc,precision", [(2, 0), (3, 0), (6, 0), (2, 1), (3, 1)])
def test_rows_that_do_not_fit_leave_the_hyperplane_layout(checker, nc, precision):
    rows = _host(checker, {}, nc, precision, 0)
    hyper = _host(checker, {"PIKS_SWEEP_FLOW": "0"}, nc, precision, 0)
    assert (rows["rows"], hyper["rows"]) == (1, 0)
    assert rows["bytes"] > hyper["bytes"]
    # they fit: nothing changes
    assert _host(checker, {}, nc, precision, 0, str(rows["bytes"])) == rows
    # they do not: what PIKS_SWEEP_FLOW=0 lays out, to the last index
    assert _host(checker, {}, nc, precision, 0, str(rows["bytes"] - 1)) == hyper
    assert _host(checker, {}, nc, precision, 0, str(hyper["bytes"])) == hyper


def test_sweeps_asked_for_stay_whatever_fits(checker):
    # tiles; and the rows' layout where it is no larger (64 velocities)
    for env, nc, sweep in (({}, 3, 2), ({"PIKS_SWEEP_FLOW": "1"}, 3, 0), ({}, 4, 0)):
        got = _host(checker, env, nc, 0, sweep)
        assert _host(checker, env, nc, 0, sweep, str(got["bytes"] - 1)) == got
