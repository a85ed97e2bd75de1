"""Records of the row sweep for rows too long for two x indices in a word
(build_pencil_schedule in piks3d_amd/csrc/geometry.cpp): the last length whose
records hold both and the first whose do not, and on a short image both kinds
of record against each other.  tests/pencil_wide_check.cpp, compiled with g++."""
import os
import shutil
import subprocess

import pytest

from piks3d_amd import images

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(REPO, "piks3d_amd", "csrc")
LAYERS = 2


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("pencil_wide") / "pencil_wide_check"
    subprocess.run([gxx, "-O2", "-std=c++17", "-I" + CSRC, "-I" + os.path.join(REPO, "include"), "-o", str(out),
                    os.path.join(HERE, "pencil_wide_check.cpp"), os.path.join(CSRC, "geometry.cpp"), "-lpthread"],
                   check=True)
    return str(out)


@pytest.mark.parametrize("shape,wide", [((12, 11, 19), 0), ((5, 6, 16382 - 2 * LAYERS), 0),
                                        ((5, 6, 16383 - 2 * LAYERS), 1), ((6, 5, 40000), 1)])
def test_records_of_long_rows(checker, tmp_path, shape, wide):
    img = images.box_blocks(shape, max(4, shape[2] // 40), 1, 3, 5)
    path = str(tmp_path / "image.raw")
    images.write_raw(path, img)
    nz, ny, nx = shape
    r = subprocess.run([checker, path, str(nx), str(ny), str(nz), str(LAYERS), "2", "3"], capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "wide %d " % wide in r.stdout and r.stdout.strip().endswith("bad 0")
