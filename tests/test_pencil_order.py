"""The row sweep's records where the storage order has y as its outer axis
(build_pencil_schedule in piks3d_amd/csrc/geometry.cpp: images whose two layers
of z exceed a window's 32-bit offsets): the same cells, task by task, as where z
is.  tests/pencil_order_check.cpp, compiled with g++; the window's limit is
reached on small images with large slots."""
import os
import shutil
import subprocess

import pytest

from piks3d_amd import images

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(REPO, "piks3d_amd", "csrc")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("pencil_order") / "pencil_order_check"
    subprocess.run([gxx, "-O2", "-std=c++17", "-I" + CSRC, "-I" + os.path.join(REPO, "include"), "-o", str(out),
                    os.path.join(HERE, "pencil_order_check.cpp"), os.path.join(CSRC, "geometry.cpp"), "-lpthread"],
                   check=True)
    return str(out)


# (nz, ny, nx), elements per slot: 2^28 / slot is a window's limit in cells
@pytest.mark.parametrize("rows", [4, 1000])
@pytest.mark.parametrize("shape,slot", [((6, 31, 20), 1 << 18), ((9, 40, 13), 1 << 18), ((3, 50, 17), 1 << 18)])
def test_records_over_y_layers_name_the_same_cells(checker, tmp_path, shape, slot, rows):
    img = images.box_blocks(shape, 14, 1, 4, 7)
    path = str(tmp_path / "image.raw")
    images.write_raw(path, img)
    nz, ny, nx = shape
    r = subprocess.run([checker, path, str(nx), str(ny), str(nz), "2", "2", str(rows), str(slot)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    words = r.stdout.split()
    assert int(words[1]) > 0 > int(words[2])     # z is the outer axis of the first, y of the second
    assert int(words[4]) > 0 and words[-1] == "0"
