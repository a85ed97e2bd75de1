"""Host checks of the pencil sweep's schedule (build_pencil_schedule in
piks3d_amd/csrc/geometry.cpp): tests/pencil_records_check.cpp, compiled from
the library's geometry sources with g++, compares it task by task with the
hyperplane schedule of the same image (which tests/test_flow_records.py and
the GPU tests tie to the oracle): every task once, the same sources (switched
wall slots included, src/solver.F90:184-204 and analogues), waits on the
nearest swept row per axis, rows after the rows they read.  Ragged sides and
strips of one row, of a few, and of more rows than the image has."""
import os
import shutil
import subprocess

import pytest

from piks3d_amd import images

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(REPO, "piks3d_amd", "csrc")

CASES = [
    ("pack", lambda: images.sphere_pack(40, 0.40, 3.0, 6.0, seed=5, shape=(37, 41, 45)), 2, 2),
    ("sphere", lambda: images.centered_sphere(64, 28.0), 4, 2),
    ("boxes", lambda: images.box_blocks((14, 13, 16), 14, 2, 6, 3), 2, 1),
]


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("pencil_records") / "pencil_records_check"
    subprocess.run([gxx, "-O2", "-std=c++17", "-I" + CSRC, "-I" + os.path.join(REPO, "include"), "-o", str(out),
                    os.path.join(HERE, "pencil_records_check.cpp"), os.path.join(CSRC, "geometry.cpp"),
                    "-lpthread"], check=True)
    return str(out)


def _run(checker, tmp_path, case, *extra):
    name, make, layers, order = case
    img = make()
    path = str(tmp_path / (name + ".raw"))
    images.write_raw(path, img)
    nz, ny, nx = img.shape
    return subprocess.run([checker, path, str(nx), str(ny), str(nz), str(layers), str(order), *extra],
                          capture_output=True, text=True, timeout=300)


@pytest.mark.parametrize("rows", [1, 7, 1000])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_pencil_records(checker, tmp_path, case, rows):
    r = _run(checker, tmp_path, case, str(rows))
    assert r.returncode == 0, r.stdout + r.stderr
    assert "bad 0" in r.stdout
    assert "switched reads 0," not in r.stdout   # the images exercise switched reads


def test_planted_mistakes_are_found(checker, tmp_path):
    r = _run(checker, tmp_path, CASES[0], "7", "plant")
    assert "planted: wait mark 1, source 1" in r.stdout
    assert r.returncode == 1
    assert "FAIL wait mark" in r.stdout and "FAIL source" in r.stdout
