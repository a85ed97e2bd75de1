"""A sweep by rows whose waits gave up is reported once, and the context goes
on: tests/row_failure_check.cpp sets the poll limit of the kernel's own bounded
waits to 0 from the host."""
import os
import shutil
import subprocess

import pytest

import piks3d_amd
from piks3d_amd import images

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.parametrize("graph", ["0", "1"])
def test_failed_wait_is_reported_once(graph, tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe, raw = str(tmp_path / "row_failure_check"), str(tmp_path / "image.raw")
    lib = os.path.dirname(piks3d_amd.LIB_PATH)
    subprocess.run([gxx, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
                    "-I" + os.path.join(REPO, "piks3d_amd", "csrc"), "-I" + os.path.join(REPO, "include"), "-o", exe,
                    os.path.join(HERE, "row_failure_check.cpp"), "-L" + lib, "-lpiks3d", "-Wl,-rpath," + lib,
                    "-L" + os.path.join(ROCM, "lib"), "-lamdhip64", "-Wl,-rpath," + os.path.join(ROCM, "lib")],
                   check=True)
    images.write_raw(raw, images.sphere_pack(24, 0.40, 3.0, 6.0, seed=3))
    print("24^3 pack, graph", graph, flush=True)
    r = subprocess.run([exe, raw, "24", "24", "24", graph], capture_output=True, text=True, timeout=100,
                       env={k: v for k, v in os.environ.items() if not k.startswith("PIKS_")})
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split() == ["0", "-5", "0", "0", "kind", "2", "finite", "1"], r.stdout
