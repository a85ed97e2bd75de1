"""Rows of 2^14 - 1 cells and more, whose records hold one x index: the sweep
by rows against the hyperplane launches, bit for bit, in each precision and
with several Knudsen numbers."""
import numpy as np
import pytest

from piks3d_amd import MultiSolver, Solver, images
from piks3d_amd.params import Params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,nc", [("fp64", 4), ("fp64", 3), ("refined", 2), ("multi", 2)])
@pytest.mark.parametrize("nx", [16378, 16379])     # Nx = 16382 (short records), 16383 (long ones)
def test_long_rows_equal_hyperplanes(nx, kind, nc, monkeypatch):
    img = images.box_blocks((4, 5, nx), nx // 20, 1, 3, 5)
    p = Params(nx=nx, ny=5, nz=4, fluid_layer=2, wall_ext_order=2, nc_fundamental=nc, half_range=True,
               exact_quadrature=nc == 3, chk_converge_step=10, max_step=100, eps=0.0, kn=0.7, press_drop=1.0, accom=1.0)
    print(nx, kind, nc, flush=True)

    def run(flow):
        monkeypatch.delenv("PIKS_SWEEP_FLOW", raising=False)
        if flow is not None:
            monkeypatch.setenv("PIKS_SWEEP_FLOW", flow)
        with (MultiSolver(p, img, [0.1, 5.0]) if kind == "multi" else
              Solver(p, img, precision="fp32" if kind == "refined" else "fp64")) as s:
            if kind == "refined":
                s.set_correction_block(2)
            s.iterate(4)
            path = s.info.sweep_path
            return np.stack([np.asarray(m) for m in s.macro()]), s.f(), path

    ref, got = run("0"), run(None)
    assert (ref[2], got[2]) == (0, 2 if kind == "fp64" and nc == 4 else 0)
    assert np.isfinite(ref[0]).all()
    assert np.array_equal(ref[0], got[0])
    assert np.array_equal(ref[1], got[1])
