"""The sweep by rows (one launch, a wave per row of cells) against the
hyperplane launches (PIKS_SWEEP_FLOW=0), bit for bit, at the edges of its
dispatch: velocity counts around its chunks of 64 (8, 27, 64, 216 per
octant), several Knudsen numbers, the refined precision, ragged sides down to
rows of a single swept cell, and fewer or more waves than rows."""
import numpy as np
import pytest

from piks3d_amd import MultiSolver, Solver, images
from piks3d_amd.params import Params

pytestmark = pytest.mark.gpu


def _case(shape, nc, seed=9):
    nx, ny, nz = shape
    img = images.box_blocks((nz, ny, nx), max(1, nx * ny * nz // 200), 1, 3, seed)
    p = Params(nx=nx, ny=ny, nz=nz, fluid_layer=2, wall_ext_order=2, nc_fundamental=nc, half_range=True,
               exact_quadrature=nc == 3, chk_converge_step=10, max_step=100, eps=0.0, kn=0.7, press_drop=1.0, accom=1.0)
    return p, img


def _run(make, waves, hyper, monkeypatch):
    for k in ("PIKS_SWEEP_FLOW", "PIKS_FLOW_WAVES"):
        monkeypatch.delenv(k, raising=False)
    if hyper:
        monkeypatch.setenv("PIKS_SWEEP_FLOW", "0")
    if waves:
        monkeypatch.setenv("PIKS_FLOW_WAVES", str(waves))
    with make() as s:
        out = []
        for _ in range(3):
            s.iterate(1)
            out.append(np.stack([np.asarray(m) for m in s.macro()]))
        return s.f(), s.fw(), out


@pytest.mark.parametrize("waves", [0, 8, 600])
@pytest.mark.parametrize("kind,shape,nc", [
    ("fp64", (21, 13, 18), 2), ("fp64", (9, 30, 11), 3), ("fp64", (33, 17, 12), 4),
    ("fp64", (12, 11, 16), 6), ("refined", (19, 14, 23), 4), ("refined", (11, 12, 13), 3), ("multi", (17, 12, 15), 3),
    ("multi", (16, 19, 13), 4)])
def test_rows_equal_hyperplanes(kind, shape, nc, waves, monkeypatch):
    p, img = _case(shape, nc)
    print(kind, shape, nc, waves, flush=True)
    if kind == "multi":
        make = lambda: MultiSolver(p, img, [0.1, 0.7, 5.0])
    else:
        make = lambda: Solver(p, img, precision="fp64" if kind == "fp64" else "fp32")
    ref = _run(make, 0, True, monkeypatch)
    got = _run(make, waves, False, monkeypatch)
    assert np.isfinite(ref[0]).all()
    for a, b in zip(got[:2] + tuple(got[2]), ref[:2] + tuple(ref[2])):
        assert np.array_equal(a, b)
