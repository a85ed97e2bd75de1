"""Every kernel of the sweep by rows against the hyperplane launches
(PIKS_SWEEP_FLOW=0), bit for bit, each context saying which of the two it runs:
the FP64 iteration, and in the refined precision whole defect-correction
blocks (the FP64 iteration of a block, first and later FP32 corrections, and the
block that folds the last one's correction), at velocity counts around the chunks
of 64 (8, 27, 64, 216 per octant), with one and several Knudsen numbers."""
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


def _run(p, img, kn, precision, block, steps, env, monkeypatch):
    for k in ("PIKS_SWEEP_FLOW", "PIKS_FLOW_WAVES", "PIKS_DC_BLOCK"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    with (MultiSolver(p, img, kn, precision=precision) if kn else Solver(p, img, precision=precision)) as s:
        kind = s.sweep_kind()
        if block:
            s.set_correction_block(block)
        s.iterate(steps)     # no field is read on the way: reading folds a correction
        n32 = s.get_info().steps_fp32
        fields = [np.stack(s.macro_rhs(r)) for r in range(len(kn))] if kn else [np.stack(s.macro())]
        return kind, n32, fields + [s.f(), s.fw()]


@pytest.mark.parametrize("waves", [0, 8])
@pytest.mark.parametrize("precision,shape,nc,kn", [
    ("fp64", (21, 13, 18), 2, ()), ("fp64", (9, 30, 11), 3, ()), ("fp64", (33, 17, 12), 4, ()),
    ("fp64", (12, 11, 16), 6, ()), ("fp64", (17, 12, 15), 3, (0.1, 0.7, 5.0)), ("fp64", (10, 12, 9), 6, (0.2, 3.0)),
    ("fp32", (14, 19, 12), 2, ()), ("fp32", (11, 12, 13), 3, ()), ("fp32", (19, 14, 23), 4, ()),
    ("fp32", (12, 11, 16), 6, ()), ("fp32", (13, 12, 11), 4, (0.1, 0.7, 5.0)), ("fp32", (10, 12, 9), 6, (0.2, 3.0))])
def test_rows_kernels_equal_hyperplanes(precision, shape, nc, kn, waves, monkeypatch):
    p, img = _case(shape, nc)
    print(precision, shape, nc, kn, waves, flush=True)
    # blocks of 3: block, first, later, fold, first, later, fold, first (8 steps)
    block, steps = (3, 8) if precision == "fp32" else (0, 5)
    rows = {"PIKS_FLOW_WAVES": str(waves)} if waves else {}
    ref = _run(p, img, kn, precision, block, steps, {"PIKS_SWEEP_FLOW": "0"}, monkeypatch)
    got = _run(p, img, kn, precision, block, steps, rows, monkeypatch)
    assert (ref[0], got[0]) == ("hyperplanes", "rows")
    assert ref[1] == got[1] == (5 if precision == "fp32" else 0)
    assert np.isfinite(ref[2][0]).all()
    for a, b in zip(got[2], ref[2]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("how", ["parameter", "environment"])
def test_tiles_asked_for_run_whatever_the_flow_setting(how, monkeypatch):
    p, img = _case((21, 13, 18), 4)
    if how == "parameter":
        p.sweep = 2
    tiles = {"PIKS_SWEEP_TILES": "1"} if how == "environment" else {}
    monkeypatch.delenv("PIKS_SWEEP_TILES", raising=False)
    ref = _run(p, img, (), "fp64", 0, 3, tiles, monkeypatch)
    got = _run(p, img, (), "fp64", 0, 3, {"PIKS_SWEEP_FLOW": "1", **tiles}, monkeypatch)
    assert ref[0] == got[0] == "tiles"
    for a, b in zip(got[2], ref[2]):
        assert np.array_equal(a, b)
