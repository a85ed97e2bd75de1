"""A request whose rows layout (whole-line slots, partial moments per 64
velocities) exceeds the server's memory budget runs on the hyperplane launches'
layout if that fits, with the same result bit for bit."""
import pytest

from piks3d_amd import Server, images
from piks3d_amd.params import Params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,precision", [(2, "fp64"), (2, "fp32"), (6, "fp64")])
def test_request_beyond_the_budget_takes_the_smaller_layout(nc, precision, monkeypatch):
    img = images.box_blocks((15, 14, 17), 10, 2, 4, 3)
    p = Params(nx=17, ny=14, nz=15, fluid_layer=2, wall_ext_order=2, nc_fundamental=nc, half_range=True,
               chk_converge_step=5, max_step=20, eps=0.0, kn=0.7, press_drop=1.0, accom=1.0)

    def solve(budget=0, flow=None):
        monkeypatch.delenv("PIKS_SWEEP_FLOW", raising=False)
        if flow is not None:
            monkeypatch.setenv("PIKS_SWEEP_FLOW", flow)
        with Server(max_slots=2, prep_threads=1, memory_budget=budget, tuning=None) as s:
            return s.wait(s.submit(p, img, precision=precision))

    print(nc, precision, flush=True)
    rows, hyper = solve(), solve(flow="0")
    assert rows["device_bytes"] > hyper["device_bytes"]
    got = solve(budget=hyper["device_bytes"])
    assert got["error_code"] == 0 and got["steps"] == 20
    assert got["device_bytes"] == hyper["device_bytes"]
    for key in ("mass", "permeability", "error", "steps"):
        assert got[key] == hyper[key] == rows[key], key
