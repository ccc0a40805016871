"""The tiled 3D kernel's damped update where den = 1 + e leaves the range of
its short float64 reciprocal: one damping value far outside anything the
frontend makes sends the whole run through the general division.  Against
the oracle library on the same arguments, bit for bit."""
import numpy as np
import pytest

import cases
import simwave_amd as sw
from simwave_amd.middleware import Middleware
from test_gpu_receivers import _forward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [0.0, 1e22, 3e33, -2e30])
def test_damping_far_out_of_range(gpu, value, monkeypatch):
    print("damping value", value, flush=True)
    monkeypatch.setenv("SIMWAVE_HIP_TILE", "17")
    parts = cases.make_case(dim=3, shape=(30, 24, 70), h=12.5, space_order=8, damping=50.0,
                            tf=0.04)()
    kw = Middleware.normalize(**sw.Solver(**parts).forward_arguments())
    kw["damping_mask"] = kw["damping_mask"].copy()
    if value:
        kw["damping_mask"][17, 12, 30] = value
    (u_h, r_h), (u_o, r_o) = _forward(kw, "hip"), _forward(kw, "oracle")
    assert np.any(u_o) and np.array_equal(u_h, u_o)
    assert np.array_equal(r_h, r_o)
