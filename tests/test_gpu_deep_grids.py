"""Grids with more z planes than a launch takes blocks along y or z (65536): the
tiled kernel's set-up shares them between fewer blocks.  Variable density, which
ran on the z-marching kernel before, against that kernel, bit for bit."""
import numpy as np
import pytest

import cases
import simwave_amd as sw
from simwave_amd.device import DeviceForward

pytestmark = pytest.mark.gpu


def test_more_planes_than_blocks(gpu, monkeypatch):
    print("deep grid", flush=True)
    solver = sw.Solver(**cases.make_case(dim=3, shape=(66000, 15, 15), space_order=6,
                                         density=True, damping=20.0, tf=0.004, window=2,
                                         src=[(659560.0, 70.0, 70.0)])())
    assert solver.space_model.extended_shape[0] - 6 > 65536
    dev = DeviceForward(solver)
    dev.run()
    assert dev.timings()[7] == 1
    want = dev.results()
    monkeypatch.setenv("SIMWAVE_HIP_ZMARCH", "1")
    dev.reset()
    dev.run()
    assert dev.timings()[7] == 2
    got = dev.results()
    assert np.abs(want[0]).max() > 0
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)
