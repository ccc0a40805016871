"""The allocation-free entry near the size of its scratch: constant-density grids
keep the tiled kernel, whose packed coefficients are then formed from the
models and whose source terms read q and e of the source boxes' planes alone.
Bit for bit the allocating entry's results; a grid whose padded tiles do not
fit takes another kernel, with the same bits."""
import numpy as np
import pytest

import cases
import simwave_amd as sw
from simwave_amd.device import DeviceForward
from test_zz_no_alloc import _call

pytestmark = pytest.mark.gpu

F64 = np.float64
D, N = "null_dirichlet", "null_neumann"
ENDS = [(20.0, 320.0, 300.0), (1180.0, 900.0, 700.0)]      # first and last planes

# grid (extended by the halo alone: 4.5 to 5.4 M points in float32, 2.3 to 2.7
# in float64), kernel expected (1 tiled, 2 z-marching)
CASES = {
    "so12": (dict(shape=(150, 161, 183), space_order=12), 1),
    "so20_neumann": (dict(shape=(150, 140, 164), space_order=20, bc=(N,) * 6), 1),
    "so10_damped": (dict(shape=(130, 150, 170), space_order=10, damping=60.0), 1),
    "f64_so4": (dict(shape=(121, 130, 151), space_order=4, dtype=F64), 1),
    "f64_so8": (dict(shape=(117, 130, 147), space_order=8, dtype=F64), 1),
    "f64_so16": (dict(shape=(104, 120, 140), space_order=16, dtype=F64), 1),
    "so12_small": (dict(shape=(24, 30, 41), space_order=12, src=[(100.0, 120.0, 150.0)]), 1),
    "so12_ends": (dict(shape=(150, 161, 175), space_order=12, src=ENDS, multi=True), 2),
    "f64_so4_no_fit": (dict(shape=(340, 200, 33), space_order=4, dtype=F64), 2),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_noalloc_keeps_tiles(gpu, name):
    params, kernel = CASES[name]
    print("noalloc tiles", name, flush=True)
    params = dict(dict(dim=3, damping=0.0, tf=0.008, window=3), **params)
    dev = DeviceForward(sw.Solver(**cases.make_case(**params)()))
    u_a, r_a = _call(dev, noalloc=False)
    u_n, r_n = _call(dev, noalloc=True)
    assert dev.timings()[7] == kernel
    assert np.abs(u_a).max() > 0
    assert np.array_equal(u_n, u_a) and np.array_equal(r_n, r_a)
