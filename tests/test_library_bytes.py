"""The bytes a shot is admitted by: what the library holds per point, with the
tiles' padding, and on the device that a shot runs within them on the kernel it
takes by itself."""
import numpy as np
import pytest

import cases
import simwave_amd as sw
from simwave_amd.device import DeviceForward, library_bytes
from simwave_amd.serving import shot_bytes

F32, F64 = np.float32, np.float64


def test_arrays_counted():
    n = 100 * 120
    assert library_bytes((100, 120), 8, 4, False) == 4 * n * 4
    assert library_bytes((100, 120), 8, 4, True) == 4 * n * 4       # no sums below order 12
    assert library_bytes((100, 120), 12, 8, True) == 6 * n * 8
    n = 28 * 29 * 73
    tiles = 20 * 24 * 128                                           # 21 rows, 65 points
    assert library_bytes((28, 29, 73), 8, 4, False) == (2 * n + 2 * tiles) * 4
    assert library_bytes((28, 29, 73), 8, 4, True) == (2 * n + 6 * tiles) * 4
    tiles = 20 * 32 * 96                                            # 16 rows, 32 points
    assert library_bytes((28, 29, 73), 8, 8, True) == (2 * n + 6 * tiles) * 8
    # a thin interior: the z-marching kernel's sums are the larger part
    n = 25 * 25 * 25
    assert library_bytes((25, 25, 25), 16, 4, True) == (2 * n + max(6 * 9 * 16 * 64, 3 * n)) * 4


@pytest.mark.parametrize("params", [dict(dim=2, n=60, density=True, space_order=8),
                                    dict(dim=2, n=60, density=True, space_order=16),
                                    dict(dim=3, shape=(12, 20, 30), density=True),
                                    dict(dim=3, shape=(12, 20, 30), dtype=F64)])
def test_shot_counts_its_arrays(params):
    solver = sw.Solver(**cases.make_case(tf=0.02, **params)())
    sm = solver.space_model
    esz = np.dtype(sm.dtype).itemsize
    own = (solver.num_snapshots + 2 + 2 + params.get("density", False)) * np.prod(sm.extended_shape)
    rec = solver.time_model.timesteps * solver.receivers.count
    lib = library_bytes(sm.extended_shape, sm.space_order, esz, params.get("density", False))
    assert shot_bytes(solver) == (own + rec) * esz + lib


@pytest.mark.gpu
@pytest.mark.parametrize("density", [False, True])
@pytest.mark.parametrize("dtype", [F32, F64])
@pytest.mark.parametrize("so", [2, 4, 6, 8, 12, 20])
def test_run_fits_the_counted_bytes(gpu, so, dtype, density, monkeypatch):
    print("counted bytes", so, dtype.__name__, density, flush=True)
    # one row and one point more than whole tiles of 8 by 64
    solver = sw.Solver(**cases.make_case(dim=3, shape=(60, 145, 193), space_order=so, dtype=dtype,
                                         density=density, damping=0.0, tf=0.004)())
    sm = solver.space_model
    dev = DeviceForward(solver)
    dev.run()
    kernel = dev.timings()[7]
    need = library_bytes(sm.extended_shape, so, np.dtype(dtype).itemsize, density)
    # 2 MB for the damping mask and the source and receiver tables
    monkeypatch.setenv("SIMWAVE_HIP_RUN_MB", str(need // 2 ** 20 + 2))
    dev.reset()
    dev.run()
    assert dev.timings()[7] == kernel
