"""The planes per z chunk that the tiled kernel takes by itself, on grids either
side of the rule's lines (1 M and 3 M interior points, radius, density, type),
against other chunk lengths: the same bits."""
import numpy as np
import pytest

import cases
import simwave_amd as sw
from simwave_amd.device import DeviceForward

pytestmark = pytest.mark.gpu

F32, F64 = np.float32, np.float64
GRIDS = [(False, F32, 18, (99, 100, 100)), (False, F32, 20, (101, 100, 100)),
         (False, F64, 10, (101, 100, 100)), (False, F64, 8, (143, 145, 146)),
         (False, F64, 16, (143, 145, 146)), (True, F32, 18, (103, 100, 101)),
         (True, F64, 4, (103, 100, 101)), (True, F64, 16, (146, 145, 147))]


@pytest.mark.parametrize("density,dtype,so,shape", GRIDS)
def test_chunk_length_keeps_bits(gpu, density, dtype, so, shape, monkeypatch):
    print("z chunks", density, dtype.__name__, so, shape, flush=True)
    solver = sw.Solver(**cases.make_case(dim=3, shape=shape, space_order=so, dtype=dtype,
                                         density=density, damping=0.0, tf=0.008)())
    outs = []
    for zlen in ("", "1", "2", "7"):
        monkeypatch.setenv("SIMWAVE_HIP_ZLEN", zlen)
        dev = DeviceForward(solver)
        dev.run()
        assert dev.timings()[7] == 1
        outs.append(dev.results())
    assert np.abs(outs[0][0]).max() > 0
    for u, rec in outs[1:]:
        np.testing.assert_array_equal(u, outs[0][0])
        np.testing.assert_array_equal(rec, outs[0][1])
