"""The receiver gather inside the 3D step launches, whose group size, rounds and
values in flight follow the LDS of each tile: every default tile and the
z-marching kernels, on boxes of one point up to more axis weights than the
launch keeps in LDS (32), against the oracle bit for bit."""
import numpy as np
import pytest

import cases
import simwave_amd as sw
from simwave_amd.middleware import Middleware
from test_gpu_receivers import F32, F64, _boxes, _forward

pytestmark = pytest.mark.gpu

# density, type, space order, SIMWAVE_HIP_TILE (None: the z-marching kernel)
LAUNCHES = ([(False, F32, so, t) for so, t in ((6, 17), (8, 17), (8, 10), (12, 8), (20, 8))] +
            [(False, F64, so, t) for so, t in ((2, 18), (4, 18), (6, 18), (8, 10), (12, 4), (20, 8))] +
            [(True, F32, so, 0) for so in (2, 4, 6, 8, 12)] +
            [(True, F64, so, 0) for so in (2, 4, 6, 8, 12)] +
            [(vd, t, so, None) for vd in (False, True) for t in (F32, F64) for so in (2, 6, 8)])


@pytest.mark.parametrize("density,dtype,so,tile", LAUNCHES)
def test_gather_beside_step(gpu, density, dtype, so, tile, monkeypatch):
    print("gather beside", density, dtype.__name__, so, tile, flush=True)
    if tile is None:
        monkeypatch.setenv("SIMWAVE_HIP_ZMARCH", "1")
    else:
        monkeypatch.setenv("SIMWAVE_HIP_TILE", str(tile))
    parts = cases.make_case(dim=3, n=34, space_order=so, dtype=dtype, density=density,
                            tf=0.012, damping=0.0)()
    kw = Middleware.normalize(**sw.Solver(**parts).forward_arguments())
    for count, widths in ((1, (9,)), (67, (1, 9, 10, 11, 23))):
        rng = np.random.default_rng([so, count])
        kw["u_full"] = rng.standard_normal(kw["u_full"].shape).astype(dtype)
        iv, vals, off = _boxes(rng, kw["velocity_model"].shape, count, widths, dtype)
        kw.update(rec_points_interval=iv, rec_points_interval_size=len(iv),
                  rec_points_values=vals, rec_points_values_size=len(vals),
                  rec_points_values_offset=off, num_receivers=count,
                  shot_record=np.zeros((kw["shot_record"].shape[0], count), dtype=dtype))
        (u_h, r_h), (u_o, r_o) = _forward(kw, "hip"), _forward(kw, "oracle")
        assert np.array_equal(u_h, u_o)
        assert np.any(r_o) and np.array_equal(r_h, r_o)
