"""The cooperative receiver gather on boxes of every shape the C ABI takes,
against the oracle library on the same arguments (bit for bit: both sum a
receiver's products in box order).  Boxes of one point, of the window widths
the frontend makes, cut at the grid's edges, longer than one LDS round and
with more axis weights than the kernel keeps in LDS; receiver counts around
the kernel's group sizes."""
import ctypes

import numpy as np
import pytest

import cases
import harness
import simwave_amd as sw
from simwave_amd.middleware import Middleware

pytestmark = pytest.mark.gpu

F32, F64 = np.float32, np.float64


def _forward(kw, kind):
    kw = dict(kw, u_full=kw["u_full"].copy(), shot_record=np.zeros_like(kw["shot_record"]))
    dens = "variable_density" if kw.get("density_model") is not None else "constant_density"
    prec = "-DFLOAT" if kw["velocity_model"].dtype == F32 else "-DDOUBLE"
    lib = ctypes.CDLL(harness.LibraryCompiler(kind).compile(kw["velocity_model"].ndim, dens, prec,
                                                            "forward"))
    argtypes, args = Middleware.ordered(kw)
    lib.forward.argtypes = argtypes
    lib.forward.restype = ctypes.c_double
    assert lib.forward(*args) >= 0
    return kw["u_full"], kw["shot_record"]


def _boxes(rng, shape, count, widths, dtype):
    iv, vals, off = [], [], [0]
    for r in range(count):
        for n in shape:
            w = min(int(widths[int(rng.integers(len(widths)))]), n)
            lo = int(rng.integers(0, n - w + 1))
            iv += [lo, lo + w - 1]
            vals.append(rng.uniform(-1.0, 1.0, w))
        off.append(sum(len(v) for v in vals))
    return (np.array(iv, dtype=np.uint), np.concatenate(vals).astype(dtype),
            np.array(off, dtype=np.uint))


CASES = [(dim, dtype, count, widths)
         for dim, dtype in ((2, F32), (2, F64), (3, F32), (3, F64))
         for count, widths in ((1, (9,)), (7, (1, 2)), (8, (8, 9)), (17, (3, 9, 21)),
                               (33, (1, 9, 40)))]


@pytest.mark.parametrize("dim,dtype,count,widths", CASES)
def test_receiver_boxes(gpu, dim, dtype, count, widths):
    print("receivers", dim, dtype.__name__, count, widths, flush=True)
    parts = cases.make_case(dim=dim, n=30, space_order=4, dtype=dtype, tf=0.03)()
    kw = Middleware.normalize(**sw.Solver(**parts).forward_arguments())
    rng = np.random.default_rng([dim, count, len(widths)])
    kw["u_full"] = rng.standard_normal(kw["u_full"].shape).astype(dtype)
    iv, vals, off = _boxes(rng, kw["velocity_model"].shape, count, widths, dtype)
    kw.update(rec_points_interval=iv, rec_points_interval_size=len(iv), rec_points_values=vals,
              rec_points_values_size=len(vals), rec_points_values_offset=off,
              num_receivers=count,
              shot_record=np.zeros((kw["shot_record"].shape[0], count), dtype=dtype))
    (u_h, r_h), (u_o, r_o) = _forward(kw, "hip"), _forward(kw, "oracle")
    assert np.array_equal(u_h, u_o)
    assert np.any(r_o) and np.array_equal(r_h, r_o)
