"""The reverse-update kernels at the sizes where they can go wrong: rows that
end inside a vector, grids narrower than a tile, tiles of one row, every
boundary code on every face (the mirror points are computed apart), receiver
boxes that reach the halo, odd step counts and checkpoint intervals (the
gradient of two steps is added at once).

Against the float64 oracle within the bounds of test_gpu_adjoint (1e-10 in
float64, where only the order of sums differs; 1e-4 in float32); the tiled and
the one-point kernels, and every checkpoint interval, give the same bits (the
same operations in the same order).
"""
import os

import numpy as np
import pytest

import cases
import harness
import simwave_amd as sw
from simwave_amd import adjoint
from simwave_amd.middleware import Middleware
from test_gpu_adjoint import F32, F64, REC_TOL, TOL, oracle

pytestmark = pytest.mark.gpu

D, N, O = "null_dirichlet", "null_neumann", "none"
GRIDS = {
    "3d_so2": ((9, 66, 67), 2, (N, D, D, D, D, D)),
    "3d_so8": ((9, 13, 66), 8, (N, N, N, N, N, N)),
    "3d_so12": ((8, 9, 65), 12, (D, N, N, D, N, D)),
    "3d_so20": ((11, 12, 13), 20, (N, D, O, N, D, N)),
    "2d_so4": ((9, 259), 4, (N, D, D, N)),
    "2d_so20": ((11, 12), 20, (N, N, D, N)),
    "2d_so8": ((70, 9), 8, (D, D, D, D)),
}


def shot(name, dtype, damping):
    shape, so, bc = GRIDS[name]
    ext = [(n - 1) * 10.0 for n in shape]
    rec = [tuple(f * e for f, e in zip(row, ext))
           for row in ((0.02, 0.5, 0.5), (0.5, 0.01, 0.3), (0.4, 0.6, 0.99), (0.97, 0.98, 0.02))]
    parts = cases.make_case(dim=len(shape), shape=shape, space_order=so, dtype=dtype, bc=bc,
                            damping=damping, tf=0.03, window=2, rec=rec)()
    solver = sw.Solver(**parts)
    return solver, Middleware.normalize(**solver.forward_arguments())


# A Neumann face r+1 points from a Dirichlet one mirrors the plane that the
# other face zeroes, so that plane has an adjoint, and the gradient's step
# difference holds its zero in place of the value before it: the gradient on
# that plane is not the oracle's, in every version of these kernels.
THIN = pytest.mark.xfail(strict=True, reason="zeroed plane inside a mirror's reach")
ORACLE = [pytest.param(n, d, marks=THIN if (n, d) == ("3d_so20", 0.0) else ())
          for n in sorted(GRIDS) for d in (0.0, 20.0)]


def residual(kw, dtype):
    shape = (kw["end_timestep"], kw["num_receivers"])
    return np.random.default_rng(17).standard_normal(shape).astype(dtype)


@pytest.mark.parametrize("dtype", [F64, F32], ids=["f64", "f32"])
@pytest.mark.parametrize("name,damping", ORACLE)
def test_reverse_update_matches_oracle(name, damping, dtype):
    print("reverse update", name, damping, np.dtype(dtype).name, flush=True)
    solver, kw = shot(name, dtype, damping)
    rr = residual(kw, dtype)
    d_ref, g_ref, gw_ref = oracle(kw, rr.astype(F64))
    _, img_ref, _ = oracle(kw, rr.astype(F64), image=True)
    out = adjoint.gradient(solver, rr, checkpoint_every=3, wavelet_gradient=True)
    img = adjoint.image(solver, rr, checkpoint_every=3)
    assert np.abs(g_ref).max() > 0
    assert harness.rel_l2(out["shot_record"], d_ref) < REC_TOL[dtype]
    assert harness.rel_l2(out["grad_wavelet"], gw_ref) < TOL[dtype]
    assert harness.rel_l2(img, img_ref) < TOL[dtype]
    assert harness.rel_l2(out["grad_velocity"], g_ref) < TOL[dtype]


@pytest.mark.parametrize("dtype", [F64, F32], ids=["f64", "f32"])
@pytest.mark.parametrize("damping", [0.0, 20.0], ids=["undamped", "damped"])
@pytest.mark.parametrize("name", sorted(GRIDS))
def test_reverse_update_same_bits(name, damping, dtype):
    print("reverse update bits", name, damping, np.dtype(dtype).name, flush=True)
    solver, kw = shot(name, dtype, damping)
    rr = residual(kw, dtype)
    outs = [adjoint.gradient(solver, rr, checkpoint_every=k, wavelet_gradient=True)
            for k in (3, kw["end_timestep"], 1, 2, 4)]
    os.environ["SIMWAVE_HIP_UNTILED"] = "1"
    try:
        outs.append(adjoint.gradient(solver, rr, checkpoint_every=3, wavelet_gradient=True))
    finally:
        del os.environ["SIMWAVE_HIP_UNTILED"]
    for o in outs[1:]:
        for key in ("shot_record", "grad_velocity", "grad_wavelet"):
            np.testing.assert_array_equal(o[key], outs[0][key])
