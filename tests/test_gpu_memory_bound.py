"""Runs whose device memory holds everything but the tiled kernel's packed
coefficients (bounded here by SIMWAVE_HIP_RUN_MB): they take the other kernels
and give the same bits; a bound below those kernels' arrays is an error."""
import math

import numpy as np
import pytest
import torch  # noqa: F401  (one HIP runtime per process: torch's, so before the library)

import cases
import simwave_amd as sw
from simwave_amd import adjoint
from simwave_amd.device import DeviceForward

pytestmark = pytest.mark.gpu

# experiment, and the arrays of one value per point that the z-marching or
# generic kernels hold besides the wavefields (q, e)
CASES = {
    "cd_so12": dict(space_order=12, shape=(90, 100, 120)),
    "cd_f64": dict(space_order=4, shape=(70, 80, 100), dtype=np.float64),
    "vd_so8": dict(space_order=8, shape=(128, 128, 128), density=True),
    "vd_oblong": dict(space_order=4, shape=(90, 96, 130), density=True),
}


def solver_of(name):
    s = sw.Solver(**cases.make_case(dim=3, tf=0.012, damping=20.0, window=3, **CASES[name])())
    s._middleware.verbose = False
    return s


def bound(solver, arrays):
    sm = solver.space_model
    mb = np.prod(sm.extended_shape) * np.dtype(sm.dtype).itemsize / 2.0 ** 20
    assert mb > 4                       # a megabyte is a fraction of an array
    return str(math.ceil((arrays + 0.4) * mb))


@pytest.mark.parametrize("name", sorted(CASES))
def test_forward_without_room_for_packed_coefficients(name, monkeypatch):
    print("bounded forward", name, flush=True)
    solver = solver_of(name)
    dev = DeviceForward(solver)
    dev.run()
    assert dev.timings()[7] == 1        # tiled
    want = dev.results()
    host = solver.forward()
    monkeypatch.setenv("SIMWAVE_HIP_RUN_MB", bound(solver, 2))
    dev.reset()
    dev.run()
    assert dev.timings()[7] != 1
    for a, b in zip(dev.results(), want):
        np.testing.assert_array_equal(a, b)
    dev.reset()
    dev.plan()
    assert dev.run_steps(dev.steps) == 0
    for a, b in zip(dev.results(), want):
        np.testing.assert_array_equal(a, b)
    dev.release_plan()
    # the host entry holds the three slots, the halo frame's indices and values
    # (below one array) and the density too
    monkeypatch.setenv("SIMWAVE_HIP_RUN_MB", bound(solver, 6 + CASES[name].get("density", 0)))
    for a, b in zip(solver.forward(), host):
        np.testing.assert_array_equal(a, b)
    monkeypatch.setenv("SIMWAVE_HIP_RUN_MB", bound(solver, 1))
    with pytest.raises(RuntimeError, match="out of memory"):
        dev.run()


@pytest.mark.parametrize("stride", [1, 2, 3])
def test_host_call_that_saves_levels(stride, monkeypatch):
    """Buffers are taken as slots are first used: the run starts over as long
    as no output has been returned."""
    print("bounded host call, stride", stride, flush=True)
    params = dict(CASES["vd_oblong"], stride=stride)
    s = sw.Solver(**cases.make_case(dim=3, tf=0.012, damping=20.0, window=3, **params)())
    s._middleware.verbose = False
    want = s.forward()
    # q, e, the density, four slots and the halo frame
    for arrays in (8, 13):              # without and with some of the packed values
        monkeypatch.setenv("SIMWAVE_HIP_RUN_MB", bound(s, arrays))
        for a, b in zip(s.forward(), want):
            np.testing.assert_array_equal(a, b)
    monkeypatch.setenv("SIMWAVE_HIP_RUN_MB", bound(s, 4))
    with pytest.raises(RuntimeError, match="out of memory"):
        s.forward()


@pytest.mark.parametrize("name", ["cd_so12", "cd_f64"])
def test_gradient_without_room_for_packed_coefficients(name, monkeypatch):
    print("bounded gradient", name, flush=True)
    solver = solver_of(name)
    T = solver.time_model.timesteps
    dtype = solver.space_model.dtype
    rr = np.random.default_rng(2).standard_normal((T, solver.receivers.count)).astype(dtype)
    want = adjoint.gradient(solver, rr, checkpoint_every=T)
    # q, e, C, two adjoint levels with their products, the sums, T + 2 levels
    monkeypatch.setenv("SIMWAVE_HIP_RUN_MB", bound(solver, 8 + T + 2))
    got = adjoint.gradient(solver, rr, checkpoint_every=T)
    for key in ("shot_record", "grad_velocity"):
        np.testing.assert_array_equal(got[key], want[key])
    monkeypatch.setenv("SIMWAVE_HIP_RUN_MB", bound(solver, T + 2))
    with pytest.raises(RuntimeError, match="out of memory"):
        adjoint.gradient(solver, rr, checkpoint_every=T)
