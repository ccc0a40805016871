"""The list of device blocks that one gradient keeps for the next
(sw_common.cpp), with made-up addresses, and on the device: the bits of a
repeated gradient, of one after another size, and the trim."""
import ctypes

import numpy as np
import pytest

import cases
from simwave_amd import adjoint
from simwave_amd import build as hipbuild
from simwave_amd.device import DeviceForward


@pytest.fixture
def common():
    lib = ctypes.CDLL(hipbuild.common_library_path())
    take, put, evict = (lib["simwave_hip_block_" + n] for n in ("take", "put", "evict"))
    u64, p = ctypes.c_ulonglong, ctypes.c_void_p
    take.restype = evict.restype = p
    take.argtypes = [ctypes.c_int, u64, ctypes.POINTER(u64)]
    put.argtypes = [ctypes.c_int, p, u64, u64]
    evict.argtypes = [ctypes.c_int, u64]

    def take_(device, need):
        got = u64(0)
        return take(device, need, ctypes.byref(got)), got.value
    yield take_, put, evict
    for device in (901, 902):
        while evict(device, 0):
            pass


def test_best_fit_within_a_quarter(common):
    take, put, evict = common
    assert put(901, 0x1000, 1000, 5000) == 1 and put(901, 0x2000, 1200, 5000) == 1
    assert put(902, 0x3000, 1000, 5000) == 1
    assert take(901, 900) == (0x1000, 1000)
    assert take(901, 900)[0] is None           # 1200 is a third larger
    assert take(901, 1201)[0] is None
    assert take(901, 1200) == (0x2000, 1200)
    assert take(901, 1000)[0] is None and take(902, 1000) == (0x3000, 1000)


def test_limit_and_eviction_order(common):
    take, put, evict = common
    assert put(901, 0x1000, 3000, 5000) == 1
    assert put(901, 0x2000, 2001, 5000) == 0   # over the limit
    assert put(901, 0x2000, 2000, 5000) == 1
    assert put(901, 0x4000, 6000, 5000) == 0
    assert evict(901, 5000) is None
    assert evict(901, 2500) == 0x1000          # the oldest
    assert evict(901, 2500) is None
    assert evict(902, 0) is None
    assert evict(901, 0) == 0x2000 and evict(901, 0) is None


@pytest.mark.gpu
def test_gradients_of_changing_sizes_keep_their_bits():
    import torch
    print("kept blocks", flush=True)

    def run(shape):
        _, solver, kw = cases.adjoint_shot("3d_so8", dtype=np.float32, shape=shape)
        rr = np.random.default_rng(4).standard_normal(
            (kw["end_timestep"], kw["num_receivers"])).astype(np.float32)
        return solver, adjoint.gradient(solver, rr, checkpoint_every=4)["grad_velocity"]
    shapes = [(60, 64, 70), (60, 64, 71), (40, 80, 50)]
    first = []
    for s in shapes:
        solver, g = run(s)
        first.append(g)
        lib = DeviceForward(solver, buffers="torch")._lib
        assert lib.simwave_hip_trim_pool() == 0      # nothing kept: fresh memory
    for s, g in list(zip(shapes, first)) * 2:
        np.testing.assert_array_equal(run(s)[1], g)
    held = torch.cuda.mem_get_info()[0]
    assert lib.simwave_hip_trim_pool() == 0
    assert torch.cuda.mem_get_info()[0] > held
