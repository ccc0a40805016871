"""The tiled 3D kernel with variable density (square planes, and planes with
nx != ny, where the reference's x-axis first derivatives step by nx
elements), and the float64-product quotients of both densities where they
become subnormal: against the oracle library, bit for bit.  SIMWAVE_HIP_TILE
forces the kernel on grids below its size rule."""
import numpy as np
import pytest

import cases
import harness
import simwave_amd as sw
from simwave_amd.middleware import Middleware
from test_gpu_parity import _step_kernel_of_last_run
from test_gpu_receivers import _forward

pytestmark = pytest.mark.gpu

F32, F64 = np.float32, np.float64
BC = ("null_neumann", "null_dirichlet", "null_neumann", "none", "null_dirichlet", "null_neumann")

CASES = {
    # every radius family, both types
    **{"so%d" % so: dict(shape=(24 + so, 30, 30), space_order=so)
       for so in (2, 4, 6, 8, 10, 12, 16, 18, 20)},
    **{"f64_so%d" % so: dict(shape=(24 + so, 28, 28), space_order=so, dtype=F64)
       for so in (4, 8, 10, 16, 20)},
    # several tiles across, odd widths, damping under branch-free tiles
    "wide": dict(shape=(40, 141, 141), space_order=8, damping=40.0, tf=0.03),
    "wide_h12p5": dict(shape=(40, 139, 139), space_order=8, h=12.5, damping=50.0, tf=0.04),
    "wide_so12": dict(shape=(34, 101, 101), space_order=12, damping=40.0, tf=0.03),
    "wide_f64": dict(shape=(36, 75, 75), space_order=8, dtype=F64, damping=40.0, tf=0.03),
    # faces, sources at the surface, several wavelets
    "faces": dict(shape=(30, 33, 33), space_order=8, damping=0.0, bc=BC,
                  src=[(0.0, 100.0, 120.0), (8.0, 5.0, 200.0)], multi=True),
    "dirichlet": dict(shape=(44, 37, 37), space_order=8, bc=("null_dirichlet",) * 6),
    # nx != ny, either one larger, thin and wide
    "oblong_xy": dict(shape=(26, 40, 29), space_order=4),
    "oblong_yx": dict(shape=(26, 27, 68), space_order=8),
    "oblong_thin": dict(shape=(30, 25, 130), space_order=8, damping=0.0, bc=BC),
    "oblong_long": dict(shape=(24, 150, 26), space_order=16, damping=20.0, tf=0.03),
    "oblong_so20": dict(shape=(44, 34, 45), space_order=20, tf=0.03),
    "oblong_f64": dict(shape=(28, 31, 50), space_order=8, dtype=F64),
    "oblong_f64_so12": dict(shape=(34, 36, 30), space_order=12, dtype=F64),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_variable_density_tiles(gpu, name, monkeypatch):
    print("tiled variable density", name, flush=True)
    monkeypatch.setenv("SIMWAVE_HIP_TILE", "0")
    params = dict(dict(dim=3, density=True, tf=0.05), **CASES[name])
    setup = cases.make_case(**params)
    u_h, r_h = harness.run(setup, "hip")
    assert _step_kernel_of_last_run(3, "vd", "f64" if params.get("dtype") == F64 else "f32") == 1
    u_o, r_o = harness.run(setup, "oracle")
    assert np.array_equal(u_h, u_o) and np.array_equal(r_h, r_o)


@pytest.mark.parametrize("density", [False, True])
@pytest.mark.parametrize("scale", [1e-44, 1e-37, 1e-33])
def test_subnormal_quotients(gpu, density, scale, monkeypatch):
    """Random initial levels so small that the quotients of h = 10 m are
    subnormal or close to it."""
    print("subnormal quotients", density, scale, flush=True)
    monkeypatch.setenv("SIMWAVE_HIP_TILE", "17")
    parts = cases.make_case(dim=3, shape=(30, 32, 32), space_order=8, density=density, damping=30.0,
                            tf=0.02)()
    kw = Middleware.normalize(**sw.Solver(**parts).forward_arguments())
    rng = np.random.default_rng(4)
    kw["u_full"] = (rng.standard_normal(kw["u_full"].shape) * scale).astype(F32)
    kw["wavelet"] = np.zeros_like(kw["wavelet"])
    (u_h, r_h), (u_o, r_o) = _forward(kw, "hip"), _forward(kw, "oracle")
    assert np.any(u_o) and np.array_equal(u_h, u_o) and np.array_equal(r_h, r_o)


@pytest.mark.parametrize("dtype", [F32, F64], ids=["f32", "f64"])
@pytest.mark.parametrize("shape", [(19, 8, 133), (13, 67, 67), (12, 131, 20)])
def test_radius2_tiles(gpu, shape, dtype, monkeypatch):
    """Radius 2 has a tile of its own: 4 rows, 64 points (float64 32)."""
    print("radius 2 tiles", shape, np.dtype(dtype).name, flush=True)
    monkeypatch.setenv("SIMWAVE_HIP_TILE", "0")
    setup = cases.make_case(dim=3, density=True, tf=0.05, shape=shape, space_order=4, dtype=dtype,
                            bc=BC, window=3)
    u_h, r_h = harness.run(setup, "hip")
    assert _step_kernel_of_last_run(3, "vd", "f64" if dtype is F64 else "f32") == 1
    u_o, r_o = harness.run(setup, "oracle")
    assert np.array_equal(u_h, u_o) and np.array_equal(r_h, r_o)
