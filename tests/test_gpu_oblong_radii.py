"""Variable density with nx != ny on the tiled kernel at every radius and type,
with both forms of the quotients, by default and where nothing fits a whole
tile: against the oracle library, bit for bit."""
import numpy as np
import pytest

import cases
import harness
from test_gpu_parity import _step_kernel_of_last_run

pytestmark = pytest.mark.gpu

F32, F64 = np.float32, np.float64


@pytest.mark.parametrize("quotients", ["", "SIMWAVE_HIP_IEEE_DIV"], ids=["default", "ieee"])
@pytest.mark.parametrize("dtype", [F32, F64], ids=["f32", "f64"])
@pytest.mark.parametrize("so", range(2, 21, 2))
def test_oblong_every_radius(gpu, so, dtype, quotients, monkeypatch):
    print("oblong", so, np.dtype(dtype).name, quotients, flush=True)
    if quotients:
        monkeypatch.setenv(quotients, "1")
    r = so // 2
    for i, (nx, ny) in enumerate(((r + 9, 75), (67, r + 6))):
        setup = cases.make_case(dim=3, density=True, shape=(r + 5 + i, nx, ny), space_order=so,
                                dtype=dtype, tf=0.02, damping=20.0 * i, window=2,
                                bc=("null_neumann", "null_dirichlet", "none", "null_neumann",
                                    "null_dirichlet", "none"))
        u_h, r_h = harness.run(setup, "hip")
        assert _step_kernel_of_last_run(3, "vd", "f64" if dtype is F64 else "f32") == 1
        u_o, r_o = harness.run(setup, "oracle")
        assert np.any(u_o) and np.array_equal(u_h, u_o) and np.array_equal(r_h, r_o)
