"""An earlier failed HIP call of the thread is no failure of the next transfer, of a step
in one launch or of the next integrator."""
import ctypes

import numpy as np
import pytest

from physicsbasedanimationtoolkit_amd import _native, pbat

from test_gpu_local import DT, build, grid

pytestmark = pytest.mark.gpu


@pytest.fixture
def fail_a_hip_call(gpu_device):
    hip = ctypes.CDLL(_native.LIBRARY_PATH)  # finds the runtime the library is linked to

    def fail():
        p = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 60)) != 0 and not p.value

    yield fail
    hip.hipGetLastError()  # clears it


def test_later_calls(fail_a_hip_call):
    X, E, dbc = grid(4, 3, 5)
    d = build(X, E, dbc)[0]
    g = pbat.gpu.vbd.Integrator(d)
    x = (X + 0.01).astype(np.float32)
    fail_a_hip_call()
    g.x = x
    fail_a_hip_call()
    assert np.array_equal(g.x, x)
    fail_a_hip_call()
    fresh = pbat.gpu.vbd.Integrator(d)
    assert np.array_equal(fresh.x, X.astype(np.float32))
    fail_a_hip_call()
    fresh.step(DT, 1, 1)
    assert np.isfinite(fresh.x).all()
