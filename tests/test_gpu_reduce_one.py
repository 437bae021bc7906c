"""The 1-D reduce of short vectors (one workgroup, one launch) at the edges of its passes and of its range."""
import ctypes
from types import SimpleNamespace

import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

PASS = 16 * 1024 * 4  # floats one pass of the workgroup takes
MOST = 1 << 18        # the longest vector it takes; one more runs the two passes


@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 4095, PASS - 1, PASS, PASS + 1, PASS + 4, 3 * PASS - 3, MOST, MOST + 1])
def test_reduce_one(gpu, n, off):
    x = np.abs(O.normal(n + off, 900 + n % 1000, 0.0, 1.0))
    xb, yb = gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer(4)
    at = SimpleNamespace(ptr=ctypes.c_void_p(ctypes.cast(xb.ptr, ctypes.c_void_p).value + 4 * off))
    gpu.launch(gpu.make_desc("reduce", [n]), [at], yb)
    y = float(yb.download(np.float32, (1,))[0])
    exact = float(np.sum(x[off:].astype(np.float64)))
    # Positive values: each f32 addition on a value's way rounds by half an ulp at most. At most 11 in the
    # one workgroup and the final rounding; in the two passes 12 to a partial and 17 among the partials.
    assert abs(y - exact) <= (12 if n <= MOST else 29) * 2.0 ** -24 * exact


@pytest.mark.parametrize("n", [1000, MOST])
def test_reduce_one_special_values(gpu, n):
    for bad in (np.inf, -np.inf, np.nan):
        x = np.ones(n, np.float32)
        x[n - 1] = bad
        xb, yb = gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer(4)
        gpu.launch(gpu.make_desc("reduce", [n]), [xb], yb)
        y = yb.download(np.float32, (1,))[0]
        assert np.isnan(y) if np.isnan(bad) else y == bad
