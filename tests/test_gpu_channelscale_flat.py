"""channelscale over the flat array: row lengths that divide neither a 16-byte access nor a workgroup's share,
shorter than one access, and totals at the edges of the two workgroup sizes. One multiply per element: the
results are the same bits."""
import ctypes
from types import SimpleNamespace

import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L, C", [(1, 1), (1, 3), (5, 1), (4099, 1), (1025, 2), (341, 3), (257, 4), (1, 1023), (3, 1025), (9, 2047),
                                  (512, 4097), (1, 70001), (2048, 1024), (2049, 1023), (523, 4099), (32000, 83), (300001, 7)])
@pytest.mark.parametrize("off", [0, 1])
def test_flat(gpu, L, C, off):
    X = O.normal(L * C + off, 51 + C, 0.0, 1.0)
    S = O.uniform(C + off, 52, 0.5, 1.5)
    es, guard = 4, 16
    at = lambda b: SimpleNamespace(ptr=ctypes.c_void_p(b.ptr.value + off * es))
    xb, sb, yb = gpu.DeviceBuffer.from_array(X), gpu.DeviceBuffer.from_array(S), gpu.DeviceBuffer((L * C + off + guard) * es)
    yb.fill(0xFF)
    gpu.launch(gpu.make_desc("channelscale", [L, C]), [at(xb), at(sb)], at(yb))
    Y = yb.download(np.uint32, (L * C + off + guard,))
    want = X[off:].reshape(L, C) * S[off:]
    assert np.array_equal(Y[off:off + L * C], want.ravel().view(np.uint32))
    assert (Y[:off] == 0xFFFFFFFF).all() and (Y[off + L * C:] == 0xFFFFFFFF).all()  # nothing stored outside Y
