"""Q8_0 activations that end where their allocation ends.

With at most eight activation rows the tile kernels copy 512-byte slices (four block pairs) of each
row into LDS; where K is no multiple of 256 the last slice must stop at the row's end. X sits in
the last bytes of a 2 MiB allocation, so a read past it leaves the allocation.
"""
import ctypes as C

import numpy as np
import pytest

import _oracle as O
from test_gpu_q8_0 import frob, make_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 40, 192), (4, 77, 192), (8, 33, 320), (1, 20, 8256), (5, 20, 64)])
def test_activations_end_with_their_allocation(gpu, M, N, K):
    size = 2 << 20
    blocks, _, _ = make_weights(N, K, 5 + K)
    Xh = O.f16_bits(O.normal(M * K, 6 + M, 0.0, 1.0)).reshape(M, K)
    image = np.zeros(size // 2, np.uint16)
    image[-M * K:] = Xh.ravel()
    xb, wb, yb = gpu.DeviceBuffer.from_array(image), gpu.DeviceBuffer.from_array(blocks), gpu.DeviceBuffer(M * N * 4)

    class Tail:
        ptr = C.c_void_p(xb.ptr.value + size - M * K * 2)

    gpu.launch(gpu.make_desc("gemm", [M, N, K], dtype="q8_0", layout="TN"), [Tail, wb], yb)
    assert frob(yb.download(np.float32, (M, N)), O.q8_0_gemm(Xh, blocks, N)) <= 1e-5
