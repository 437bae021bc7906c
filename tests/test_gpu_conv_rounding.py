"""Rounding of the any-shape conv's sums: no further from binary64 than conv_tile (plan variant 6), which
took these shapes before, from reductions that fit one MFMA chain to a 3x3 kernel of 32 channels."""
import numpy as np
import pytest

import _oracle as O
from test_gpu_conv_any import VARIANTS, launch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,K", [(2, 1), (12, 1), (16, 1), (32, 1), (5, 3), (32, 3)])
@pytest.mark.parametrize("layout", ["NCHW", "NT"])
def test_rounds_off_no_more_than_conv_tile(gpu, layout, C, K):
    H, W, Oc = 40, 37, 64
    x = O.normal(C * H * W, 30 + C, 0.0, 1.0).reshape(1, C, H, W)
    w = O.normal(Oc * C * K * K, 31 + C, 0.0, 0.1).reshape(Oc, C, K, K)
    win = np.lib.stride_tricks.sliding_window_view(x[0].astype(np.float64), (K, K), axis=(1, 2))
    r = np.tensordot(w.astype(np.float64), win, axes=([1, 2, 3], [0, 3, 4]))
    d = gpu.make_desc("conv", [H, W, C, K, K, Oc], layout=layout)
    ins = [x, w] if layout == "NCHW" else [np.ascontiguousarray(x[0].transpose(1, 2, 0)), np.ascontiguousarray(w.transpose(0, 2, 3, 1))]
    err = lambda v: float(np.linalg.norm(launch(gpu, d, ins, r.shape, v).astype(np.float64) - r) / np.linalg.norm(r))
    before = err(6)
    # At least 85,000 outputs: the ratio of two such 2-norms scatters by 1 / sqrt(2 * 85000) = 0.25%.
    for v in VARIANTS:
        assert err(v) <= 1.01 * before, v
