"""The any-shape conv kernel at the edges of its tiles, against the CPU oracle.

Every compiled variant (plan family 7, numbers 10-13) over both layouts, padding, strides, kernel sizes,
channel counts that are and are not multiples of 4 (the two HWC loads) and reductions shorter than, equal
to and one past a 32-k step. Gate: f32 sums of K products in any order, Frobenius <= 1e-5 as for the
other conv kernels.
"""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

VARIANTS = [10, 11, 12, 13]


def frob(got, ref):
    g, r = got.astype(np.float64), np.asarray(ref, np.float64)
    return float(np.linalg.norm(g - r) / np.linalg.norm(r))


def launch(uk, d, ins, shape, variant):
    p = uk.Plan()
    p.family, p.variant = 7, variant
    y = uk.DeviceBuffer(int(np.prod(shape)) * 4 + 256)
    y.fill(0xFF)
    uk.launch(d, [uk.DeviceBuffer.from_array(a) for a in ins], y, plan=p)
    flat = y.download(np.uint32, (int(np.prod(shape)) + 64,))
    assert (flat[-64:] == 0xFFFFFFFF).all()  # nothing stored past the output
    return flat[:-64].view(np.float32).reshape(shape)


# N, C, H, W, Oc, K, pad, stride: single pixels, ragged pixel and channel tiles, padding wider than the kernel's half
NCHW = [(1, 1, 1, 1, 1, 1, 0, 1), (2, 3, 9, 7, 17, 5, 2, 1), (1, 32, 8, 8, 64, 1, 0, 1), (3, 7, 13, 15, 65, 3, 1, 2),
        (1, 11, 20, 9, 33, 3, 3, 1), (2, 2, 17, 23, 5, 7, 0, 3), (1, 64, 12, 11, 130, 3, 1, 1)]


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("N,C,H,W,Oc,K,pad,stride", NCHW)
def test_nchw(gpu, variant, N, C, H, W, Oc, K, pad, stride):
    x = O.normal(N * C * H * W, 50 + C, 0.0, 1.0).reshape(N, C, H, W)
    w = O.normal(Oc * C * K * K, 51 + Oc, 0.0, 0.1).reshape(Oc, C, K, K)
    s = O.normal(Oc, 52, 1.0, 0.1)
    d = gpu.make_desc("conv", [H, W, C, K, K, Oc], layout="NCHW", batch=N, pad=pad, stride=stride, epilogue="channelscale")
    ref = O.conv_nchw(x, w, s, pad, stride)
    assert frob(launch(gpu, d, [x, w, s], ref.shape, variant), ref) <= 1e-5


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("C,H,W,Oc,K", [(1, 3, 3, 1, 3), (4, 9, 17, 5, 3), (5, 11, 10, 33, 3), (32, 18, 9, 64, 3), (36, 7, 20, 65, 1),
                                        (8, 12, 12, 20, 5)])
def test_hwc(gpu, variant, C, H, W, Oc, K):
    x = O.normal(C * H * W, 60 + C, 0.0, 1.0).reshape(H, W, C)
    w = O.normal(Oc * C * K * K, 61 + Oc, 0.0, 0.1).reshape(Oc, K, K, C)
    d = gpu.make_desc("conv", [H, W, C, K, K, Oc])
    ref = O.conv_nchw(np.ascontiguousarray(x.transpose(2, 0, 1))[None], np.ascontiguousarray(w.transpose(0, 3, 1, 2)),
                      np.ones(Oc, np.float32), 0, 1)[0]
    assert frob(launch(gpu, d, [x, w], ref.shape, variant), ref) <= 1e-5


@pytest.mark.parametrize("variant", VARIANTS)
def test_infinities_stay_in_their_windows(gpu, variant):
    # C = 5, 3x3: K = 45 leaves a partial step whose missing k must add nothing, and the zero padding
    # must not meet the infinite input.
    N, C, H, W, Oc = 1, 5, 12, 13, 9
    x = O.normal(C * H * W, 70, 0.0, 1.0).reshape(N, C, H, W)
    x[0, C - 1, H - 1, W - 1] = np.inf
    w = np.abs(O.normal(Oc * C * 9, 71, 0.0, 0.1)).reshape(Oc, C, 3, 3)
    d = gpu.make_desc("conv", [H, W, C, 3, 3, Oc], layout="NCHW", batch=N, pad=1)
    y = launch(gpu, d, [x, w], (N, Oc, H, W), variant)
    hit = np.zeros((H, W), bool)
    hit[H - 2:, W - 2:] = True
    assert np.isposinf(y[0][:, hit]).all() and np.isfinite(y[0][:, ~hit]).all()
