"""Launches of more workgroups than one grid dimension holds (2^32 work items): the kernels that fold their
grid, at the first, a middle and the last rows, with nothing stored past the end."""
import ctypes as C

import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu


def read(uk, buf, offset, count, dtype=np.float32):
    out = np.empty(count, dtype)
    assert uk.lib.uk_memcpy_dtoh(out.ctypes.data_as(C.c_void_p), C.c_void_p(buf.ptr.value + offset), out.nbytes) == 0
    return out


def output(uk, nbytes):
    b = uk.DeviceBuffer(nbytes + 64)
    b.fill(0xFF)
    return b


def guard(uk, buf, nbytes):
    return (read(uk, buf, nbytes, 16, np.uint32) == 0xFFFFFFFF).all()


@pytest.mark.parametrize("variant, batch", [(10, (1 << 24) + 5), (11, (1 << 23) + 5), (12, (1 << 23) + 5), (13, (1 << 24) + 5)])
def test_conv_images(gpu, variant, batch):
    # One workgroup per image, of 256 or 512 threads.
    d = gpu.make_desc("conv", [2, 2, 2, 2, 2, 1], layout="NCHW", batch=batch)
    plan = gpu.Plan()
    plan.family, plan.variant = 7, variant
    check_conv(gpu, d, plan, batch, 8, 1)


def test_conv_images_by_the_solvers_plan(gpu):
    batch = (1 << 24) + 5
    d = gpu.make_desc("conv", [3, 3, 3, 3, 3, 16], layout="NCHW", batch=batch)
    check_conv(gpu, d, gpu.solve(d).plan, batch, 27, 16)


def check_conv(gpu, d, plan, batch, K, Oc):
    # Small integers: every sum is exact.
    x = np.resize(np.arange(8191, dtype=np.uint32) * np.uint32(2654435761) >> np.uint32(28), batch * K).astype(np.float32).reshape(batch, K)
    w = (np.arange(Oc * K, dtype=np.float32) % 7).reshape(Oc, K)
    xb, wb, yb = gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer.from_array(w), output(gpu, batch * Oc * 4)
    gpu.launch(d, [xb, wb], yb, plan=plan)
    assert np.array_equal(read(gpu, yb, 0, batch * Oc).reshape(batch, Oc), x @ w.T) and guard(gpu, yb, batch * Oc * 4)


def test_q8_0_tiles(gpu):
    # 8.4 M tiles of 512 threads (34 GB of outputs, of which three rows are read back).
    M, N, K = 1048560, 8193, 64
    from test_gpu_q8_0 import make_weights
    blocks, _, _ = make_weights(N, K, 5)
    Xh = np.resize(O.f16_bits(O.normal(4099 * K, 6, 0.0, 1.0)), M * K).reshape(M, K)
    p = gpu.Plan()
    p.family, p.variant = 8, 13
    xb, wb, yb = gpu.DeviceBuffer.from_array(Xh), gpu.DeviceBuffer.from_array(blocks), output(gpu, M * N * 4)
    gpu.launch(gpu.make_desc("gemm", [M, N, K], dtype="q8_0", layout="TN"), [xb, wb], yb, plan=p)
    rows = [0, M // 2 + 7, M - 1]
    want = O.q8_0_gemm(Xh[rows], blocks, N)
    for r, ref in zip(rows, want):
        got = read(gpu, yb, r * N * 4, N)
        assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)
    assert guard(gpu, yb, M * N * 4)


def test_row_sums(gpu):
    # Four rows of 64 threads to a workgroup of 256: 2^24 workgroups and one row more.
    L, n = (1 << 26) + 1, 5
    x = np.resize(np.arange(13, dtype=np.float32), L * n).reshape(L, n)
    xb, yb = gpu.DeviceBuffer.from_array(x), output(gpu, L * 4)
    p = gpu.Plan()
    p.family = 2
    gpu.launch(gpu.make_desc("reduce", [L, n]), [xb], yb, plan=p)
    assert np.array_equal(read(gpu, yb, 0, L), x.sum(axis=1)) and guard(gpu, yb, L * 4)


def test_channelscale(gpu):
    # 4.3e9 floats in workgroups of 4096: the fold into y starts at 2^20 of them.
    L, n = (1 << 20) + 3, 4097
    s = O.uniform(n, 9, 0.5, 1.5)
    xb, sb, yb = gpu.DeviceBuffer(L * n * 4), gpu.DeviceBuffer.from_array(s), output(gpu, L * n * 4)
    xb.fill(0x3F)
    gpu.launch(gpu.make_desc("channelscale", [L, n]), [xb, sb], yb)
    want = s * np.full(1, 0x3F3F3F3F, np.uint32).view(np.float32)
    for r in (0, L // 2, L - 1):
        assert np.array_equal(read(gpu, yb, r * n * 4, n), want)
    assert guard(gpu, yb, L * n * 4)


def test_row_sums_of_multiples_of_four(gpu):
    # Registers-resident rows of 64: 2^24 workgroups and one row more, in two launches.
    L, n = (1 << 26) + 1, 64
    xb, yb = gpu.DeviceBuffer(L * n * 4), output(gpu, L * 4)
    xb.fill(0x3F)
    gpu.launch(gpu.make_desc("reduce", [L, n]), [xb], yb)
    want = 64 * np.full(1, 0x3F3F3F3F, np.uint32).view(np.float32)
    assert (read(gpu, yb, 0, L) == want).all() and guard(gpu, yb, L * 4)


def test_softmax_in_two_launches(gpu):
    # Every element 1/64, in place of X; read back at the start, around the second launch's first row and at the end.
    L, n = (1 << 26) + 1, 64
    xb = output(gpu, L * n * 4)
    xb.fill(0x3F)
    gpu.launch(gpu.make_desc("softmax", [L, n]), [xb], xb)
    for r in (0, (1 << 26) - 8, L - 1):
        assert (read(gpu, xb, r * n * 4, n) == 1 / 64).all()


def test_pixels_of_a_1x1_conv(gpu):
    d = gpu.make_desc("conv", [16384, 16384, 1, 1, 1, 1], layout="NCHW", batch=4)
    n = 4 << 28
    xb, wb, yb = gpu.DeviceBuffer(n * 4), gpu.DeviceBuffer.from_array(np.float32([2])), output(gpu, n * 4)
    xb.fill(0x3F)
    gpu.launch(d, [xb, wb], yb)
    want = 2 * np.full(1, 0x3F3F3F3F, np.uint32).view(np.float32)
    for at in (0, n // 2, n - 4096):
        assert (read(gpu, yb, at * 4, 4096) == want).all()
    assert guard(gpu, yb, n * 4)


@pytest.mark.parametrize("variant", [7, 0])
def test_gemm_tiles(gpu, variant):
    # 1.3 M tiles of 16x16, or of 64x64: the fold into y starts at 2^20 of them. Small integers: exact.
    M, N = (4194240, 80) if variant == 7 else (4194240, 1025)
    a = (np.arange(M, dtype=np.int64) * 7 % 13).astype(np.float16)
    b = (np.arange(N) % 11).astype(np.float16)
    p = gpu.Plan()
    p.family, p.variant = 6, variant
    ab, bb, cb = gpu.DeviceBuffer.from_array(a), gpu.DeviceBuffer.from_array(b), output(gpu, M * N * 2)
    gpu.launch(gpu.make_desc("gemm", [M, N, 1], dtype="fp16", layout="TN"), [ab, bb], cb, plan=p)
    for r in (0, M // 2 + 3, M - 1):
        assert np.array_equal(read(gpu, cb, r * N * 2, N, np.float16), a[r] * b)
    assert guard(gpu, cb, M * N * 2)
