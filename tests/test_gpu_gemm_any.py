"""The any-shape GEMM kernels at the edges of their tiles, against the CPU oracle.

Every compiled variant (plan family 6) in both layouts and types, at sizes one below, at and above
its tile, row segment (128 bytes of k) and chunk (16 bytes) boundaries, through operands aligned
to one element only. Bounds: f32 sums of K products in [-1, 1] in any order stay within
K * 2^-24 * sum|a b| of the exact sum, Frobenius about sqrt(K) * 2^-24 (2e-6 at K = 1100), gate 1e-5; f16
results add one rounding to half (2^-11 relative at most, 2.1e-4 Frobenius), gate 1e-3.
"""
import ctypes as C

import numpy as np
import pytest

import _oracle as O
from test_gpu_gemm import f16_inputs, frob

pytestmark = pytest.mark.gpu

VARIANTS = [0, 2, 3, 4, 5, 6, 7, 8, 9, 10]
F16_ONLY = (5, 6)
# ragged around 64/128/256 tiles; K below a chunk, across a chunk, across segments and k groups
SHAPES = [(1, 1, 1), (1, 3, 2), (5, 7, 3), (16, 64, 64), (17, 65, 63), (63, 33, 9), (65, 129, 257), (130, 255, 72),
          (257, 260, 1091)]


def run(uk, A, B, dtype, layout, variant, off, family=6):
    """One launch with every operand `off` elements past a 256-byte boundary."""
    M, K = A.shape
    N = B.shape[0] if layout == "TN" else B.shape[1]
    es = A.itemsize
    d = uk.make_desc("gemm", [M, N, K], dtype=dtype, layout=layout)
    p = uk.Plan()
    p.family, p.variant = family, variant
    guard = 64
    bufs = []
    for a in (A, B):
        flat = np.zeros(a.size + off, a.dtype)
        flat[off:] = a.ravel()
        bufs.append(uk.DeviceBuffer.from_array(flat))
    out = uk.DeviceBuffer((M * N + off + guard) * es)
    out.fill(0xFF)

    class At:
        def __init__(self, b):
            self.ptr = C.c_void_p(b.ptr.value + off * es)

    uk.launch(d, [At(b) for b in bufs], At(out), plan=p)
    flat = out.download(A.dtype, (M * N + off + guard,)).view(np.uint16 if es == 2 else np.uint32)
    edge = np.iinfo(flat.dtype).max
    assert (flat[:off] == edge).all() and (flat[off + M * N:] == edge).all()  # nothing stored outside C
    return flat[off:off + M * N].reshape(M, N).view(A.dtype)


@pytest.mark.parametrize("layout", ["TN", "NT"])
@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("dtype", ["fp16", "fp32"])
def test_edges(gpu, dtype, variant, layout):
    if dtype == "fp32" and variant in F16_ONLY:
        pytest.skip("compiled for f16 only")
    for i, (M, N, K) in enumerate(SHAPES):
        if dtype == "fp16":
            A, B = f16_inputs(M, N, K, 900 + i, tn=(layout == "TN"))
            R = O.gemm_f16q(A, B, layout == "TN")
        else:
            A = O.uniform(M * K, 910 + i, -1.0, 1.0).reshape(M, K)
            B = O.uniform(N * K, 920 + i, -1.0, 1.0).reshape((N, K) if layout == "TN" else (K, N))
            R = O.gemm_f32(A, B, layout == "TN")
        got = run(gpu, A, B, dtype, layout, variant, off=i % 4)
        if dtype == "fp16":
            got = O.f16_to_f32(got)
        assert frob(got, R) <= (1e-3 if dtype == "fp16" else 1e-5), (M, N, K)


@pytest.mark.parametrize("layout", ["TN", "NT"])
@pytest.mark.parametrize("variant", VARIANTS)
def test_non_finite_values_stay_in_their_rows_and_columns(gpu, variant, layout):
    # K = 70 leaves a partial segment and N, M partial tiles: what lies past an edge must not reach a
    # sum (0 * inf is NaN). One infinity in the last row of A and one NaN in the last column of B.
    M, N, K = 35, 37, 70
    A, B = f16_inputs(M, N, K, 77)
    A, B = O.f16_to_f32(A), O.f16_to_f32(B)
    A[M - 1, K - 1] = np.inf
    B[N - 1, 0] = np.nan
    Ah, Bh = O.f16_bits(A), O.f16_bits(B if layout == "TN" else np.ascontiguousarray(B.T))
    got = O.f16_to_f32(run(gpu, Ah, Bh, "fp16", layout, variant, off=1))
    want = A.astype(np.float64) @ B.T.astype(np.float64)
    assert np.isnan(got[:, N - 1]).all()
    assert np.array_equal(got[M - 1, :N - 1], want[M - 1, :N - 1].astype(np.float32))  # +-inf
    assert frob(got[:M - 1, :N - 1], want[:M - 1, :N - 1]) <= 1e-3


@pytest.mark.parametrize("layout", ["TN", "NT"])
@pytest.mark.parametrize("variant", [7, 8, 9, 10])
@pytest.mark.parametrize("dtype, K", [("fp16", 4999), ("fp32", 2501)])
def test_skinny_unrolled_loop(gpu, dtype, K, variant, layout):
    # Wavefronts take the segments of k in turn, up to four of their own at a time: with 78 whole segments (156 steps
    # in NT) each of up to sixteen runs the unrolled loop, some the one-segment remainder, one the partial segment.
    M, N = 17, 65
    if dtype == "fp16":
        A, B = f16_inputs(M, N, K, 940, tn=(layout == "TN"))
        got, R = O.f16_to_f32(run(gpu, A, B, dtype, layout, variant, off=1)), O.gemm_f16q(A, B, layout == "TN")
    else:
        A = O.uniform(M * K, 941, -1.0, 1.0).reshape(M, K)
        B = O.uniform(N * K, 942, -1.0, 1.0).reshape((N, K) if layout == "TN" else (K, N))
        got, R = run(gpu, A, B, dtype, layout, variant, off=1), O.gemm_f32(A, B, layout == "TN")
    assert frob(got, R) <= (1e-3 if dtype == "fp16" else 1e-5)


Q8_TILES = [11, 12, 13]  # 32x64, 64x64, 32x32


@pytest.mark.parametrize("variant", Q8_TILES)
@pytest.mark.parametrize("M,N,K", [(1, 1, 64), (17, 33, 64), (31, 65, 192), (64, 128, 320), (129, 130, 1088)])
def test_q8_0_tiles(gpu, variant, M, N, K):
    # Edges of the tiles in M and N, and numbers of block pairs that leave k groups without one (K = 64
    # to 320 over four groups). f32 sums of exact products: the gate of the other Q8_0 tests.
    from test_gpu_q8_0 import make_weights, q8_gpu
    p = gpu.Plan()
    p.family, p.variant = 8, variant
    blocks, _, _ = make_weights(N, K, 40 + variant)
    Xh = O.f16_bits(O.normal(M * K, 41 + M, 0.0, 1.0)).reshape(M, K)
    assert frob(q8_gpu(gpu, Xh, blocks, N, plan=p), O.q8_0_gemm(Xh, blocks, N)) <= 1e-5


@pytest.mark.parametrize("variant", Q8_TILES)
def test_q8_0_tiles_keep_infinities(gpu, variant):
    # An infinite activation in the last block pair of the last row: that row's outputs are +-inf (a
    # k group without a pair of its own must add nothing), the others finite.
    from test_gpu_q8_0 import make_weights, q8_gpu
    M, N, K = 33, 40, 192
    p = gpu.Plan()
    p.family, p.variant = 8, variant
    blocks, q, _ = make_weights(N, K, 3)
    X = O.normal(M * K, 4, 0.0, 1.0).reshape(M, K)
    X[M - 1, K - 1] = np.inf
    y = q8_gpu(gpu, O.f16_bits(X), blocks, N, plan=p)
    sign = np.asarray(q).reshape(N, K)[:, K - 1]
    assert np.array_equal(y[M - 1][sign != 0], np.where(sign[sign != 0] > 0, np.inf, -np.inf).astype(np.float32))
    assert np.isfinite(y[:M - 1]).all()


@pytest.mark.parametrize("M, N, K", [(1, 1, 1), (255, 191, 63), (256, 192, 64), (257, 193, 65), (513, 385, 321), (130, 960, 72)])
def test_256x192(gpu, M, N, K):
    # Variant 11, compiled for B [N][K] only: the edges of its tile, and columns of no power of two.
    A, B = f16_inputs(M, N, K, 930 + N, tn=True)
    got = O.f16_to_f32(run(gpu, A, B, "fp16", "TN", 11, off=N % 4))
    assert frob(got, O.gemm_f16q(A, B, True)) <= 1e-3
    if M == 257:
        with pytest.raises(gpu.UnikernError):
            run(gpu, A, B.reshape(K, N), "fp16", "NT", 11, off=0)


@pytest.mark.parametrize("dtype, layout, M, N, K", [("fp32", "TN", 64, 64, 64), ("fp32", "NT", 64, 192, 64), ("fp32", "NT", 128, 960, 128),
                                                    ("fp32", "TN", 64, 1984, 512), ("fp16", "TN", 128, 128, 32),
                                                    ("fp16", "TN", 128, 640, 1024), ("fp16", "TN", 128, 1664, 96)])
def test_few_whole_tiles_take_any_element_alignment(gpu, dtype, layout, M, N, K):
    # The solver's own plan, whichever kernel it names, at shapes of whole tiles too few for the aligned kernels.
    plan = gpu.solve(gpu.make_desc("gemm", [M, N, K], dtype=dtype, layout=layout)).plan
    if dtype == "fp16":
        A, B = f16_inputs(M, N, K, 950, tn=True)
        R = O.gemm_f16q(A, B, True)
    else:
        A = O.uniform(M * K, 951, -1.0, 1.0).reshape(M, K)
        B = O.uniform(N * K, 952, -1.0, 1.0).reshape((N, K) if layout == "TN" else (K, N))
        R = O.gemm_f32(A, B, layout == "TN")
    for off in (0, 1):
        got = run(gpu, A, B, dtype, layout, plan.variant, off, plan.family)
        if dtype == "fp16":
            got = O.f16_to_f32(got)
        assert frob(got, R) <= (1e-3 if dtype == "fp16" else 1e-5)
