"""Rounding of Q8_0 sums with more than 16 activation rows.

An output is a sum of K/32 scaled blocks in f32. The split-k kernels sum one chain per wavefront; the
tiles sum in blocks of four, which rounds off less (1.02 times as much at K = 128). So the sixteen-wavefront kernel
(variant 1, any K) bounds the tiles' error against binary64 over the same inputs, and the solver takes
no split-k kernel of fewer, longer chains in its place.
"""
import numpy as np
import pytest

import _oracle as O

TILES = [11, 12, 13]


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 192, 640, 2112, 4096, 9792, 11008])
def test_tiles_round_off_no_more_than_sixteen_chains(gpu, K):
    from test_gpu_q8_0 import frob, make_weights, q8_gpu
    M, N = 96, 320
    blocks, _, _ = make_weights(N, K, 60 + K)
    Xh = O.f16_bits(O.normal(M * K, 61 + K, 0.0, 1.0)).reshape(M, K)
    r = O.q8_0_gemm(Xh, blocks, N)
    ys = {}
    for v in [1] + TILES:
        p = gpu.Plan()
        p.family, p.variant = 8, v
        ys[v] = q8_gpu(gpu, Xh, blocks, N, plan=p)
    for v in TILES:
        if K == 64:  # one block pair: the same two fused multiply-adds
            assert np.array_equal(ys[v].view(np.uint32), ys[1].view(np.uint32))
        # 30720 outputs: the ratio of two such 2-norms scatters by 1 / sqrt(2 * 30720) = 0.4%.
        assert frob(ys[v], r) <= 1.01 * frob(ys[1], r), v


@pytest.mark.parametrize("M,N,K", [(72, 64, 9536), (132, 563, 9792), (256, 67, 8320), (34, 175, 9856), (106, 508, 10752),
                                   (259, 64, 9664), (128, 384, 8768)])
def test_solver_keeps_sixteen_chains(uk, M, N, K):
    # Shapes whose cheapest split-k kernel by the weight stream has sixteen wavefronts: a kernel of
    # fewer takes longer and rounds off more.
    s = uk.solve(uk.make_desc("gemm", [M, N, K], dtype="q8_0", layout="TN"))
    assert s.key.startswith("q8_0:tile") or s.plan.split_k == 16


def test_solver_keeps_the_streams_kernel_over_several_rounds(uk):
    s = uk.solve(uk.make_desc("gemm", [375, 250, 10752], dtype="q8_0", layout="TN"))
    assert s.key == "q8_0:waves=8,pairs=4,vec=4,nt=3"
