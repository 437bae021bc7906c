"""Softmax of rows of any length, element by element against binary64.

A 2-norm sees only the large elements. Here every x - max is exact in f32 (multiples of 1/1024 down to
-104, maximum 0), so an element y_i over the row's largest, 1/s, is e^x_i with the roundings of the
exponential (an ulp of v_exp_f32 and half an ulp of its argument) and of two quotients: at most
2^-23 + 2^-24 + 2 * 2^-24. Elements under the normal range are denormals, not zeros.
"""
import numpy as np
import pytest

import _oracle as O
from test_gpu_rows import run_op

pytestmark = pytest.mark.gpu


# One row length per team width (64, 256 and 1024 threads a row), with and without a partial float4, and
# more than 512 rows for the 256-thread teams.
@pytest.mark.parametrize("L, C", [(5, 83), (3, 429), (700, 2051), (600, 5003), (2, 2051), (3, 16388), (2, 70001)])
def test_every_element(gpu, L, C):
    k = (O.uniform(L * C, 40 + C, 0.0, 1.0).reshape(L, C) * 104 * 1024).astype(np.int64)
    k[:, C // 2] = 0
    X = (-k / 1024.0).astype(np.float32)
    p = gpu.Plan()
    p.family = 2
    Y = run_op(gpu, "softmax", X, plan=p).astype(np.float64)
    E = np.exp(X.astype(np.float64))
    R = E / E.sum(axis=1, keepdims=True)
    normal = R >= 2.0 ** -125
    ratio = Y / Y[:, C // 2][:, None]
    assert np.all(np.abs(ratio - E)[normal] <= 5 * 2.0 ** -24 * E[normal])
    # A denormal numerator and its quotient each round by half of 2^-149.
    assert np.all(np.abs(Y - R)[~normal] <= 1.01 * 2.0 ** -149 + 2.0 ** -20 * R[~normal])
    assert (~normal).any() and np.all(Y[R >= 2.0 ** -148] > 0)


@pytest.mark.parametrize("L, C", [(2000, 429), (700, 2051), (600, 5003), (400, 5003), (300, 16388)])
def test_the_rows_sum_adds_little(gpu, L, C):
    # A row's sum is shared by all its elements. With the threads' sums added in binary64 what is left of a row's
    # distance is the elements' own roundings (about 2^-25 rms for the quotient and as much for v_exp_f32) and those of
    # a thread's few additions: 3.2e-8 to 4.3e-8 measured, 8.0e-8 to 9.5e-8 with all the additions in f32.
    X = O.normal(L * C, 50 + C, 0.0, 8.0).reshape(L, C)
    p = gpu.Plan()
    p.family = 2
    Y = run_op(gpu, "softmax", X, plan=p).astype(np.float64)
    E = np.exp(X.astype(np.float64) - X.max(axis=1, keepdims=True).astype(np.float64))
    R = E / E.sum(axis=1, keepdims=True)
    assert np.linalg.norm(Y - R) <= 6.5e-8 * np.linalg.norm(R)
