"""Rows of any length through the unaligned register-resident kernel (plan family 2), at the edges of
every compiled width: the width itself, one float more than the one before it, and a length that leaves
a partial float4. Gates as for the other row kernels: max_rel 1e-5 against binary64, row-sum
|y - r| <= 1e-5 sum|x|.
"""
import numpy as np
import pytest

import _oracle as O
from test_gpu_rows import check_rowsum, max_rel, rmsnorm64, run_op, softmax64

pytestmark = pytest.mark.gpu

CAPS = sorted({t * n * 4 for t, n in [(64, 1), (64, 2), (64, 3), (64, 4), (64, 6), (64, 8), (256, 3), (256, 4), (256, 5), (256, 6),
                                      (256, 8), (256, 10), (256, 12), (256, 16), (1024, 1), (1024, 2), (1024, 3), (1024, 4),
                                      (1024, 5), (1024, 6), (1024, 8), (1024, 10), (1024, 12), (1024, 15), (1024, 18)]})
LENGTHS = sorted({c for i, cap in enumerate(CAPS) for c in (cap, (CAPS[i - 1] if i else 0) + 1, cap - 1)}) + [73729]


def plan(uk):
    p = uk.Plan()
    p.family = 2
    return p


@pytest.mark.parametrize("C", LENGTHS)
def test_every_width(gpu, C):
    # 3 rows take the 1024-thread teams; 513 rows the 256-thread ones (up to 16384 floats, kept to
    # widths whose 513 rows are quick on the host).
    for L in (3, 513) if 2048 < C <= 6145 else (3,):
        X = O.normal(L * C, 7 + C, 0.0, 2.0).reshape(L, C)
        W = O.normal(C, 8 + C, 1.0, 0.1)
        check_rowsum(X, run_op(gpu, "reduce", X, plan=plan(gpu)))
        assert max_rel(run_op(gpu, "rmsnorm", X, W, plan=plan(gpu)), rmsnorm64(X, W)) <= 1e-5
        assert max_rel(run_op(gpu, "softmax", X * 4, plan=plan(gpu)), softmax64(X * 4)) <= 1e-5


@pytest.mark.parametrize("C", [5, 257, 3001, 20001])
def test_softmax_masked_and_non_finite_rows(gpu, C):
    X = O.normal(8 * C, 3 + C, 0.0, 2.0).reshape(8, C)
    lowest = np.finfo(np.float32).min
    X[1, 1:] = -np.inf      # one live element
    X[2, ::2] = lowest      # a mask of the lowest value
    X[3, :] = lowest        # nothing but the mask: uniform
    X[4, :] = -np.inf
    X[5, C - 1] = np.inf
    X[6, 0] = np.nan
    Y = run_op(gpu, "softmax", X, plan=plan(gpu))
    live = [0, 1, 2, 3, 7]
    with np.errstate(over="ignore"):
        assert max_rel(Y[live], softmax64(X[live])) <= 1e-5
    assert np.isnan(Y[[4, 5, 6]]).all()
