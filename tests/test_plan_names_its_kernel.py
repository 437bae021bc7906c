"""A plan's fields say what is launched: the variant, tile, grid and threads of one kernel, the same whether
the plan comes from the solver, a ledger or a caller, and one key for one kernel."""
import numpy as np
import pytest

import _oracle as O


@pytest.mark.parametrize("layout, tile, threads", [("NT", (16, 64, 16), 1024), ("TN", (16, 16, 32), 512)])
def test_one_tile_products(uk, layout, tile, threads):
    p = uk.solve(uk.make_desc("gemm", [64, 64, 96], dtype="fp32", layout=layout)).plan
    assert (p.variant, p.tile_m, p.tile_n, p.tile_k) == (7, *tile)
    assert (p.threads, p.split_k) == (threads, threads // 64)
    assert p.grid == -(-64 // tile[0]) * -(-64 // tile[1])


def test_any_shape_keys(uk):
    key = lambda dims, **kw: uk.solve(uk.make_desc("gemm", dims, **kw))
    names = {}
    for M in (1, 17, 64, 65, 130, 1000):
        for N in (16, 64, 100, 1161, 4095):
            for K in (64, 333, 4095):
                s = key([M, N, K], dtype="fp16", layout="TN")
                names.setdefault(s.key, set()).add(s.plan.variant)
    assert all(len(v) == 1 for v in names.values()), names


def test_rows_of_any_length(uk):
    p = uk.solve(uk.make_desc("softmax", [2048, 5003])).plan
    assert p.key.decode() == f"rows_any:tpr={p.tpr},nv={p.vec}" and p.tpr * p.vec * 4 >= 5003
    assert uk.solve(uk.make_desc("softmax", [64, 80001])).key == "rows_stream"


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["TN", "NT"])
@pytest.mark.parametrize("variant", [0, 7])
def test_a_named_gemm_variant_runs(gpu, variant, layout):
    # The 64 rows of a one-tile product sum in the same order as the first 64 of 65, which no rule for one
    # tile applies to.
    from test_gpu_gemm_any import run
    M, N, K = 65, 48, 1000
    A = O.uniform(M * K, 21, -1.0, 1.0).reshape(M, K)
    B = O.uniform(N * K, 22, -1.0, 1.0).reshape((N, K) if layout == "TN" else (K, N))
    whole = run(gpu, A, B, "fp32", layout, variant, 0)
    assert np.array_equal(run(gpu, A[:64], B, "fp32", layout, variant, 0).view(np.uint32), whole[:64].view(np.uint32))


@pytest.mark.gpu
def test_a_named_row_width_runs(gpu):
    # Teams of 64 and of 1024 threads sum a row in different orders.
    from test_gpu_rows import check_rowsum, run_op
    X = O.normal(64 * 403, 23, 0.0, 1.0).reshape(64, 403)
    ys = []
    for tpr, nv in [(64, 2), (1024, 1)]:
        p = gpu.Plan()
        p.family, p.tpr, p.vec = 2, tpr, nv
        ys.append(run_op(gpu, "reduce", X, plan=p))
        check_rowsum(X, ys[-1])
    assert (ys[0] != ys[1]).any()
    p = gpu.Plan()
    p.family, p.tpr, p.vec = 2, 64, 2  # holds 512 floats: the launch takes a width that holds the row
    check_rowsum(X.reshape(-1, 806), run_op(gpu, "reduce", X.reshape(-1, 806), plan=p))
