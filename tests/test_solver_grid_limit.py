"""No plan names a kernel whose grid holds 2^32 work items or more in one dimension: the runtime would run
what is left of them modulo 2^32."""
import pytest

ITEMS = 1 << 32


@pytest.mark.parametrize("desc, refused", [
    (dict(op="conv", dims=[16384, 16384, 1, 1, 1, 1], layout="NCHW", batch=4), "conv_tile:s4"),
    (dict(op="gemm", dims=[131072, 262144, 64], dtype="fp32", layout="TN"), "gemm_f32"),
    (dict(op="gemm", dims=[1, 1 << 26, 256], dtype="q8_0", layout="TN"), "q8_0:gemv"),
    (dict(op="gemm", dims=[4, (1 << 26) + 64, 64], dtype="q8_0", layout="TN"), "q8_0:waves=16"),
])
def test_kernels_of_one_grid_dimension(uk, desc, refused):
    d = dict(desc)
    s = uk.solve(uk.make_desc(d.pop("op"), d.pop("dims"), **d))
    assert not s.key.startswith(refused) and f"candidate {refused}" not in s.log
    assert "violates one grid dimension's work items" in s.log
    folds = s.key.startswith(("conv_any", "gemm_tile", "gemm_skinny", "gemm_generic", "q8_0:tile"))
    assert folds or s.plan.grid * s.plan.threads < ITEMS
