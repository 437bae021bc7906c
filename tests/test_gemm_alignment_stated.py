"""The solver's account of a plan states the alignment its launch asks for."""


def test_alignment_is_stated(uk):
    why = lambda dims: uk.solve(uk.make_desc("gemm", dims, dtype="fp16", layout="TN")).log.splitlines()[0]
    assert "gemm_skinny:32x32" in why([128, 2048, 4096]) and "16-byte aligned operands" in why([128, 2048, 4096])
    assert "any element alignment" in why([128, 2048, 4095])
