"""The tuner's candidates (CPU): no two of a call that the library runs alike."""
import pytest

from xkblas_amd import tuner


@pytest.mark.parametrize("dtype,mode", [(0, 0), (1, 0), (1, 2)])
def test_potrf_without_a_block_order_has_one_candidate(dtype, mode):
    cands = tuner.candidates("potrf", dtype, mode, 8192, 8192, 8192)
    assert cands == [{"tile": 0, "nb": 0, "split": 0, "kernel": 0}]
    assert tuner.heuristic("potrf", dtype, mode, 8192, 8192, 8192) == cands[0]


@pytest.mark.parametrize("op,mode", [("potrf", 2), ("potrf", 3), ("trsm", 0), ("gemm", 0), ("syrk", 0)])
def test_candidates_differ(op, mode):
    cands = tuner.candidates(op, 0, mode, 8192, 8192, 8192)
    assert len(cands) > 2 and len({tuple(sorted(c.items())) for c in cands}) == len(cands)


@pytest.mark.parametrize("op", ["gemm", "syrk", "trsm", "potrf"])
@pytest.mark.parametrize("m", [64, 68, 214, 365, 1000, 8192, 30000])
def test_the_rule_is_a_candidate(op, m):
    for dtype, mode in ((0, 0), (1, 0)) + (((0, 2), (0, 3)) if op in ("trsm", "potrf") else ()):
        assert tuner.heuristic(op, dtype, mode, m, 300, m) in tuner.candidates(op, dtype, mode, m, 300, m)
