"""The autotuner's cases: each has candidates that are different launches."""
from fringe_amd import _lib, autotune


def test_no_case_where_the_schedule_chooses_nothing():
    for n, _, prec in autotune.SOLVE_CASES:
        assert not autotune.matrix_cores_only(n, prec)
    for n, prec in autotune.LAYOUT_CASES:
        assert not autotune.matrix_cores_only(n, prec)
    assert autotune.matrix_cores_only(32, "fp64") and not autotune.matrix_cores_only(33, "fp64")
    assert [autotune.matrix_cores_only(n, "mixed") for n in (32, 33, 48, 49, 64, 65)] == [True, False, False, True, True,
                                                                                          False]


def test_gram_candidates():
    assert set(autotune.GRAM_CANDIDATES) == set(_lib.GRAM_VARIANTS) - {"staged12"}
