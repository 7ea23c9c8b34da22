"""KS2's decision is a largest count: no similar count lies beyond a count that
is not similar, for every number of dates and threshold."""
import ctypes

import numpy as np
import pytest

from fringe_amd import _lib


@pytest.mark.parametrize("prob", [0.0, 1e-12, 1e-3, 0.05, 0.5, 0.9, 0.999999, 1.0, 1.5, float("nan")])
def test_ks_table_is_a_prefix(prob):
    L = _lib.lib()
    for n in range(1, 129):
        t = (ctypes.c_uint8 * (n + 1))()
        L.fringe_ks_table(n, prob, t)
        assert np.all(np.diff(np.array(t, dtype=int)) <= 0), n
