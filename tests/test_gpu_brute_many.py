"""Brute correlation of more slices than one grid of 2^32 threads has workgroups for."""
import numpy as np
import pytest

from emida_amd import kernels as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def test_more_slices_than_one_grid():
    size, res, n = (2, 2), (3, 3), (1 << 24) + 5
    rng = np.random.default_rng(4)
    pics, ref = rng.standard_normal(4 * n, dtype=np.float32), rng.standard_normal(4, dtype=np.float32)
    got = K.run_cross_corr(pics, ref, size, res, 1, n).reshape(n, 9)
    for first in (0, (1 << 24) - 8, n - 8):
        part = pics[4 * first:4 * (first + 8)]
        np.testing.assert_array_equal(got[first:first + 8].ravel(), O.cross_corr(part, ref, size, res, 1, 8))
    # every slice: the value at shift 0, a sum of four products, each side rounding four times
    p = pics.reshape(n, 4)
    assert (np.abs(got[:, 4] - p @ ref) <= 8 * 2.0**-24 * (np.abs(p) @ np.abs(ref))).all()
