"""Slice sums where a thread's number of loads changes (1, 2, 4 and 10 pixels, one group of
10,240 pixels and more), in the reference's order: bit for bit against the oracle."""
import numpy as np
import pytest

from emida_amd import kernels as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("IN", [np.uint16, np.float32, np.float64])
@pytest.mark.parametrize("size", [(2, 2), (32, 32), (41, 25), (64, 32), (683, 3), (64, 64), (241, 17), (128, 80), (209, 49),
                                  (128, 160), (1217, 17), (256, 256)])
def test_sums(IN, size):
    rng = np.random.default_rng(size[0])
    src = (size[0] + 7, size[1] + 5)
    begins = [(0, 0), (7, 5), (3, 1)]
    pics = (rng.integers(0, 60000, (2, src[1], src[0])) if IN == np.uint16
            else rng.standard_normal((2, src[1], src[0])) * 1000).astype(IN)
    got = K.run_sum(pics.ravel(), begins, src, size, 2)
    np.testing.assert_array_equal(got, O.sums(pics.ravel(), begins, src, size, 2))
