"""Brute correlation of small slices, which take one thread per shift or one wave per slice,
and of the sizes next to theirs: bit for bit against the oracle's chain of fused operations,
one slice and many, infinities and NaN only in the shifts whose overlap holds them."""
import numpy as np
import pytest

from emida_amd import kernels as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(1, 48), (1, 49), (48, 1), (49, 1), (2, 2), (6, 8), (7, 7), (8, 8), (24, 8), (16, 16), (16, 17), (17, 16),
         (32, 8), (33, 8), (60, 4), (120, 2), (10, 10)]


def _windows(size):
    full = (2 * size[0] - 1, 2 * size[1] - 1)
    return {full, (min(9, full[0]), min(9, full[1])), (2 * size[0] + 1, 1), (1, 2 * size[1] + 1),
            (min(34, full[0]), min(16, full[1]))}


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("ref_slices,batch", [(1, 1), (3, 70)])
def test_bitexact(dt, size, ref_slices, batch):
    rng = np.random.default_rng(size[0] * 100 + size[1])
    n = size[0] * size[1]
    pics = rng.standard_normal(n * ref_slices * batch).astype(dt)
    ref = rng.standard_normal(n * ref_slices).astype(dt)
    for res in sorted(_windows(size)):
        got = K.run_cross_corr(pics, ref, size, res, ref_slices, batch)
        np.testing.assert_array_equal(got, O.cross_corr(pics, ref, size, res, ref_slices, batch), err_msg=str(res))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("size", [(6, 8), (8, 8), (24, 8), (16, 16)])
@pytest.mark.parametrize("where", ["pattern", "reference"])
def test_not_finite(dt, size, where):
    rng = np.random.default_rng(6)
    n = size[0] * size[1]
    pics, ref = rng.standard_normal(2 * n).astype(dt), rng.standard_normal(n).astype(dt)
    a = pics if where == "pattern" else ref
    a[1], a[n - 2] = np.inf, np.nan
    res = (2 * size[0] - 1, 2 * size[1] - 1)
    got, exp = K.run_cross_corr(pics, ref, size, res, 1, 2), O.cross_corr(pics, ref, size, res, 1, 2)
    assert np.isfinite(exp).any() and not np.isfinite(exp).all()
    np.testing.assert_array_equal(got, exp)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("size", [(7, 7), (10, 10), (12, 12), (16, 16), (24, 8), (17, 16), (60, 4), (100, 2)])
def test_two_slices_for_every_cu(dt, size):
    """From 512 slices on small ones of several tiles take one wave to a workgroup."""
    for n in (511, 515):
        rng = np.random.default_rng(n)
        pics = rng.standard_normal(size[0] * size[1] * n).astype(dt)
        ref = rng.standard_normal(size[0] * size[1]).astype(dt)
        res = (2 * size[0] - 1, 2 * size[1] - 1)
        np.testing.assert_array_equal(K.run_cross_corr(pics, ref, size, res, 1, n),
                                      O.cross_corr(pics, ref, size, res, 1, n))
