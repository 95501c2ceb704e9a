"""Brute correlation on the matrix cores at the edges of its tiles, bit for bit against
the oracle's fma chain (float and double)."""
import numpy as np
import pytest

from emida_amd import kernels as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# slice widths around the tile widths (16, 32, 48) and their multiples, windows on one and
# on both sides of a tile, windows past the slice, one to several row chunks
@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("size,res,ref_slices,batch", [
    ((1, 1), (3, 3), 1, 1),
    ((3, 40), (7, 81), 2, 1),
    ((15, 17), (29, 33), 1, 2),
    ((16, 16), (33, 31), 3, 1),
    ((17, 15), (16, 2), 2, 2),
    ((31, 33), (61, 34), 1, 1),
    ((33, 31), (35, 61), 2, 1),
    ((47, 20), (95, 17), 1, 1),
    ((49, 9), (49, 19), 1, 1),
    ((75, 61), (41, 33), 2, 3),
    ((96, 7), (191, 13), 1, 2),
    ((129, 65), (257, 49), 1, 1),
    ((300, 12), (101, 23), 1, 1),
    ((128, 128), (255, 255), 2, 1),
])
def test_matrix_core_brute_bitexact(dt, size, res, ref_slices, batch):
    rng = np.random.default_rng(31)
    n = size[0] * size[1]
    pics = rng.standard_normal(n * ref_slices * batch).astype(dt)
    ref = rng.standard_normal(n * ref_slices).astype(dt)
    got = K.run_cross_corr(pics, ref, size, res, ref_slices, batch)
    np.testing.assert_array_equal(got, O.cross_corr(pics, ref, size, res, ref_slices, batch))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_matrix_core_brute_range_of_values(dt):
    """Subnormal products and sums, and values far apart, keep the chain's bits."""
    rng = np.random.default_rng(5)
    size, res = (37, 21), (73, 41)
    lo = np.finfo(dt).minexp // 2
    for e0, e1 in ((lo - 8, lo + 4), (-60, 60)):
        v = [np.ldexp(rng.standard_normal(37 * 21), rng.integers(e0, e1, 37 * 21)).astype(dt) for _ in range(2)]
        np.testing.assert_array_equal(K.run_cross_corr(v[0], v[1], size, res), O.cross_corr(v[0], v[1], size, res, 1, 1))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("where", ["pattern", "reference"])
def test_matrix_core_brute_not_finite(dt, where):
    """Infinities and NaN reach the shifts whose overlap holds them and no others, and the
    other slices of the launch not at all."""
    rng = np.random.default_rng(6)
    size, res, n = (40, 24), (79, 47), 40 * 24
    pics, ref = rng.standard_normal(2 * n).astype(dt), rng.standard_normal(n).astype(dt)
    a = pics if where == "pattern" else ref
    a[3], a[n - 5] = np.inf, np.nan
    got = K.run_cross_corr(pics, ref, size, res, 1, 2)
    exp = O.cross_corr(pics, ref, size, res, 1, 2)
    assert np.isfinite(exp).any() and not np.isfinite(exp).all()
    np.testing.assert_array_equal(got, exp)
