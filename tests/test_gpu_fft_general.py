"""The general FFT path (non-square slices, large sides): every transform length per axis,
odd and one-off sides, launches of few and of many slices, against numpy's double FFT."""
import numpy as np
import pytest

import emida_amd
from emida_amd import kernels as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIDES = [(2, 3), (5, 2), (3, 9), (8, 5), (16, 17), (24, 10), (17, 33), (48, 25), (33, 64), (64, 48), (65, 12), (96, 97),
         (97, 60), (128, 66), (40, 129), (160, 192), (193, 20), (256, 200), (31, 256)]


def _circular(p, r):
    """(2s)^2 circular correlation, unnormalised as the reference's C2R."""
    sy, sx = p.shape[-2:]
    c = np.fft.irfft2(np.fft.rfft2(p, (2 * sy, 2 * sx)) * np.conj(np.fft.rfft2(r, (2 * sy, 2 * sx))), (2 * sy, 2 * sx))
    return c * (4.0 * sx * sy)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("size", SIDES + [(96, 96), (160, 160)])
def test_correlation_buffers(dt, size):
    sx, sy = size
    rng = np.random.default_rng(sx * 1000 + sy)
    p, r = (rng.standard_normal((n, sy, sx)).astype(dt) for n in (6, 2))
    got = K.run_cross_corr_fft(p.ravel(), r.ravel(), size, 2, 3).reshape(3, 2, 2 * sy, 2 * sx)
    exp = _circular(p.astype(float).reshape(3, 2, sy, sx), r.astype(float))
    top = np.abs(exp).max(axis=(2, 3), keepdims=True)
    tol = 1e-12 if dt == np.float64 else 3e-6 * np.log2(2 * max(size))
    assert (np.abs(got - exp) / top).max() < tol


@pytest.mark.parametrize("dt,tol", [(np.float64, 1e-11), (np.float32, 3e-5)])
@pytest.mark.parametrize("size", SIDES)
@pytest.mark.parametrize("k,n", [(2, 1), (3, 40)])
def test_pipeline(dt, tol, size, k, n):
    """Arg-max, neighbourhood and offsets of the whole path; the largest value must be the
    oracle correlation's up to rounding, and everything else follows from its place."""
    sx, sy = size
    fit = 3
    rng = np.random.default_rng(sx + 7 * sy)
    w, h = 2 * sx + 9, 2 * sy + 5
    ref = rng.integers(0, 60000, (h, w)).astype(np.uint16)
    pics = np.stack([np.roll(ref, (i % 2, -(i % 3 % 2)), (0, 1)) for i in range(n)])
    begins = [(int(x), int(y)) for y in np.linspace(0, h - sy, k) for x in np.linspace(0, w - sx, k)]
    nb = len(begins)
    with emida_amd.GpuOffset(dt, np.uint16, (w, h), begins, size, (2 * sx - 1, 2 * sy - 1), n,
                             emida_amd.CROSS_POLICY_FFT, fit) as g:
        g.allocate_memory(ref)
        m, nbh = g.new_result_buffers()
        g.get_offset_core(m, nbh, g.transfer_pic_to_device_async(pics))
        offs, coefs = g.finalize(m, nbh)
        m, nbh = m.copy(), nbh.reshape(n * nb, fit, fit).copy()
    hx, hy = O.hann(sx), O.hann(sy)
    few = pics[:2]
    cut = lambda a: O.prepare(a.ravel(), hx, hy, O.sums(a.ravel(), begins, (w, h), size, len(a) if a.ndim == 3 else 1),
                              begins, (w, h), size, None, len(a) if a.ndim == 3 else 1)
    exp = _circular(cut(few).reshape(-1, nb, sy, sx), cut(ref).reshape(nb, sy, sx)).reshape(-1, 2 * sy, 2 * sx)
    scale = np.abs(exp).max(axis=(1, 2))
    for i in range(len(exp)):
        at = int(m["index"][i])
        y, x = divmod(at, 2 * sx)
        if scale[i] > 0:
            assert abs(m["data"][i] - exp[i].max()) < tol * scale[i]
            assert abs(exp[i, y, x] - exp[i].max()) < tol * scale[i]
        dx, dy = (x + sx) % (2 * sx) - sx, (y + sy) % (2 * sy) - sy
        if abs(dx) + 1 < sx and abs(dy) + 1 < sy:
            hood = exp[i][np.ix_(np.arange(dy - 1, dy + 2) % (2 * sy), np.arange(dx - 1, dx + 2) % (2 * sx))]
            assert np.abs(nbh[i] - hood).max() <= tol * scale[i]
            assert nbh[i, 1, 1] == m["data"][i]
    # patterns repeat with period 6: so do the results, wherever they lie in the launch
    for i in range(6, n):
        np.testing.assert_array_equal(m["index"][i * nb:(i + 1) * nb], m["index"][(i - 6) * nb:(i - 5) * nb])
        np.testing.assert_array_equal(nbh[i * nb:(i + 1) * nb], nbh[(i - 6) * nb:(i - 5) * nb])
        np.testing.assert_array_equal(offs[i * nb:(i + 1) * nb], offs[(i - 6) * nb:(i - 5) * nb])
