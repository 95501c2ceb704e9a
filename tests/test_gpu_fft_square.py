"""The single-kernel FFT paths: every transform length, its smallest and largest slice side,
odd sides, one slice and several, against numpy's double FFT."""
import numpy as np
import pytest

from emida_amd import kernels as K

pytestmark = pytest.mark.gpu

F64 = [2, 3, 4, 5, 8, 9, 15, 16, 17, 31, 32, 33, 50, 63, 64]


@pytest.mark.parametrize("dt,side", [(np.float64, s) for s in F64] + [(np.float32, s) for s in F64 + [65, 97, 127, 128]])
@pytest.mark.parametrize("n", [1, 5])
def test_correlation_buffers(dt, side, n):
    rng = np.random.default_rng(side * 10 + n)
    p, r = (rng.standard_normal((m, side, side)).astype(dt) for m in (2 * n, 2))
    got = K.run_cross_corr_fft(p.ravel(), r.ravel(), (side, side), 2, n).reshape(n, 2, 2 * side, 2 * side)
    full = (2 * side, 2 * side)
    spec = np.fft.rfft2(p.astype(float).reshape(n, 2, side, side), full) * np.conj(np.fft.rfft2(r.astype(float), full))
    exp = np.fft.irfft2(spec, full) * (4.0 * side * side)
    # each of the 3 log2(2 side) + 1 passes rounds its values to half an ulp, the pads add none:
    # errors sum to well below eps times the passes of both axes, against the largest value
    passes = 6 * np.log2(4 * side) + 2
    err = np.abs(got - exp).max(axis=(2, 3)) / np.abs(exp).max(axis=(2, 3))
    assert err.max() < np.finfo(dt).eps * passes * (4 if dt == np.float64 else 1)
