"""The deformation post-step at the ROI counts where its kernel changes form (lanes and
waves per pattern), with ties in the median, and where the inverse iteration gives way to
the Jacobi rotations, against the numpy restatement (oracle/post.py)."""
import ctypes

import numpy as np
import pytest

from emida_amd import _capi as C
from emida_amd import post as G
from emida_amd.gpu_offset import DeviceBuffer
from oracle import post as P

pytestmark = pytest.mark.gpu
CALIB = np.array([436.0, 436.0, 436.0])


def _data(n, n_pat, seed, ties=False):
    rng = np.random.default_rng(seed)
    mids = rng.uniform(32, 841, (n, 2)).round()
    offs, coefs = np.empty((n_pat, n, 2)), rng.normal(0, 1, (n_pat, n, 6))
    coefs[..., 3], coefs[..., 5] = -rng.uniform(0.5, 2.0, (2, n_pat, n))
    if ties:
        coefs[..., 3:] = coefs[..., 3:].round(1)
    for p in range(n_pat):
        Ft = np.eye(3) + rng.normal(0, 2e-3, (3, 3))
        offs[p] = P.apply_transform(Ft, mids, CALIB) + rng.normal(0, 0.02, (n, 2)) - mids
    return mids, offs, coefs


def _check(res, mids, offs, coefs):
    data = [np.column_stack([mids, offs[i], coefs[i]]) for i in range(len(offs))]
    mask, quality, H, F, eps, omega = P.post_process(data, CALIB)
    np.testing.assert_array_equal(res["mask"], mask)
    np.testing.assert_array_equal(res["quality"], quality)
    for name, exp in (("H", H), ("F", F), ("epsilon", eps), ("omega", omega)):
        assert np.abs(res[name][mask] - exp[mask]).max() < 1e-9, name


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("n", [30, 64, 65, 128, 129, 256, 257, 448, 449, 1024, 1025, 2048, 2049, 8192])
def test_fit_at_kernel_sizes(n, ties):
    mids, offs, coefs = _data(n, 5 if n < 2000 else 2, n, ties)
    _check(G.fit_deformation(mids, offs, coefs, CALIB), mids, offs, coefs)


def test_pointers_off_sixteen_bytes():
    """Inputs and outputs at any multiple of 8 bytes."""
    mids, offs, coefs = _data(100, 3, 1)
    ins = [DeviceBuffer(a.nbytes + 8) for a in (mids, offs, coefs)]
    for b, a in zip(ins, (mids, offs, coefs)):
        b.upload(a.ravel(), 8)
    names = ("quality", "H", "F", "epsilon", "omega")
    outs = {k: DeviceBuffer(8 + 3 * (8 if k == "quality" else 72)) for k in names}
    mask = DeviceBuffer(12)
    at = lambda b: ctypes.c_void_p(b.ptr.value + 8)
    C.check(C.lib().emida_fit_deformation(at(ins[0]), 0, 100, at(ins[1]), at(ins[2]), 3, C.Calib(*CALIB), 1e-6, 10,
                                          mask.ptr, *(at(outs[k]) for k in names), None))
    res = {k: b.download(np.float64, offset=8).reshape((3,) if k == "quality" else (3, 3, 3)) for k, b in outs.items()}
    res["mask"] = mask.download(np.int32).astype(bool)
    _check(res, mids, offs, coefs)


def test_without_inverse_iteration():
    """Noise as large as the pattern (slow convergence) and NaN offsets."""
    rng = np.random.default_rng(2)
    mids, offs, coefs = _data(60, 4, 3)
    offs += rng.normal(0, 300, offs.shape)
    _check(G.fit_deformation(mids, offs, coefs, CALIB), mids, offs, coefs)
    offs[1] = np.nan
    res = G.fit_deformation(mids, offs, coefs, CALIB)
    assert res["mask"].all() and np.isfinite(res["F"][0]).all() and not np.isfinite(res["F"][1]).all()
