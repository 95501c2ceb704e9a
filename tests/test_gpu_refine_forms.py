"""Exact refinement of the matrix-core policy against the brute policy, bit for bit, in
launches of more patterns than run the brute kernels themselves: one and four waves per
slice, every slice-width class and widths between, peaks in one box, on the window's border
(the neighbourhood's clamp leaves the window) and spread over two or many boxes, flat
screens that are swept, and every mode of the screen."""
import math

import numpy as np
import pytest

import emida_amd
from emida_amd import synth

pytestmark = pytest.mark.gpu

MFMA, BRUTE = emida_amd.CROSS_POLICY_BRUTE_MFMA, emida_amd.CROSS_POLICY_BRUTE


def _refined(T, size, n):
    """n, which must be more than the patterns of a launch that runs the brute kernels."""
    assert n > int(128 / math.sqrt(size[0] * size[1])) + (np.dtype(T) == np.float32), (size, n)
    return n


def _run(policy, T, ref, pics, begins, size, cross, fit, mode=None):
    n, h, w = pics.shape
    with emida_amd.GpuOffset(T, np.uint16, (w, h), begins, size, cross, n, policy, fit, mfma_mode=mode) as g:
        g.allocate_memory(ref)
        m, nb = g.new_result_buffers()
        i = g.transfer_pic_to_device_async(pics)
        g.get_offset_core(m, nb, i)
        offs, coefs = g.finalize(m, nb)
        return m["data"].copy(), m["index"].copy(), nb.copy(), offs, coefs


def _same(T, ref, pics, begins, size, cross, fit, mode=None):
    got = _run(MFMA, T, ref, pics, begins, size, cross, fit, mode)
    exp = _run(BRUTE, T, ref, pics, begins, size, cross, fit)
    for a, b, what in zip(got, exp, ("values", "indices", "neighbourhoods", "offsets", "coefficients")):
        np.testing.assert_array_equal(a, b, err_msg=what)
    return exp


def _pictures(kind, n, size, rng):
    if kind == "bands":
        ps = synth.PatternSet("refine", 256, n, t_range=3.0)
        return ps.ref, ps.pics
    ref = rng.integers(0, 4000, (256, 256)).astype(np.uint16)
    if kind == "noise":  # no common content: many spread candidates
        return ref, rng.integers(0, 4000, (n, 256, 256)).astype(np.uint16)
    if kind == "two":  # the same content at two places: two peaks, nearly equal
        a, b = (np.roll(ref, (s * size[1] // 4, s * size[0] // 4), (0, 1)).astype(int) for s in (-1, 1))
        return ref, np.stack([(a + b) // 2 + rng.integers(0, 3, a.shape) for _ in range(n)]).astype(np.uint16)
    if kind == "flat":  # constant, and single pixels against a broad blob: ties and swept slices
        y, x = np.mgrid[0:256, 0:256]
        ref = (30000 * np.exp(-((x - 128.0) ** 2 + (y - 128.0) ** 2) / 2e4)).astype(np.uint16)
        pics = np.full((n, 256, 256), 100, np.uint16)
        pics[:, ::40, ::40] = 60000
        return ref, pics
    # "border": shifts of the window's reach, so that peaks lie on its border
    r = _reach(size)
    return ref, np.stack([np.roll(ref, ((i % 3 - 1) * r, (i % 2 * 2 - 1) * r), (0, 1)) for i in range(n)])


def _reach(size):
    return min(8, min(size) // 4)


def _grid(size, k):
    return [(int(x), int(y)) for y in np.linspace(0, 256 - size[1], k) for x in np.linspace(0, 256 - size[0], k)]


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("size,cross,k,n,fit", [
    ((8, 5), (15, 9), 3, 24, 3),        # 216 slices: four waves each
    ((8, 8), (15, 15), 6, 24, 5),       # 864: one wave each
    ((16, 16), (31, 31), 3, 12, 9),
    ((16, 50), (31, 99), 9, 10, 5),
    ((24, 40), (47, 79), 3, 7, 5),
    ((32, 32), (63, 63), 3, 6, 7),
    ((32, 32), (63, 63), 12, 6, 7),
    ((40, 24), (79, 47), 3, 6, 5),
    ((40, 24), (79, 47), 12, 6, 5),
    ((56, 33), (111, 65), 3, 5, 9),
    ((64, 64), (127, 127), 3, 4, 5),
    ((64, 64), (127, 127), 14, 4, 5),
    ((72, 33), (143, 65), 3, 4, 5),
    ((72, 33), (143, 65), 14, 4, 5),
    ((120, 17), (239, 33), 3, 4, 7),
    ((128, 128), (255, 255), 2, 3, 7),
])
@pytest.mark.parametrize("kind", ["bands", "noise", "two", "flat"])
def test_whole_window(T, size, cross, k, n, fit, kind):
    if kind == "flat" and k * k * n * size[0] * size[1] > 2e6:
        k = 3  # swept slices cost a whole brute window each
    rng = np.random.default_rng(8)
    ref, pics = _pictures(kind, _refined(T, size, n), size, rng)
    _same(T, ref, pics, _grid(size, k), size, cross, fit)


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("size", [(8, 24), (16, 16), (32, 32), (56, 40), (64, 64), (128, 96)])
@pytest.mark.parametrize("k", [3, 14])
def test_peaks_on_the_border(T, size, k):
    """Windows as wide as the shifts, and one narrower and wider."""
    n = _refined(T, size, int(128 / math.sqrt(size[0] * size[1])) + 2)
    ref, pics = _pictures("border", n, size, np.random.default_rng(3))
    for wider, fit in ((0, 9), (-1, 5), (1, 3)):
        cross = (2 * (_reach(size) + wider) + 1,) * 2
        index = _same(T, ref, pics, _grid(size, k), size, cross, fit)[1]
        x, y = index % cross[0], index // cross[0]
        edge = (x == 0) | (x == cross[0] - 1) | (y == 0) | (y == cross[1] - 1)
        assert wider != 0 or edge.mean() > 0.5


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("mode", [emida_amd.MFMA_BF16, emida_amd.MFMA_BF16_SPLIT, emida_amd.MFMA_F16,
                                  emida_amd.MFMA_F16_SPLIT])
def test_modes(T, mode):
    rng = np.random.default_rng(5)
    for size, n in (((128, 128), 3), ((32, 24), 7)):
        cross = (2 * size[0] - 1, 2 * size[1] - 1)
        for kind in ("noise", "flat"):
            ref, pics = _pictures(kind, _refined(T, size, n), size, rng)
            _same(T, ref, pics, _grid(size, 2), size, cross, 7, mode)
