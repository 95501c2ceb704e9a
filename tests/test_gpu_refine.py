"""Exact refinement of the matrix-core policy against the brute policy, bit for bit: one
and four waves per slice, every slice-width class, peaks in one box, at the window's edge
and spread over several boxes, and swept slices."""
import numpy as np
import pytest

import emida_amd
from emida_amd import synth

pytestmark = pytest.mark.gpu


def _run(policy, T, ref, pics, begins, size, cross, fit):
    n, h, w = pics.shape
    with emida_amd.GpuOffset(T, np.uint16, (w, h), begins, size, cross, n, policy, fit) as g:
        g.allocate_memory(ref)
        m, nb = g.new_result_buffers()
        i = g.transfer_pic_to_device_async(pics)
        g.get_offset_core(m, nb, i)
        offs, coefs = g.finalize(m, nb)
        return m["data"].copy(), m["index"].copy(), nb.copy(), offs, coefs


def _pictures(kind, n, rng):
    if kind == "bands":
        ps = synth.PatternSet("refine", 256, n, t_range=3.0)
        return ps.ref, ps.pics
    if kind == "noise":  # no common content: several spread candidates
        return (rng.integers(0, 4000, (256, 256)).astype(np.uint16),
                rng.integers(0, 4000, (n, 256, 256)).astype(np.uint16))
    if kind == "blob":  # a broad blob against single pixels: flat screens, swept slices
        y, x = np.mgrid[0:256, 0:256]
        ref = (30000 * np.exp(-((x - 128.0) ** 2 + (y - 128.0) ** 2) / 2e4)).astype(np.uint16)
        pics = np.full((n, 256, 256), 100, np.uint16)
        pics[:, ::40, ::40] = 60000
        return ref, pics
    ref = rng.integers(0, 4000, (256, 256)).astype(np.uint16)  # "edge": peaks on the window's border
    return ref, np.stack([np.roll(ref, (9 * (i % 3 - 1), 7 * (i % 2 * 2 - 1)), (0, 1)) for i in range(n)])


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("size,cross,k,n", [
    ((8, 5), (15, 9), 3, 2),
    ((32, 32), (63, 63), 5, 40),    # 1,000 slices: one wave each
    ((32, 32), (19, 15), 3, 2),     # four waves each
    ((40, 24), (79, 47), 4, 3),
    ((64, 64), (127, 127), 3, 9),
    ((72, 33), (143, 65), 2, 3),
    ((128, 128), (255, 255), 2, 2),
])
@pytest.mark.parametrize("kind", ["bands", "noise", "edge", "blob"])
def test_refined_equals_brute(T, size, cross, k, n, kind):
    ref, pics = _pictures(kind, n, np.random.default_rng(8))
    xs = np.linspace(0, 256 - size[0], k).astype(int)
    ys = np.linspace(0, 256 - size[1], k).astype(int)
    begins = [(int(x), int(y)) for y in ys for x in xs]
    got = _run(emida_amd.CROSS_POLICY_BRUTE_MFMA, T, ref, pics, begins, size, cross, 5)
    exp = _run(emida_amd.CROSS_POLICY_BRUTE, T, ref, pics, begins, size, cross, 5)
    for a, b in zip(got, exp):
        np.testing.assert_array_equal(a, b)
