"""get_offset with other pixels in every call on one handle: each call's results are those of
its own pixels, of every part of them, also where calls of two handles take turns."""
import numpy as np
import pytest

import emida_amd

pytestmark = pytest.mark.gpu


def _handle(size, n, begins):
    return emida_amd.GpuOffset(np.float32, np.uint16, size, begins, (32, 32), (63, 63), n, emida_amd.CROSS_POLICY_FFT, 3)


# staged by one thread (180 KB), by several (1.5 MB, 6 MB), not staged (9.4 MB)
@pytest.mark.parametrize("side,n", [(300, 1), (873, 1), (1000, 3), (1250, 3)])
def test_pixels_of_each_call(side, n):
    rng = np.random.default_rng(side)
    ref = rng.integers(0, 60000, (side, side)).astype(np.uint16)
    # ROIs over the whole picture: a stale part shows in the ROIs that lie in it
    at = np.linspace(0, side - 32, 12).astype(int)
    begins = [(int(x), int(y)) for y in at for x in at]
    calls = []
    for i in range(6):
        calls.append(np.stack([np.roll(ref, (i - 3, j - 1), (0, 1)) for j in range(n)]))
    with _handle((side, side), n, begins) as a, _handle((side, side), n, begins) as b:
        a.allocate_memory(ref)
        b.allocate_memory(ref)
        dev = emida_amd.DeviceBuffer
        out = [dev(n * len(begins) * k) for k in (8, 36, 16, 48)]
        exp = []
        for pics in calls:
            a.process_device(dev.from_array(pics), n, *out)
            emida_amd.synchronize()
            exp.append(out[2].download(np.float64).reshape(-1, 2))
        assert all((exp[i] != exp[j]).any() for i in range(6) for j in range(i))
        for g in (a, b, a):
            for pics, e in zip(calls, exp):
                np.testing.assert_array_equal(g.get_offset(pics)[0], e)
        for pics, e in zip(calls, exp):  # taking turns
            np.testing.assert_array_equal(a.get_offset(pics)[0], e)
            np.testing.assert_array_equal(b.get_offset(calls[0])[0], exp[0])
