"""Device memory of refined matrix-core objects: launches of few patterns, which run the
brute kernels, find room for their correlation buffers in the candidate lists, so nothing
is held for them beyond what a batch needs; batches too small for that hold one launch's."""
import numpy as np
import pytest

import emida_amd
from emida_amd import synth

pytestmark = pytest.mark.gpu


def _held(T, size, cross, begins, batch):
    ps = synth.PatternSet("memory", 256, 1, t_range=2.0)
    with emida_amd.GpuOffset(T, np.uint16, ps.size, begins, size, cross, batch,
                             emida_amd.CROSS_POLICY_BRUTE_MFMA, 3) as g:
        g.allocate_memory(ps.ref)
        return g.device_bytes


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("size", [(16, 16), (32, 32), (64, 40), (128, 128)])
def test_nothing_beyond_a_batch(T, size):
    begins = synth.grid_begins(256, 4, size[0])
    cross = (2 * size[0] - 1, 2 * size[1] - 1)
    b = [_held(T, size, cross, begins, n) for n in (8, 16, 32)]
    per = (b[2] - b[1]) / 16
    assert b[2] - b[1] == 2 * (b[1] - b[0])
    # what does not grow with the batch: the reference slices in half and in full precision,
    # their norms, the windows and the corners
    fixed = b[0] - 8 * per
    t = np.dtype(T).itemsize
    assert fixed <= len(begins) * (size[0] * size[1] * (2 + t) + 16) + sum(size) * (t + 4) + 64
    # a batch of one: its lists or its correlation buffers
    lists, corr = len(begins) * cross[1] * 256, len(begins) * cross[0] * cross[1] * t
    assert _held(T, size, cross, begins, 1) <= fixed + per + max(0, corr - lists) + 64
