"""get_offset from host memory: pictures below and above the size that is copied by several
threads, byte counts that are no multiple of 16, batches above the staging, unaligned and
pinned memory and several handles at a time give the device pass's results bit for bit."""
import threading

import numpy as np
import pytest

import emida_amd
from emida_amd.gpu_offset import PinnedBuffer

pytestmark = pytest.mark.gpu


def _handle(size, IN, n):
    T = np.float64 if IN == np.float64 else np.float32
    return emida_amd.GpuOffset(T, IN, size, [(3, 2), (size[0] - 36, size[1] - 40)], (32, 32), (63, 63), n,
                               emida_amd.CROSS_POLICY_FFT, 3)


def _pics(size, IN, n):
    rng = np.random.default_rng(size[0] + n)
    ref = rng.integers(0, 60000, size[::-1]).astype(IN)
    pics = np.stack([np.roll(ref, (1, i % 3), (0, 1)) for i in range(n)])
    return ref, pics + rng.integers(0, 500, pics.shape).astype(IN)


def _device(g, pics, n):
    b = [emida_amd.DeviceBuffer(2 * n * k) for k in (16, 72, 16, 48)]
    g.process_device(emida_amd.DeviceBuffer.from_array(pics), n, *b)
    emida_amd.synchronize()
    return b[2].download(np.float64).reshape(-1, 2), b[3].download(np.float64).reshape(-1, 6)


# by one thread: 15,138 and 524,262 bytes; by several from 524,288, tails of 0, 2, 14 and 8
# bytes; 8,388,608: the last that is staged; 8,396,800: the first that is not
@pytest.mark.parametrize("size,IN,n", [((87, 87), np.uint16, 1), ((87, 3013), np.uint16, 1), ((512, 512), np.uint16, 1),
                                       ((113, 2321), np.uint16, 1), ((113, 2327), np.uint16, 1), ((181, 207), np.float64, 3),
                                       ((1024, 1024), np.float32, 2), ((1025, 1024), np.float32, 2)])
def test_same_as_device(size, IN, n):
    ref, pics = _pics(size, IN, n)
    with _handle(size, IN, n) as g:
        g.allocate_memory(ref)
        exp = _device(g, pics, n)
        pinned = PinnedBuffer(pics.size, IN)
        pinned.array[:] = pics.ravel()
        raw = np.zeros(pics.nbytes + 64, np.uint8)
        at = -raw.ctypes.data % 16 + pics.itemsize  # off the 16-byte grid
        odd = raw[at:at + pics.nbytes].view(IN)
        odd[:] = pics.ravel()
        for src in (pics, pinned.array, odd, pics):
            for a, b in zip(g.get_offset(src), exp):
                np.testing.assert_array_equal(a, b)


def test_handles_in_threads():
    ref, pics = _pics((700, 640), np.uint16, 6)
    exp, got = [None] * 6, [None] * 6

    def work(i, out):
        with _handle((700, 640), np.uint16, 1) as g:
            g.allocate_memory(ref)
            for _ in range(8):
                out[i] = g.get_offset(pics[i])

    for i in range(6):
        work(i, exp)
    ts = [threading.Thread(target=work, args=(i, got)) for i in range(6)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for a, b in zip(got, exp):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y)
