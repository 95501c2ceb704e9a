"""Refined matrix-core launches of few patterns, which run the brute kernels: the counts
around the switch give the brute policy's results bit for bit, pattern by pattern the
same as in one large launch, also behind the server with scratch for one pattern."""
import math

import numpy as np
import pytest

import emida_amd
from emida_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,IN", [(np.float32, np.uint16), (np.float64, np.uint16), (np.float64, np.float64)])
@pytest.mark.parametrize("size,cross", [((16, 16), (31, 31)), ((32, 32), (63, 63)), ((64, 40), (99, 41)),
                                        ((128, 128), (255, 255))])
def test_counts_around_the_switch(T, IN, size, cross):
    last = int(128 / math.sqrt(size[0] * size[1])) + (T == np.float32)
    n = last + 2
    ps = synth.PatternSet("direct", 256, n, t_range=2.0)
    begins = [(5, 9), (256 - size[0], 256 - size[1]), (61, 33)]
    dt = np.float32 if T == np.float32 else np.float64

    def outs(policy):
        res = {}
        with emida_amd.GpuOffset(T, IN, ps.size, begins, size, cross, n, policy, 5) as g:
            g.allocate_memory(ps.ref.astype(IN))
            pics = emida_amd.DeviceBuffer.from_array(ps.pics.astype(IN))
            for m in (n, last + 1, last, 1):
                b = [emida_amd.DeviceBuffer(k * m * len(begins)) for k in (2 * dt().itemsize, 25 * dt().itemsize, 16, 48)]
                g.process_device(pics, m, *b)
                emida_amd.synchronize()
                mx = b[0].download(emida_amd.data_index_dtype(dt))  # its padding bytes are not written
                res[m] = [mx["data"], mx["index"], b[1].download(dt), b[2].download(np.float64), b[3].download(np.float64)]
        return res

    got, exp = outs(emida_amd.CROSS_POLICY_BRUTE_MFMA), outs(emida_amd.CROSS_POLICY_BRUTE)
    for m in got:
        for a, b, whole in zip(got[m], exp[m], exp[n]):
            np.testing.assert_array_equal(a, b)
        # offsets of the first patterns do not depend on the launch they are in
        np.testing.assert_array_equal(got[m][3], exp[n][3][:len(got[m][3])])


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("max_batch", [1, 6])
def test_served(T, max_batch):
    ps = synth.PatternSet("direct", 256, 6, t_range=2.0)
    begins = synth.grid_begins(256, 4, 16)
    with emida_amd.GpuOffset(T, np.uint16, ps.size, begins, (32, 32), (63, 63), 6, emida_amd.CROSS_POLICY_BRUTE, 5) as g:
        g.allocate_memory(ps.ref)
        offs, coefs = g.get_offset(ps.pics)
    with emida_amd.Server(max_batch=max_batch, streams=2) as srv:
        pid = srv.add_plan(T, ps.ref, begins, (32, 32), None, emida_amd.CROSS_POLICY_BRUTE_MFMA, 5)
        reqs = [srv.submit(pid, p) for p in ps.pics]
        for i, (rid, o, c) in enumerate(reqs):
            srv.wait(rid)
            np.testing.assert_array_equal(o, offs[16 * i:16 * (i + 1)])
            np.testing.assert_array_equal(c, coefs[16 * i:16 * (i + 1)])
