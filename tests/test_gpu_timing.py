"""The kernel names of get_timing: those of the launches that were timed."""
import numpy as np
import pytest

import emida_amd
from emida_amd import synth

pytestmark = pytest.mark.gpu

GENERAL = "fftg_rows_kernel+fftg_cols_kernel+fftg_rows_inv_kernel+fftg_peak_kernel"


# refined matrix-core launches of up to 4 patterns of 32 x 32 in double run the brute kernel
@pytest.mark.parametrize("T,policy,size,counts,name", [
    (np.float32, emida_amd.CROSS_POLICY_FFT, (32, 32), (8, 1), "fft_kernel"),
    (np.float32, emida_amd.CROSS_POLICY_FFT, (80, 80), (8, 1), "fft256_kernel"),
    (np.float32, emida_amd.CROSS_POLICY_FFT, (40, 24), (8, 1), GENERAL),
    (np.float64, emida_amd.CROSS_POLICY_BRUTE, (32, 32), (8, 1), "cross_corr_mm_kernel"),
    (np.float64, emida_amd.CROSS_POLICY_BRUTE_MFMA, (32, 32), (8,), "mfma_corr_kernel"),
    (np.float64, emida_amd.CROSS_POLICY_BRUTE_MFMA, (32, 32), (1, 4), "cross_corr_mm_kernel"),
    (np.float64, emida_amd.CROSS_POLICY_BRUTE_MFMA, (32, 32), (8, 2, 5), "mfma_corr_kernel+cross_corr_mm_kernel"),
])
def test_names_are_those_of_the_launches(T, policy, size, counts, name):
    ps = synth.PatternSet("timing", 256, 8, t_range=2.0)
    begins = [(3, 4), (100, 90)]
    with emida_amd.GpuOffset(T, np.uint16, ps.size, begins, size, (2 * size[0] - 1, 2 * size[1] - 1), 8, policy, 3) as g:
        g.allocate_memory(ps.ref)
        pics = emida_amd.DeviceBuffer.from_array(ps.pics)
        res = [emida_amd.DeviceBuffer(n * 16) for n in (16, 72, 16, 48)]
        g.set_timing(True)
        for n in counts:
            g.process_device(pics, n, *res)
        g.set_timing(False)
        g.process_device(pics, 3, *res)
        emida_amd.synchronize()
        got, ms, launches = g.get_timing()
        assert (got, launches) == (name, len(counts)) and ms > 0
