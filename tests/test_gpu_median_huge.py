"""The noise estimate of a plane of more than 2^32 pixels of which the interior mask leaves fewer.

Sixty per cent of the rows hold 3 and the others 1, the sign alternating: the median of the absolute values is 3.
"""

import numpy as np
import pytest
import torch

from pymoresane_amd import _lib

pytestmark = pytest.mark.gpu


def test_median_of_more_than_2_to_the_32_pixels(hip):
    n, excl = 65537, 1000
    assert n * n >= 2 ** 32 > n * n - (2 * excl) ** 2
    print("median of a %d^2 plane" % n, flush=True)
    lib = _lib.lib()
    x = torch.empty((n, n), device="cuda")
    x[: n * 2 // 5] = 1.0
    x[n * 2 // 5:] = 3.0
    x[::2] *= -1
    thr = torch.zeros(1, dtype=torch.float64, device="cuda")
    work = torch.empty(lib.pms_threshold_work_bytes(1, n, n), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    _lib.check(lib.pms_estimate_threshold(x.data_ptr(), 1, n, n, 0, excl, thr.data_ptr(), work.data_ptr(), None))
    torch.cuda.synchronize()
    assert thr.item() == np.float64(3.0) / 0.6745
