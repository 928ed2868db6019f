"""The noise estimate and the thresholding keep to parts of their own of the workspace that they share.

An estimate of one stack on one stream and a thresholding of another on a second stream may use one workspace,
so the thresholding must not write where the estimate keeps its scratch.
"""

import numpy as np
import pytest
import torch

from pymoresane_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("s,h,w", [(1, 8, 8), (3, 200, 210), (5, 513, 500)])
def test_thresholding_leaves_the_estimates_scratch_alone(hip, s, h, w):
    print("threshold workspace %d x %dx%d" % (s, h, w), flush=True)
    lib = _lib.lib()
    x = torch.from_numpy(np.random.default_rng(h).standard_normal((s, h, w)).astype(np.float32)).cuda()
    thr, out = torch.ones(s, dtype=torch.float64, device="cuda"), torch.empty_like(x)
    total = lib.pms_threshold_work_bytes(s, h, w)
    maxima = s * 256 * 4  # one float for each block of a plane's thresholding, at most 256
    work = torch.full((total,), 0x5a, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    _lib.check(lib.pms_apply_threshold(x.data_ptr(), s, h, w, thr.data_ptr(), 1.0, out.data_ptr(), work.data_ptr(), None))
    torch.cuda.synchronize()
    assert torch.equal(out, torch.where(x.abs() > 1.0, x, torch.zeros_like(x)))
    assert bool((work[: total - maxima] == 0x5a).all())
    assert not bool((work[total - maxima:] == 0x5a).all())
