"""Thresholding where its kernels change: planes read four values at a time or one by one, outputs within the
last-level cache or past it, values on the threshold, infinities and NaN.  Values are kept or set to zero, so
the result equals numpy's bit for bit."""

import numpy as np
import pytest

from pymoresane_amd import iuwt_toolbox as tools

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 3), (3, 2, 2), (2, 6, 10), (3, 5, 7), (4, 63, 65), (2, 64, 64),
                                   (5, 250, 254), (3, 1021, 1024), (5, 3700, 3700), (2, 6001, 6001)])
def test_threshold_keeps_or_zeroes(hip, shape):
    print("threshold of %s" % (shape,), flush=True)
    rng = np.random.default_rng(shape[1])
    x = rng.standard_normal(shape).astype(np.float32)
    thr = np.linspace(0.25, 0.5, shape[0])
    flat = x.reshape(shape[0], -1)
    flat[0, 0] = 4 * thr[0]  # on the threshold: not above it
    flat[-1, -1] = np.inf
    if flat.shape[1] > 2:
        flat[0, 1], flat[-1, -2] = np.nan, -np.inf
    got = tools.apply_threshold(x, thr, 4)
    want = np.where(np.abs(x.astype(np.float64)) > 4 * thr[:, None, None], x, np.float32(0))
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
