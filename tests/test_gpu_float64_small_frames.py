"""Float64 cleans whose FFT frame is 4 or 8, the smallest there are.

Images of 4 in both modes and of 8 in the circular one, and subregions of those sides.  The device path
and the oracle both compute in float64; the models and residuals are float32, whose rounding (2^-24 of a
value) the bound of 1e-7 allows for, as in the larger float64 cleans' tests.
"""

import numpy as np
import pytest

from oracle import moresane64 as omain
from pymoresane_amd import synth
from pymoresane_amd.main import DataImage

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b))


@pytest.mark.parametrize("n,mode,subregion", [(4, "linear", None), (4, "circular", None), (8, "circular", None),
                                              (16, "linear", 4), (16, "circular", 4), (16, "circular", 8)])
def test_float64_clean_of_the_smallest_frames(hip, n, mode, subregion):
    print("float64 %d^2 %s subregion %s" % (n, mode, subregion), flush=True)
    rng = np.random.default_rng(n)
    psf = synth.make_gaussian_psf(2 * n if mode == "linear" else n, 1.5)
    g = np.exp(-0.5 * ((np.arange(n) - n // 2) / synth.fwhm_to_sigma(1.5)) ** 2)
    dirty = (np.outer(g, g) + rng.normal(0.0, 1e-3, (n, n))).astype(np.float32)
    kw = dict(subregion=subregion, scale_count=1, sigma_level=1, loop_gain=0.2, major_loop_miter=2, minor_loop_miter=2,
              conv_mode=mode, enforce_positivity=True)
    img, ref = DataImage(dirty, psf, None, 1.0, 1.0), omain.OracleImage(dirty, psf)
    img.moresane(precision="float64", **kw)
    ref.moresane(**kw)
    assert np.any(ref.model)
    assert _rel(img.model, ref.model) < 1e-7 and _rel(img.residual, ref.residual) < 1e-7
