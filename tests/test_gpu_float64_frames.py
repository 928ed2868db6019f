"""Float64 convolutions on power-of-two frames, at every frame side their kernels are built for.

A clean in the float64 mode, stopped after one major and one minor iteration, leaves residual = dirty -
model convolved with the PSF.  The residual and model come out in float32, so the residual may differ from
that of the float32 model by half an ulp of itself and of the model's terms; the convolution's own error,
some units of 2^-53 times the largest term, is given 1e-13.
"""

import numpy as np
import pytest

from oracle import convolution64 as oconv
from pymoresane_amd.main import DataImage
from pymoresane_amd import synth

pytestmark = pytest.mark.gpu


def _pair(n, factor):
    """Six Gaussian sources and a Gaussian PSF (its dirty image is exact, without a convolution)."""
    rng = np.random.default_rng(50 + n)
    psf = synth.make_gaussian_psf(factor * n, 4.0)
    y = np.arange(n, dtype=np.float64)
    sig = synth.fwhm_to_sigma(4.0)
    dirty = rng.normal(0.0, 1e-4, (n, n))
    for _ in range(6):
        cy, cx = rng.integers(0, n, 2)
        dirty += rng.uniform(0.1, 1.0) * np.outer(np.exp(-0.5 * ((y - cy) / sig) ** 2), np.exp(-0.5 * ((y - cx) / sig) ** 2))
    return dirty.astype(np.float32), psf


@pytest.mark.parametrize("n,mode", [(16, "linear"), (32, "circular"), (32, "linear"), (64, "circular"), (64, "linear"),
                                    (128, "linear"), (256, "circular"), (256, "linear"), (512, "linear"),
                                    (1024, "circular"), (1024, "linear"), (2048, "linear"), (4096, "linear")])
def test_float64_residual_is_the_oracles_convolution(hip, n, mode):
    print("float64 frame of %d^2 %s" % (n, mode), flush=True)
    dirty, psf = _pair(n, 2 if mode == "linear" else 1)
    img = DataImage(dirty, psf, None, 1.0, 1.0)
    img.moresane(scale_count=min(3, int(np.log2(n)) - 1), loop_gain=0.2, major_loop_miter=1, minor_loop_miter=1,
                 conv_mode=mode, precision="float64")
    oconv.set_fft_workers(8)
    try:
        spec = oconv.psf_spectrum(psf)
        want = dirty.astype(np.float64) - oconv.fft_convolve(img.model, spec, mode)
        # the model that was convolved is the float64 one; its float32 copy is off by half an ulp per pixel
        # (the PSF is positive with peak 1)
        terms = oconv.fft_convolve(np.abs(img.model), spec, mode) if n <= 1024 else np.abs(img.model).sum()
    finally:
        oconv.set_fft_workers(1)
    bound = 2.0 ** -24 * (np.abs(want) + terms) + 1e-13 * np.abs(dirty).max()
    assert np.any(img.model)
    assert np.all(np.abs(img.residual - want) <= bound)
