"""Rounding error of the float64 convolution on power-of-two frames, against extended precision (80 bits).

A transform of side p has log2(p) levels of additions and products on each axis, there and back: 4 log2(p) in a
convolution.  A level whose twiddles are good to half a unit in the last place adds a relative rms error of about
one unit of 2^-53, independent of the others', so the result stays within 1.1 * 2^-53 * sqrt(4 log2 p).  Twiddles
formed by squaring err by several units and miss that bound.

The float64 convolution has no entry point of its own (cleans return float32), so the library's C++ function is
called under its exported name.
"""

import ctypes

import numpy as np
import pytest
import scipy.fft
import torch

from pymoresane_amd import _lib

pytestmark = pytest.mark.gpu

SPECTRUM = "_ZN3pms17gfft_psf_spectrumIddEEvPKT0_iiPNS_2CxIT_EES7_P12ihipStream_t"  # gfft_psf_spectrum<double, double>
CONVOLVE = "_ZN3pms15gfft_conv_batchIdEEvPKNS_8GConvJobIT_EEiiiP12ihipStream_t"  # gfft_conv_batch<double>


class Job(ctypes.Structure):
    _fields_ = [(k, ctypes.c_void_p) for k in ("image", "spectrum", "out", "work", "pred")]


@pytest.mark.parametrize("p,n", [(256, 128), (512, 256), (512, 512), (1024, 512), (2048, 1024)])
def test_rounding_of_the_float64_convolution(hip, p, n):
    print("float64 convolution error, frame %d, image %d" % (p, n), flush=True)
    lib = _lib.lib()
    rng = np.random.default_rng(p + n)
    x, psf = rng.standard_normal((n, n)), rng.standard_normal((p, p))
    dx, dpsf = torch.from_numpy(x).cuda(), torch.from_numpy(psf).cuda()
    spectrum = torch.empty((p // 2 + 1) * p * 2, dtype=torch.float64, device="cuda")
    work = torch.empty(4 * (p // 2 + 1) * p, dtype=torch.float64, device="cuda")
    out = torch.empty((n, n), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    pointer = ctypes.c_void_p
    getattr(lib, SPECTRUM)(pointer(dpsf.data_ptr()), p, p, pointer(spectrum.data_ptr()), pointer(work.data_ptr()), None)
    job = Job(dx.data_ptr(), spectrum.data_ptr(), out.data_ptr(), work.data_ptr(), None)
    getattr(lib, CONVOLVE)(ctypes.byref(job), 1, n, p, None)
    torch.cuda.synchronize()
    frame = np.zeros((p, p), np.longdouble)
    frame[:n, :n] = x
    centred = np.roll(psf, (-(p // 2), -(p // 2)), (0, 1)).astype(np.longdouble)
    want = scipy.fft.irfft2(scipy.fft.rfft2(frame, workers=8) * scipy.fft.rfft2(centred, workers=8), s=(p, p), workers=8)
    want = want[:n, :n]
    err = float(np.sqrt(np.mean((out.cpu().numpy() - want) ** 2) / np.mean(want ** 2)))
    assert err < 1.1 * 2.0 ** -53 * np.sqrt(4 * np.log2(p)), err
