"""Convolutions on frames that are not powers of two, over the stages of their plans.

Frames whose column and row lengths use every step (one stage of radix 2 to 13, or two at once), first, between
and last; plans of one row step and of many; rows of odd length; images and results at addresses that
are not a multiple of two values (which the vector loads and stores of the row passes need); frames at
which the block shapes of the passes change.  A pass rounds every value about once a stage, each time
by some 1.5 * 2^-24 rms, in at most 8 + 8 column and 4 + 4 row stages: 5e-7 rms of the result, held to three times that.
"""

import numpy as np
import pytest
import torch

from oracle import convolution64 as oconv
from pymoresane_amd import _lib
import test_gpu_float64_frames as float64_frames

pytestmark = pytest.mark.gpu

FRAMES = [(n, "linear") for n in (3, 5, 6, 7, 9, 11, 13, 15, 21, 27, 33, 35, 36, 39, 40, 42, 65, 77, 80, 81, 91,
                                  121, 125, 135, 143, 169, 189, 195, 210, 225, 243, 286, 343, 405, 440, 625, 715, 729,
                                  1001, 1287, 2187)]
FRAMES += [(n, "circular") for n in (6, 10, 12, 14, 18, 20, 22, 24, 26, 28, 30, 48, 160, 162, 168, 700, 2002, 4992, 5040)]


@pytest.mark.parametrize("n,mode", FRAMES)
def test_convolution_of_a_frame_of_any_even_side(hip, n, mode):
    print("convolution n=%d %s" % (n, mode), flush=True)
    lib = _lib.lib()
    p = 2 * n if mode == "linear" else n
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, n)).astype(np.float32)
    psf = rng.standard_normal((p, p)).astype(np.float32)
    want = oconv.fft_convolve(x, oconv.psf_spectrum(psf), mode)
    dpsf = torch.from_numpy(psf).cuda()
    spec = torch.empty(lib.pms_fft_spectrum_bytes(p), dtype=torch.uint8, device="cuda")
    work = torch.empty(max(lib.pms_fft_work_bytes(n, p), lib.pms_fft_work_bytes(p, p)), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    _lib.check(lib.pms_psf_spectrum(dpsf.data_ptr(), p, p, spec.data_ptr(), work.data_ptr(), None))
    for at in (0, 1):  # the image and the result at the start of their buffers, and one value into them
        src = torch.full((n * n + 2,), float("nan"), device="cuda")
        out = torch.full((n * n + 2,), -7.0, device="cuda")
        src[at:at + n * n] = torch.from_numpy(x).cuda().reshape(-1)
        torch.cuda.synchronize()
        _lib.check(lib.pms_fft_convolve(src[at:].data_ptr(), n, p, spec.data_ptr(), out[at:].data_ptr(), work.data_ptr(), None))
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.all(got[:at] == -7.0) and np.all(got[at + n * n:] == -7.0)
        got = got[at:at + n * n].reshape(n, n)
        assert np.linalg.norm(got - want) <= 1.5e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("n,mode", [(20, "circular"), (44, "linear"), (66, "linear"), (126, "linear"), (182, "linear"),
                                    (150, "linear"), (312, "circular"), (500, "linear"), (1000, "circular"),
                                    (1350, "linear"), (2600, "linear")])
def test_float64_residual_on_a_frame_of_any_even_side(hip, n, mode):
    float64_frames.test_float64_residual_is_the_oracles_convolution(hip, n, mode)
