"""The 32 x 32 tile kernels of the transform against one launch per scale: the same bits.

Shapes on both sides of each rule that chooses them (256 tiles a launch, phases that fill their tiles, the pixel
limits per pair of scales), with sides that end inside a tile or a phase, and a whole deconvolution with masks
and positivity, whose operator runs masked decompositions and recompositions.
"""

import numpy as np
import pytest
import torch

from pymoresane_amd import _lib, synth
from pymoresane_amd.main import DataImage

pytestmark = pytest.mark.gpu

ONE_SCALE = {"PMS_IUWT_SMALL2": "0", "PMS_IUWT_PAIR": "0"}


def _transform(x, scales, adjust):
    lib = _lib.lib()
    h, w = x.shape
    detail = torch.full((scales - adjust, h, w), float("nan"), device="cuda")
    smooth, out = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
    work = torch.empty(lib.pms_iuwt_work_bytes(h, w), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    _lib.check(lib.pms_iuwt_decompose(x.data_ptr(), h, w, scales, adjust, detail.data_ptr(), smooth.data_ptr(),
                                      work.data_ptr(), None))
    _lib.check(lib.pms_iuwt_recompose(detail.data_ptr(), scales - adjust, h, w, adjust, smooth.data_ptr(), out.data_ptr(),
                                      work.data_ptr(), None))
    torch.cuda.synchronize()
    return detail, smooth, out


@pytest.mark.parametrize("h,w,scales,adjust", [
    (511, 513, 5, 0), (512, 512, 6, 0), (352, 800, 6, 1), (500, 517, 4, 2), (601, 1000, 5, 0), (769, 1025, 6, 0),
    (1024, 1024, 7, 0), (1024, 1025, 6, 1), (2048, 2048, 6, 0), (2047, 2050, 4, 0), (3001, 2999, 4, 0), (3600, 3500, 2, 0),
    (64, 8200, 4, 0), (8200, 64, 4, 0)])
def test_tiles_give_the_planes_of_single_scale_launches(hip, monkeypatch, h, w, scales, adjust):
    print("tiles %dx%d scales %d-%d" % (h, w, adjust, scales), flush=True)
    rng = np.random.default_rng(h + w)
    x = torch.from_numpy(rng.standard_normal((h, w)).astype(np.float32)).cuda()
    got = _transform(x, scales, adjust)
    for k, v in ONE_SCALE.items():
        monkeypatch.setenv(k, v)
    for a, b in zip(got, _transform(x, scales, adjust)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n", [512, 700])
def test_a_deconvolution_on_tiles_is_that_of_single_scale_launches(hip, monkeypatch, n):
    print("deconvolution of %d^2 on tiles" % n, flush=True)
    dirty, psf = synth.make_pair(n, 17, n_points=20, n_blobs=2)
    got = []
    for env in ({}, ONE_SCALE):
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        img = DataImage(dirty, psf, None, 1.0, 1.0)
        img.moresane(scale_count=4, loop_gain=0.2, major_loop_miter=3, enforce_positivity=True)
        got.append((img.model, img.residual, img.trace))
    assert got[0][2] == got[1][2]
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
