"""Transforms whose output takes the place of an input that an earlier scale has used up.

A decomposition's input may be its smoothed plane or any detail plane but the first, a recomposition's output
its smoothed plane or any detail plane but the first (one scale a launch reads those before the output is
written), where at least one scale lies between.  Such calls give the planes of separate buffers, bit for bit.
"""

import numpy as np
import pytest
import torch

from pymoresane_amd import _lib

pytestmark = pytest.mark.gpu

SHAPES = [(64, 80), (200, 220), (512, 512), (601, 1000), (1024, 1024), (2047, 1030)]


def _planes(n, h, w):
    return torch.full((n, h, w), float("nan"), device="cuda")


@pytest.mark.parametrize("h,w", SHAPES)
@pytest.mark.parametrize("scales", [2, 3, 4])
def test_decomposition_over_its_input(hip, h, w, scales):
    lib = _lib.lib()
    rng = np.random.default_rng(h + w)
    x = torch.from_numpy(rng.standard_normal((h, w)).astype(np.float32)).cuda()
    work = torch.empty(lib.pms_iuwt_work_bytes(h, w), dtype=torch.uint8, device="cuda")

    def run(source, detail, smooth):
        torch.cuda.synchronize()
        _lib.check(lib.pms_iuwt_decompose(source.data_ptr(), h, w, scales, 0, detail.data_ptr(), smooth.data_ptr(),
                                          work.data_ptr(), None))
        torch.cuda.synchronize()
        return detail, smooth

    want_d, want_s = run(x, _planes(scales, h, w), _planes(1, h, w)[0])
    print("decomposition over its input %dx%d, %d scales" % (h, w, scales), flush=True)
    s = x.clone()
    d, s = run(s, _planes(scales, h, w), s)
    assert torch.equal(d, want_d) and torch.equal(s, want_s)
    for k in range(1, scales):
        d = _planes(scales, h, w)
        d[k] = x
        d, s = run(d[k], d, _planes(1, h, w)[0])
        assert torch.equal(d, want_d) and torch.equal(s, want_s)


@pytest.mark.parametrize("h,w", SHAPES)
@pytest.mark.parametrize("scales", [2, 3, 4])
def test_recomposition_over_its_inputs(hip, h, w, scales):
    lib = _lib.lib()
    rng = np.random.default_rng(3 * h + w)
    planes = torch.from_numpy(rng.standard_normal((scales + 1, h, w)).astype(np.float32)).cuda()
    work = torch.empty(lib.pms_iuwt_work_bytes(h, w), dtype=torch.uint8, device="cuda")

    def run(target):
        p = planes.clone()  # the detail planes, then the smoothed one
        results = []
        for smooth in (p[scales], None):
            p.copy_(planes)
            out = _planes(1, h, w)[0] if target is None else p[target]
            torch.cuda.synchronize()
            _lib.check(lib.pms_iuwt_recompose(p.data_ptr(), scales, h, w, 0, None if smooth is None else smooth.data_ptr(),
                                              out.data_ptr(), work.data_ptr(), None))
            torch.cuda.synchronize()
            results.append(out.clone())
        return results

    want = run(None)
    print("recomposition over its inputs %dx%d, %d scales" % (h, w, scales), flush=True)
    for target in range(1, scales + 1):
        for i, (got, ref) in enumerate(zip(run(target), want)):
            if i == 1 and scales == 2:
                continue  # without a smoothed plane the one launch reads the coarsest plane around its output
            assert torch.equal(got, ref)
