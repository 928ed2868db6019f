"""Source extraction of masks whose objects cross many tiles or hold many unions a word: results and times.

Vertical lines joined by one row, one object that winds through every row, and noise with 45% set pixels.  The
results equal the scipy-based oracle's on stacks on both sides of the rule for the step that links all scales at
once (2048 tiles); the times stay near those of thin noise: 1.5 to 2.8 times, where unions one after the other in a
thread and chains walked scale after scale took 3.4 to 6 times; the bound of 4 lies between for at least one of
them at either size.
"""

import numpy as np
import pytest
import torch

from oracle import toolbox64 as otools
from pymoresane_amd import _lib
from pymoresane_amd import iuwt_toolbox as tools

pytestmark = pytest.mark.gpu


def _mask(kind, s, h, w, rng):
    yy, xx = np.arange(h)[:, None], np.arange(w)[None, :]
    if kind == "lines":
        on = (xx % 2 == 0) | (yy == 0)
    elif kind == "winding":
        on = (yy % 2 == 0) | (yy % 4 == 1) & (xx == w - 1) | (yy % 4 == 3) & (xx == 0)
    else:
        return rng.random((s, h, w)) < (0.45 if kind == "dense" else 0.01)
    return np.broadcast_to(on, (s, h, w))


@pytest.mark.parametrize("s,h,w", [(1, 33, 65), (5, 350, 350), (5, 500, 517), (7, 700, 704), (3, 1400, 1401)])
@pytest.mark.parametrize("kind", ["lines", "winding", "dense"])
def test_extraction_of_long_objects_equals_the_oracle(hip, s, h, w, kind):
    print("extraction %d x %dx%d %s" % (s, h, w, kind), flush=True)
    rng = np.random.default_rng(h + w)
    x = np.where(_mask(kind, s, h, w, rng), rng.standard_normal((s, h, w)), 0.0).astype(np.float32)
    ext, mask, labels = tools.source_extraction(x, 0.6, return_labels=True)
    rext, rmask, rlabels = otools.source_extraction(x, 0.6, return_labels=True)
    np.testing.assert_array_equal(mask, rmask)
    np.testing.assert_array_equal(ext, np.asarray(rext, np.float32))
    np.testing.assert_array_equal(labels, rlabels)


def _microseconds(x):
    lib = _lib.lib()
    s, h, w = x.shape
    ext = torch.empty_like(x)
    mask = torch.empty(x.shape, dtype=torch.uint8, device="cuda")
    work = torch.empty(lib.pms_extract_work_bytes(s, h, w), dtype=torch.uint8, device="cuda")
    start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    times = []
    for _ in range(8):
        torch.cuda.synchronize()
        start.record()
        for _ in range(5):
            _lib.check(lib.pms_source_extraction(x.data_ptr(), s, h, w, 0.75, 0, ext.data_ptr(), mask.data_ptr(), None,
                                                 work.data_ptr(), None))
        stop.record()
        torch.cuda.synchronize()
        times.append(200 * start.elapsed_time(stop))
    return min(times)


@pytest.mark.parametrize("s,n", [(5, 350), (5, 600)])
def test_long_objects_take_about_as_long_as_thin_noise(hip, s, n):
    rng = np.random.default_rng(n)
    values = rng.standard_normal((s, n, n))
    took = {}
    for kind in ("thin", "lines", "winding", "dense"):
        x = np.where(_mask(kind, s, n, n, rng), values, 0.0).astype(np.float32)
        took[kind] = _microseconds(torch.from_numpy(x).cuda())
    print("%d x %d^2: %s" % (s, n, took), flush=True)
    for kind in ("lines", "winding", "dense"):
        assert took[kind] < 4 * took["thin"]
