"""Source extraction where its tiles, bit words and quads can go wrong, against the scipy-based oracle.

Labelling works on 64 x 32 pixel tiles and one 64-bit word per row and 64 columns, the keep rule on
quads of four pixels: sides around those sizes, one-pixel planes, widths that leave part of a word or
of a quad, and masks that cross every tile border (dense noise, diagonal lines, one single object,
long serpentine objects whose union chains visit every tile).  Results are integers or copies of the
input, so they must be equal.
"""

import numpy as np
import pytest

from oracle import toolbox64 as otools
from pymoresane_amd import _lib
from pymoresane_amd import iuwt_toolbox as tools

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (1, 64), (65, 1), (31, 63), (32, 64), (33, 65), (64, 128), (63, 127), (97, 130), (100, 260), (161, 66)]


def _planes(pattern, s, h, w, rng):
    x = rng.standard_normal((s, h, w)).astype(np.float32)
    yy, xx = np.mgrid[0:h, 0:w]
    if pattern == "sparse":
        on = rng.random((s, h, w)) < 0.02
    elif pattern == "dense":
        on = rng.random((s, h, w)) < 0.45
    elif pattern == "diagonals":
        on = np.stack([((xx + yy) if k % 2 else (xx - yy)) % 5 == 0 for k in range(s)])
    elif pattern == "serpentine":
        row = (yy % 2 == 0)
        turn = (yy % 4 == 1) & (xx == w - 1) | (yy % 4 == 3) & (xx == 0)
        on = np.stack([row | turn] * s)
    else:
        on = np.ones((s, h, w), dtype=bool)
    return np.where(on, x, 0).astype(np.float32)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("pattern", ["sparse", "dense", "diagonals", "serpentine", "full"])
def test_extraction_equals_the_oracle_at_tile_edges(hip, shape, pattern):
    h, w = shape
    rng = np.random.default_rng(h * 1000 + w)
    x = _planes(pattern, 3, h, w, rng)
    if not all(p.any() for p in x):
        x[:, 0, 0] = 1.0  # the tolerance rule needs a maximum in every plane
    print("extraction %dx%d %s" % (h, w, pattern), flush=True)
    for neg in (False, True):
        ext, mask, labels = tools.source_extraction(x, 0.6, neg_comp=neg, return_labels=True)
        rext, rmask, rlabels = otools.source_extraction(x, 0.6, neg_comp=neg, return_labels=True)
        np.testing.assert_array_equal(mask, rmask)
        np.testing.assert_array_equal(ext, np.asarray(rext, np.float32))
        np.testing.assert_array_equal(labels, rlabels)


def test_extraction_with_an_unaligned_mask_buffer(hip):
    """The four-byte mask stores need an aligned mask; another one takes the elementwise stores."""
    rng = np.random.default_rng(9)
    x = _planes("dense", 2, 40, 72, rng)
    lib = _lib.lib()
    src = _lib.DeviceArray.from_host(x)
    ext = _lib.DeviceArray(x.shape)
    room = _lib.DeviceArray((x.size + 4,), np.uint8)
    mask = _lib.DeviceArray.view(room, 1, x.shape, np.uint8)
    work = _lib.DeviceArray((lib.pms_extract_work_bytes(2, 40, 72),), np.uint8)
    _lib.check(lib.pms_source_extraction(src.ptr, 2, 40, 72, 0.6, 0, ext.ptr, mask.ptr, None, work.ptr, None))
    rext, rmask = otools.source_extraction(x, 0.6)
    np.testing.assert_array_equal(mask.get(), rmask)
    np.testing.assert_array_equal(ext.get(), np.asarray(rext, np.float32))
