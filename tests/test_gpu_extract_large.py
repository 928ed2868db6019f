"""Source extraction of stacks large enough for its other kernels, against the scipy-based oracle.

Stacks of more than 1024 tiles are labelled by 128 threads a tile, and planes of 2^21 quads or more (some 2900^2
pixels) take four quads a thread in the keep rule, with vector stores where the width is a multiple of four and
elementwise ones otherwise.  Heights and widths end inside tiles, words and quads; the masks cross every tile
border.  Results are integers or copies of the input, so they must be equal.
"""

import numpy as np
import pytest

from oracle import toolbox64 as otools
from pymoresane_amd import iuwt_toolbox as tools

pytestmark = pytest.mark.gpu


def _planes(pattern, s, h, w):
    rng = np.random.default_rng(h * 10 + w)
    x = rng.standard_normal((s, h, w)).astype(np.float32)
    yy, xx = np.arange(h)[:, None], np.arange(w)[None, :]
    if pattern == "dense":
        on = rng.random((s, h, w), dtype=np.float32) < 0.45
    else:  # one object whose chain of unions visits every tile
        on = (yy % 2 == 0) | (yy % 4 == 1) & (xx == w - 1) | (yy % 4 == 3) & (xx == 0)
        on = np.broadcast_to(on, x.shape)
    return np.where(on, x, np.float32(0))


@pytest.mark.parametrize("s,h,w", [(5, 599, 700), (5, 600, 701), (2, 2900, 2904), (2, 2901, 2903)])
@pytest.mark.parametrize("pattern", ["dense", "serpentine"])
def test_extraction_of_large_stacks_equals_the_oracle(hip, s, h, w, pattern):
    x = _planes(pattern, s, h, w)
    print("extraction %d x %dx%d %s" % (s, h, w, pattern), flush=True)
    for neg in ((False, True) if h < 1000 else (False,)):
        ext, mask, labels = tools.source_extraction(x, 0.6, neg_comp=neg, return_labels=True)
        rext, rmask, rlabels = otools.source_extraction(x, 0.6, neg_comp=neg, return_labels=True)
        np.testing.assert_array_equal(mask, rmask)
        np.testing.assert_array_equal(ext, np.asarray(rext, np.float32))
        np.testing.assert_array_equal(labels, rlabels)
