"""Float64 transforms in pairs of scales at sides that are no multiple of their tiles.

The float64 transforms take two scales a launch on tiles of 16 lattice steps and leave an odd scale, and
scales longer than the side, to one-scale launches.  By-scale cleans go through every scale count, so
each side below runs pairs with and without a scale left over, with the masks of the minor loop.  As for
the other float64 cleans, decisions must equal the float64 oracle's and models and residuals agree to
the float32 rounding of the outputs (1e-7; a wrong tap errs by O(1)).
"""

import numpy as np
import pytest

from oracle import moresane64 as omain
from pymoresane_amd import synth
from pymoresane_amd.main import DataImage

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("n,stop", [(22, 3), (36, 4), (100, 5), (130, 5)])
def test_float64_by_scale_cleans_of_ragged_sides(hip, n, stop):
    print("float64 by scale, %d^2 to scale %d" % (n, stop), flush=True)
    dirty, psf = synth.make_pair(n, 70 + n, n_points=8, n_blobs=1)
    kw = dict(start_scale=1, stop_scale=stop, loop_gain=0.2, major_loop_miter=4, enforce_positivity=True)
    img = DataImage(dirty, psf, None, 1.0, 1.0)
    img.moresane_by_scale(precision="float64", **kw)
    ref = omain.OracleImage(dirty, psf)
    ref.moresane_by_scale(**kw)
    assert any(e[0] == "update" for e in ref.trace)
    assert [tuple(v for v in e if not isinstance(v, float)) for e in img.trace] == \
        [tuple(v for v in e if not isinstance(v, float)) for e in ref.trace]
    assert _rel(img.model, ref.model) < 1e-7 and _rel(img.residual, ref.residual) < 1e-7
