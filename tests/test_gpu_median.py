"""The noise estimate where its ranges of sizes meet and where its sampled range does not help.

Planes of at most 32768 noise pixels are selected in one block; larger ones through a sampled range of
keys, with 8192 or (from 2^20 pixels) 16384 samples.  The estimate is exact in every case, so it must
equal np.median of the float32 values bit for bit: at the sizes where the kernels change, odd and even
counts, with border and interior masks, on tied and quantised values, and on planes made so that the
sample misses the median's rank or so that the range holds far more keys than the sample says.
"""

import numpy as np
import pytest

from oracle import toolbox64 as otools
from pymoresane_amd import _lib
from pymoresane_amd import iuwt_toolbox as tools

pytestmark = pytest.mark.gpu


def _check(x, **kw):
    print("median of %s %s" % (x.shape, kw), flush=True)
    np.testing.assert_array_equal(tools.estimate_threshold(x, **kw), otools.estimate_threshold(x, **kw))


@pytest.mark.parametrize("shape", [(1, 1), (1, 2), (3, 5), (64, 128), (91, 90), (8193, 1), (128, 256), (181, 181),
                                   (182, 181), (250, 132), (1023, 1025), (1024, 1024), (1031, 1029)])
def test_median_at_the_edges_of_its_kernels(hip, shape):
    rng = np.random.default_rng(shape[0] * 7 + shape[1])
    _check((rng.standard_normal((2,) + shape) * 3).astype(np.float32))


@pytest.mark.parametrize("shape,edge,interior", [((200, 210), 9, 0), ((200, 210), 0, 60), ((300, 301), 20, 100),
                                                 ((1100, 1080), 7, 0), ((1100, 1080), 0, 400), ((260, 40), 2, 3)])
def test_median_of_masked_planes(hip, shape, edge, interior):
    rng = np.random.default_rng(shape[1])
    _check(rng.standard_normal((3,) + shape).astype(np.float32), edge_excl=edge, int_excl=interior)


def _sampled(area):
    """The pixels that the sample reads: four neighbours in each stratum."""
    chunks = 2048 if area < 1 << 20 else 4096
    c = np.arange(chunks, dtype=np.uint64)
    stratum = area // chunks
    at = c * stratum + (((c * 2654435761) & 0xffffffff) >> 8) % (stratum - 3)
    at -= at % 4  # an aligned plane is read in quads
    return (at[:, None] + np.arange(4, dtype=np.uint64)).ravel().astype(np.int64)


@pytest.mark.parametrize("shape", [(300, 400), (1100, 1000)])
@pytest.mark.parametrize("kind", ["zeros", "half zeros", "integers", "fine integers", "two values", "infinite",
                                  "sample high", "sample low", "sample wide"])
def test_median_where_the_sampled_range_does_not_help(hip, shape, kind):
    rng = np.random.default_rng(17)
    n = shape[0] * shape[1]
    x = rng.standard_normal(n).astype(np.float32)
    at = _sampled(n)
    if kind == "zeros":
        x[:] = 0
    elif kind == "half zeros":
        x[rng.random(n) < 0.5] = 0
    elif kind == "integers":
        x = rng.integers(0, 30, n).astype(np.float32)
    elif kind == "fine integers":
        x = rng.integers(0, 90, n).astype(np.float32) + np.float32(1e5)
    elif kind == "two values":
        x = np.where(np.arange(n) % 2 == 0, 1.0, 2.0).astype(np.float32)
    elif kind == "infinite":
        x[rng.random(n) < 0.6] = np.inf
    elif kind == "sample high":  # the range lies above nearly every key
        x[at] = 1e6 + rng.random(at.size).astype(np.float32)
    elif kind == "sample low":
        x[at] = 1e-6 * rng.random(at.size).astype(np.float32)
    else:  # nearly every key lies in the range
        x = (1 + 0.001 * rng.random(n)).astype(np.float32)
        x[at] = 0.5 + rng.random(at.size).astype(np.float32)
    _check(x.reshape((1,) + shape))
    _check(x[:-shape[1]].reshape((1, shape[0] - 1, shape[1])))


def test_median_of_planes_that_are_not_16_byte_aligned(hip):
    rng = np.random.default_rng(5)
    x = rng.standard_normal((2, 211, 215)).astype(np.float32)  # an odd plane: the second starts unaligned
    _check(x)
    base = _lib.DeviceArray.from_host(np.concatenate([np.zeros(1, np.float32), x.ravel()]))
    view = _lib.DeviceArray.view(base, 4, x.shape, np.float32)
    np.testing.assert_array_equal(tools.estimate_threshold(view), otools.estimate_threshold(x))
