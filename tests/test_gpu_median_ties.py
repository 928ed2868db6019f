"""The noise estimate of planes on which many pixels are equal: blanked images, quantised or two-valued ones.

The estimate equals np.median bit for bit where the median's rank is the last of the equal keys below the sampled
range, the first of those above it, or next to either, with odd and even counts, with and without an edge mask.
It also takes about as long as on other planes: each kind here took 7 to 140 times as long when one block selected
from the whole plane, and takes 1 to 2 times as long now; the bound of 4 lies between.
"""

import numpy as np
import pytest
import torch

from oracle import moresane64 as omain
from oracle import toolbox64 as otools
from pymoresane_amd import _lib, synth
from pymoresane_amd import iuwt_toolbox as tools
from pymoresane_amd.main import DataImage

pytestmark = pytest.mark.gpu


def _tied(kind, n, cut, rng):
    """n values of which `cut` lie at or below the first tied value's last rank."""
    x = rng.random(n) + 0.5
    if kind == "low ties":  # zeros, then distinct values
        x[:cut] = 0
    elif kind == "high ties":  # distinct values, then equal ones above them
        x[cut:] = 3.0
    elif kind == "both":  # zeros, a few distinct values, equal ones
        x[:cut - n // 64] = 0
        x[cut:] = 3.0
    elif kind == "two values":
        x[:] = 3.0
        x[:cut] = 1.0
    else:  # neighbouring values: the range between them is empty or a single key
        x[:] = np.float32(1.0)
        x[cut - n // 64:] = np.nextafter(np.float32(1), np.float32(2))
        x[cut:] = np.nextafter(np.nextafter(np.float32(1), np.float32(2)), np.float32(2))
    x = x.astype(np.float32) * rng.choice([-1, 1], n).astype(np.float32)
    return x[rng.permutation(n)]


@pytest.mark.parametrize("kind", ["low ties", "high ties", "both", "two values", "neighbours"])
@pytest.mark.parametrize("shape", [(300, 400), (301, 401), (1100, 1000), (1101, 1001)])
def test_median_next_to_tied_keys(hip, kind, shape):
    print("median of %s, %s" % (shape, kind), flush=True)
    n = shape[0] * shape[1]
    rng = np.random.default_rng(n)
    x = np.stack([_tied(kind, n, n // 2 + d, rng) for d in (-2, -1, 0, 1, 2)]).reshape((5,) + shape)
    np.testing.assert_array_equal(tools.estimate_threshold(x), otools.estimate_threshold(x))
    inner = np.zeros((5, shape[0] + 6, shape[1] + 6), np.float32)
    inner[:, 3:-3, 3:-3] = x
    np.testing.assert_array_equal(tools.estimate_threshold(inner, edge_excl=3), otools.estimate_threshold(x))


def _microseconds(x):
    lib = _lib.lib()
    s, h, w = x.shape
    thr = torch.empty(s, dtype=torch.float64, device="cuda")
    work = torch.empty(lib.pms_threshold_work_bytes(s, h, w), dtype=torch.uint8, device="cuda")
    start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    times = []
    for _ in range(6):
        torch.cuda.synchronize()
        start.record()
        _lib.check(lib.pms_estimate_threshold(x.data_ptr(), s, h, w, 0, 0, thr.data_ptr(), work.data_ptr(), None))
        stop.record()
        torch.cuda.synchronize()
        times.append(1e3 * start.elapsed_time(stop))
    return min(times)


def test_tied_planes_take_about_as_long_as_others(hip):
    n = 4096
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    x = torch.randn((7, n, n), generator=gen, device="cuda")
    u = torch.rand((7, n, n), generator=gen, device="cuda")
    usual = _microseconds(x)
    kinds = {"%d%% zeros" % round(100 * f): torch.where(u < f, torch.zeros_like(x), x) for f in (0.48, 0.5, 0.52)}
    kinds["two values"] = torch.where(u < 0.5, torch.ones_like(x), 2 * torch.ones_like(x))
    kinds["near one"] = 1 + 1e-5 * x
    kinds["integers"] = torch.floor(30 * u)
    for name, planes in kinds.items():
        took = _microseconds(planes)
        print("%s: %.0f us, %.0f us without ties" % (name, took, usual), flush=True)
        assert took < 4 * usual


def test_float64_clean_of_a_half_blanked_image(hip):
    """More than half of the wavelet coefficients are zero in the float64 mode, whose keys are eight bytes."""
    n = 256
    dirty, psf = synth.make_pair(n, 12, n_points=12, n_blobs=1)
    dirty[:, : n * 9 // 16] = 0
    kw = dict(scale_count=3, loop_gain=0.2, major_loop_miter=2, minor_loop_miter=10, sigma_level=3, enforce_positivity=True)
    img, ref = DataImage(dirty, psf, None, 1.0, 1.0), omain.OracleImage(dirty, psf)
    img.moresane(precision="float64", **kw)
    ref.moresane(**kw)
    assert np.any(ref.model)
    for a, b in ((img.model, ref.model), (img.residual, ref.residual)):
        assert np.linalg.norm(a.astype(np.float64) - b) < 1e-7 * np.linalg.norm(b)
