"""The work that users of this framework have it do, as cases that can be timed and compared.

Five kinds of case, each through a public entry point:

* ``transform``   -- IUWT of an image and the inverse of its planes (``pms_iuwt_decompose``,
                     ``pms_iuwt_recompose``): both directions of the wavelet transform, device to device;
* ``convolve``    -- FFT convolution of an image with a PSF whose spectrum is kept (``pms_fft_convolve``),
                     linear (frame twice the image) or circular (frame as large as the image);
* ``detect``      -- what follows each decomposition of a clean: noise per scale, thresholding, source
                     extraction (``pms_estimate_threshold``, ``pms_apply_threshold``,
                     ``pms_source_extraction``);
* ``deconvolve``  -- a whole clean of one image, host arrays in and out (``DataImage.moresane`` and
                     ``moresane_by_scale``), in the float32 or the float64 mode;
* ``batch``       -- many independent cleans of ragged sizes at once (``batch.run_batch``).

Sizes follow this repository's tests and benchmark: planes of 64^2 to 4096^2, odd and non-square
ones among them, 3 to 7 scales, PSFs twice the image or as large as it.
"""

import numpy as np
import torch

from pymoresane_amd import _lib, batch
from pymoresane_amd.main import DataImage

DEVICE = "cuda"

# the settings of the repository's own cleans: gain 0.2, 4 sigma, tolerance 0.75, positive models
CLEAN = dict(loop_gain=0.2, sigma_level=4, tolerance=0.75, accuracy=1e-6, minor_loop_miter=30,
             enforce_positivity=True)


def listed():
    return [
        # a small image's transform: two or three launches a direction, their latency is the whole time
        {"name": "transform_128", "kind": "transform", "h": 128, "w": 128, "scales": 4},
        # a cut-out whose sides are neither equal nor powers of two
        {"name": "transform_601x1000", "kind": "transform", "h": 601, "w": 1000, "scales": 5},
        # a full survey image, the benchmark's size
        {"name": "transform_4096", "kind": "transform", "h": 4096, "w": 4096, "scales": 7},
        # the convolution of each iteration of a small clean
        {"name": "convolve_256", "kind": "convolve", "n": 256, "mode": "linear"},
        # an image side as imagers are asked for it, not a power of two
        {"name": "convolve_1000", "kind": "convolve", "n": 1000, "mode": "linear"},
        # a PSF as large as the image, the reference's circular mode
        {"name": "convolve_2048_circular", "kind": "convolve", "n": 2048, "mode": "circular"},
        # a full survey image with a PSF of twice its side, the benchmark's size
        {"name": "convolve_4096", "kind": "convolve", "n": 4096, "mode": "linear"},
        # one major iteration's detection on a middling image whose edges are left out of the noise
        {"name": "detect_500", "kind": "detect", "h": 500, "w": 500, "scales": 5, "edge_excl": 10},
        # the same on a full survey image
        {"name": "detect_4096", "kind": "detect", "h": 4096, "w": 4096, "scales": 7, "edge_excl": 0},
        # a short clean of a small image: many small launches one after another
        {"name": "clean_256", "kind": "deconvolve", "n": 256, "scales": 4, "majors": 10, "precision": "float32",
         "by_scale": False, "mode": "linear"},
        # scale by scale in the mode that computes as the reference's serial path does
        {"name": "clean_512_float64", "kind": "deconvolve", "n": 512, "scales": 4, "majors": 4,
         "precision": "float64", "by_scale": True, "mode": "linear"},
        # a night's cut-outs of several sizes, cleaned together
        {"name": "batch_28", "kind": "batch", "n256": 16, "n512": 8, "n1024": 4, "scales": 5, "majors": 6},
    ]


def _smooth(n):
    """n with no prime factor above 13, which an FFT frame side needs."""
    for f in (2, 3, 5, 7, 11, 13):
        while n % f == 0:
            n //= f
    return n == 1


def _log_size(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("transform", "transform", "convolve", "convolve", "detect", "detect", "deconvolve", "batch"))
    if kind in ("transform", "detect"):
        h = _log_size(rng, 64, 4096)
        if rng.random() < 0.3:  # sides that are powers of two are the commonest
            h = 1 << max(6, min(12, h.bit_length() - 1))
        w = h if rng.random() < 0.5 else max(64, min(4096, int(h * (0.5 + rng.random()))))
        top = min(h, w).bit_length() - 1  # 2^scales <= the shorter side
        case = {"kind": kind, "h": h, "w": w, "scales": rng.randint(3, min(7, top))}
        if kind == "detect":
            case["edge_excl"] = rng.choice((0, 0, 0, rng.randint(1, min(h, w) // 8)))
        return case
    if kind == "convolve":
        n = 2 * _log_size(rng, 32, 2048)
        while not _smooth(n):
            n -= 2
        if rng.random() < 0.4:
            n = 1 << (n.bit_length() - 1)
        return {"kind": kind, "n": n, "mode": rng.choice(("linear", "linear", "circular"))}
    if kind == "deconvolve":
        n = 2 * _log_size(rng, 48, 384)
        while not _smooth(n):
            n -= 2
        if rng.random() < 0.5:
            n = 1 << (n.bit_length() - 1)
        return {"kind": kind, "n": n, "scales": rng.randint(3, 4), "majors": rng.randint(3, 8),
                "precision": rng.choice(("float32", "float64")), "by_scale": rng.random() < 0.3,
                "mode": rng.choice(("linear", "linear", "circular"))}
    return {"kind": "batch", "n256": rng.randint(4, 16), "n512": rng.randint(0, 8), "n1024": rng.randint(0, 4),
            "scales": rng.randint(3, 5), "majors": rng.randint(2, 6)}


# ------------------------------------------------------------------------------------------ inputs
def _sky(n, seed, points=40, blobs=4):
    """Point sources of log-uniform flux and a few broad Gaussian blobs, float64 on the GPU."""
    rng = np.random.default_rng(seed)
    sky = np.zeros((n, n))
    np.add.at(sky, (rng.integers(0, n, points), rng.integers(0, n, points)), 10.0 ** rng.uniform(-3.0, 0.0, points))
    sky = torch.from_numpy(sky).to(DEVICE)
    y = torch.arange(n, dtype=torch.float64, device=DEVICE)
    for _ in range(blobs):
        cy, cx = rng.uniform(0, n, 2)
        sig, amp = rng.uniform(2.0, 8.0), rng.uniform(0.05, 0.3)
        sky += amp * torch.outer(torch.exp(-0.5 * ((y - cy) / sig) ** 2), torch.exp(-0.5 * ((y - cx) / sig) ** 2))
    return sky


def _psf(p, fwhm=4.0):
    """An elliptical Gaussian core with a faint ring, centred at p/2, peak 1."""
    c = torch.arange(p, dtype=torch.float64, device=DEVICE) - p // 2
    th = 0.5235987755982988  # 30 degrees
    a = c[:, None] * np.cos(th) + c[None, :] * np.sin(th)
    b = c[None, :] * np.cos(th) - c[:, None] * np.sin(th)
    k = 8.0 * np.log(2.0)
    psf = torch.exp(-0.5 * k * ((a / fwhm) ** 2 + (b / (0.75 * fwhm)) ** 2))
    psf += 0.05 * torch.exp(-((torch.sqrt(a * a + b * b) - 12.0) ** 2) / 4.5)
    return psf / psf.max()


def _convolved(x, psf):
    """x (n x n) convolved with a p x p PSF centred at p/2, in 64 bits: linear for p = 2n, circular for p = n."""
    n, p = x.shape[0], psf.shape[0]
    spec = torch.fft.rfft2(torch.roll(psf.double(), (-(p // 2), -(p // 2)), (0, 1)))
    return torch.fft.irfft2(torch.fft.rfft2(x.double(), s=(p, p)) * spec, s=(p, p))[:n, :n].contiguous()


def _noise(shape, seed, scale=1.0):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32) * scale


def _image(h, w, seed):
    """Noise of unit variance with 200 point sources of flux 0.01 to 10."""
    rng = np.random.default_rng(seed)
    at = torch.from_numpy(rng.choice(h * w, size=200, replace=False)).to(DEVICE)
    flux = torch.from_numpy((10.0 ** rng.uniform(-2.0, 1.0, 200)).astype(np.float32)).to(DEVICE)
    img = _noise((h, w), seed)
    img.view(-1)[at] += flux
    return img


def _pair(n, seed, psf_factor=2, fwhm=4.0):
    """A dirty image and its PSF, float32 host arrays."""
    psf = _psf(psf_factor * n, fwhm)
    dirty = _convolved(_sky(n, seed), psf).float() + _noise((n, n), seed, 1e-3)
    return dirty.cpu().numpy(), psf.float().cpu().numpy()


# ------------------------------------------------------------------------- the transform in 64 bits
def _smoothed(x, s):
    """One a trous pass of x in 64 bits: the B3 spline at spacing 2^s on both axes, half-sample-symmetric borders."""
    for axis in (0, 1):
        n = x.shape[axis]
        i = torch.arange(n, device=x.device)
        acc = torch.zeros_like(x)
        for k, c in zip((-2, -1, 0, 1, 2), (1.0, 4.0, 6.0, 4.0, 1.0)):
            j = (i + k * (1 << s)) % (2 * n)
            j = torch.where(j < n, j, 2 * n - 1 - j)
            acc += (c / 16.0) * x.index_select(axis, j)
        x = acc
    return x


def _decomposed(x, scales):
    """(detail planes, smoothed plane) of x in 64 bits: w_s = C_s - H C_{s+1}, C_{s+1} = H C_s."""
    c, planes = x.double(), []
    for s in range(scales):
        nxt = _smoothed(c, s)
        planes.append(c - _smoothed(nxt, s))
        c = nxt
    return torch.stack(planes), c


def _recomposed(planes, smooth):
    r = smooth
    for s in reversed(range(planes.shape[0])):
        r = _smoothed(r, s) + planes[s]
    return r


# ----------------------------------------------------------------------------------------- the cases
def _bytes(n):
    return torch.empty(int(n), dtype=torch.uint8, device=DEVICE)


def _planes(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device=DEVICE)


def prepare(case, seed):
    lib = _lib.lib()
    kind = case["kind"]
    st = {"case": case, "kind": kind}
    if kind == "transform":
        h, w, s = case["h"], case["w"], case["scales"]
        st.update(x=_image(h, w, seed), detail=_planes(s, h, w), smooth=_planes(h, w), out=_planes(h, w),
                  work=_bytes(lib.pms_iuwt_work_bytes(h, w)))
    elif kind == "convolve":
        n = case["n"]
        p = 2 * n if case["mode"] == "linear" else n
        psf = _psf(p, fwhm=4.0 + 2.0 * (seed % 3)).float()
        st.update(x=_image(n, n, seed), p=p, spec=_bytes(lib.pms_fft_spectrum_bytes(p)), out=_planes(n, n),
                  work=_bytes(max(lib.pms_fft_work_bytes(n, p), lib.pms_fft_work_bytes(p, p))))
        _lib.check(lib.pms_psf_spectrum(psf.data_ptr(), p, p, st["spec"].data_ptr(), st["work"].data_ptr(), None))
        torch.cuda.synchronize()
    elif kind == "detect":
        h, w, s = case["h"], case["w"], case["scales"]
        n = max(h, w)
        sky = _sky(n, seed, points=max(40, n * n // 4096))[:h, :w]
        img = sum(_smoothed(sky, k) for k in (0, 1)) + _noise((h, w), seed, 2e-3).double()
        st.update(x=_decomposed(img, s)[0].float().contiguous(), thr=_planes(s, dtype=torch.float64),
                  keep=_planes(s, h, w), ext=_planes(s, h, w), mask=_planes(s, h, w, dtype=torch.uint8),
                  work=_bytes(max(lib.pms_threshold_work_bytes(s, h, w), lib.pms_extract_work_bytes(s, h, w))))
    elif kind == "deconvolve":
        st["dirty"], st["psf"] = _pair(case["n"], seed, 2 if case["mode"] == "linear" else 1)
    else:
        rng = np.random.default_rng(seed)
        sides = [1024] * case["n1024"] + [512] * case["n512"] + [256] * case["n256"]
        pairs = [_pair(n, seed * 100 + i, fwhm=rng.uniform(3.0, 8.0)) for i, n in enumerate(sides)]
        kw = dict(CLEAN, scale_count=case["scales"], major_loop_miter=case["majors"])
        st["jobs"] = batch.DeviceJobs(pairs, [kw] * len(pairs))
    return st


def run(st):
    lib = _lib.lib()
    case, kind = st["case"], st["kind"]
    if kind == "transform":
        h, w, s = case["h"], case["w"], case["scales"]
        work = st["work"].data_ptr()
        _lib.check(lib.pms_iuwt_decompose(st["x"].data_ptr(), h, w, s, 0, st["detail"].data_ptr(),
                                          st["smooth"].data_ptr(), work, None))
        _lib.check(lib.pms_iuwt_recompose(st["detail"].data_ptr(), s, h, w, 0, st["smooth"].data_ptr(),
                                          st["out"].data_ptr(), work, None))
        return {"detail": st["detail"], "smooth": st["smooth"], "recomposed": st["out"]}
    if kind == "convolve":
        _lib.check(lib.pms_fft_convolve(st["x"].data_ptr(), case["n"], st["p"], st["spec"].data_ptr(),
                                        st["out"].data_ptr(), st["work"].data_ptr(), None))
        return {"out": st["out"]}
    if kind == "detect":
        h, w, s = case["h"], case["w"], case["scales"]
        x, thr, keep, work = (st[k].data_ptr() for k in ("x", "thr", "keep", "work"))
        _lib.check(lib.pms_estimate_threshold(x, s, h, w, case["edge_excl"], 0, thr, work, None))
        _lib.check(lib.pms_apply_threshold(x, s, h, w, thr, 4.0, keep, work, None))
        _lib.check(lib.pms_source_extraction(keep, s, h, w, 0.75, 0, st["ext"].data_ptr(), st["mask"].data_ptr(),
                                             None, work, None))
        return {"threshold": st["thr"], "significant": st["keep"], "extracted": st["ext"], "mask": st["mask"]}
    if kind == "deconvolve":
        img = DataImage(st["dirty"], st["psf"], None, 1.0, 1.0)
        kw = dict(CLEAN, major_loop_miter=case["majors"], conv_mode=case["mode"], precision=case["precision"])
        if case["by_scale"]:
            img.moresane_by_scale(start_scale=1, stop_scale=case["scales"], **kw)
        else:
            img.moresane(scale_count=case["scales"], **kw)
        return {"model": img.model, "residual": img.residual}
    jobs = st["jobs"]
    jobs.reset()
    batch.run_batch(jobs, n_workers=8, max_batch=32)
    return jobs.results()


def work(case):
    kind = case["kind"]
    if kind == "transform":  # each direction reads and writes the image and every plane once
        p = case["h"] * case["w"]
        return {"bytes": 4.0 * p * 2 * (case["scales"] + 2), "flops": 2.0 * p * case["scales"] * 30}
    if kind == "convolve":  # the image, the PSF's half spectrum, the result; two real transforms of the frame
        n = case["n"]
        p = 2 * n if case["mode"] == "linear" else n
        return {"bytes": 8.0 * n * n + 8.0 * p * (p // 2 + 1), "flops": 5.0 * p * p * 2 * np.log2(p)}
    if kind == "detect":  # the planes in; significant and extracted values and the mask out
        return {"bytes": 13.0 * case["h"] * case["w"] * case["scales"], "flops": 4.0 * case["h"] * case["w"] * case["scales"]}
    if kind == "deconvolve":
        sizes, rounds = [case["n"]], case["majors"]
    else:
        sizes = [256] * case["n256"] + [512] * case["n512"] + [1024] * case["n1024"]
        rounds = case["majors"]
    # a major iteration: detection and update once, and at least one minor iteration's convolution and transforms
    real = 8.0 if case.get("precision") == "float64" else 4.0
    planes = 2 * (case["scales"] + 2) + 3 * case["scales"] + 20
    return {"bytes": sum(rounds * real * n * n * planes for n in sizes),
            "flops": sum(rounds * n * n * (60.0 * case["scales"] + 40 * np.log2(2 * n)) for n in sizes)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "transform":
        planes, smooth = _decomposed(_image(case["h"], case["w"], seed), case["scales"])
        return {"detail": planes, "smooth": smooth, "recomposed": _recomposed(planes, smooth)}
    if kind == "convolve":
        n = case["n"]
        p = 2 * n if case["mode"] == "linear" else n
        return {"out": _convolved(_image(n, n, seed), _psf(p, fwhm=4.0 + 2.0 * (seed % 3)).float())}
    if kind == "detect":
        x = prepare(case, seed)["x"]
        e, (s, h, w) = case["edge_excl"], x.shape
        mags = x[:, e:h - e, e:w - e].abs().reshape(s, -1).double().sort(dim=1).values
        count = mags.shape[1]
        thr = 0.5 * (mags[:, (count - 1) // 2] + mags[:, count // 2]) / 0.6745
        significant = torch.where(x.double().abs() > 4.0 * thr[:, None, None], x.double(), torch.zeros((), device=DEVICE, dtype=torch.float64))
        return {"threshold": thr, "significant": significant, "extracted": None, "mask": None}
    return None  # a clean's trajectory has no short statement in 64 bits
