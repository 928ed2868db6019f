"""The device bytes that a served request reserves while it runs (no GPU).

A server refuses a request whose footprint exceeds its budget, so what a job holds must not grow: the bytes here
are those of the job's planes, spectra and scratch when a noise estimate's scratch was 131,584 bytes.
"""

import ctypes

import pytest

from pymoresane_amd import _lib


class Geometry(ctypes.Structure):  # pms::Geometry
    _fields_ = [(k, ctypes.c_int) for k in ("n", "psf_n", "sub", "S", "lo")]
    _fields_ += [("linear", ctypes.c_bool), ("double_psf", ctypes.c_bool)]
    _fields_ += [("p_sub", ctypes.c_int), ("p_full", ctypes.c_int), ("f64", ctypes.c_bool)]


@pytest.mark.parametrize("n,precision,held", [
    (16, 0, 374016), (64, 0, 1305856), (64, 1, 2201856), (128, 1, 8274176), (256, 0, 18522368), (256, 1, 34320640),
    (512, 0, 78508288), (512, 1, 145740032), (1000, 0, 298442944), (1024, 0, 334958848), (1024, 1, 620515584),
    (2048, 0, 1426673920), (4096, 0, 6057451776), (4096, 1, 11163455744)])
def test_a_job_holds_no_more_than_it_did(n, precision, held):
    lib = _lib.load()
    geometry = lib._ZN3pms13make_geometryEiiRK19pms_moresane_paramsiPi
    geometry.restype = Geometry
    footprint = lib._ZN3pms19job_footprint_bytesERKNS_8GeometryE
    footprint.restype = ctypes.c_size_t
    prm = _lib.MoresaneParams()
    prm.n, prm.psf_n, prm.precision, prm.conv_mode = n, 2 * n, precision, 0
    g = geometry(n, 2 * n, ctypes.byref(prm), 0, None)
    assert footprint(ctypes.byref(g)) <= held
