"""The tiles of the bit-plane classifier (star_planes.h tile_words), built for the host, against the
classifier of one vertex: grids whose 64-vertex steps carry along one, two and three axes, ragged last
tiles, and fields with ties, infinities and NaN among their values."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "dmtz_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("tiles") / "libtilecheck.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I" + CSRC, "-o", so,
                           os.path.join(HERE, "native", "tilecheck.cpp")])
    L = ctypes.CDLL(so)
    for fn in (L.tc_check_f32, L.tc_check_f64):
        fn.argtypes = [ctypes.c_void_p] + [ctypes.c_int64] * 3
        fn.restype = ctypes.c_int64
    return L


def _fields(shape, dtype, rng):
    yield rng.standard_normal(shape).astype(dtype)
    yield rng.integers(0, 3, shape).astype(dtype)
    for values in ([np.inf, -np.inf], [np.inf, -np.inf, np.nan, -np.nan]):
        for share in (0.02, 0.6):
            f = rng.integers(0, 5, shape).astype(dtype)
            at = rng.random(shape) < share
            f[at] = rng.choice(values, size=int(at.sum()))
            yield f
    yield np.full(shape, np.inf, dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(2, 2, 3), (700, 2, 3), (2, 350, 3), (9, 21, 13), (3, 11, 64), (5, 7, 65), (2, 3, 500),
                                   (8, 16, 16)])
def test_tiles_equal_the_single_star(lib, dtype, shape):
    fn = lib.tc_check_f32 if dtype == np.float32 else lib.tc_check_f64
    nz, ny, nx = shape
    for f in _fields(shape, dtype, np.random.default_rng(5)):
        assert fn(np.ascontiguousarray(f).ctypes.data, nx, ny, nz) == 0
