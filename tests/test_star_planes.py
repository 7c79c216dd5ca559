"""The bit-plane classifier (star_planes.h), built for the host, against the classifier of one vertex
(lower_star.h): star codes, critical and member masks of every vertex."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from dmtz_amd import fields

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "dmtz_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("planes") / "libplanescheck.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I" + CSRC, "-o", so,
                           os.path.join(HERE, "native", "planescheck.cpp")])
    L = ctypes.CDLL(so)
    for fn in (L.sp_check_f32, L.sp_check_f64):
        fn.argtypes = [ctypes.c_void_p] + [ctypes.c_int64] * 3
        fn.restype = ctypes.c_int64
    return L


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(2, 2, 3), (3, 5, 4), (17, 19, 23), (2, 40, 33)])
def test_planes_equal_the_single_star(lib, dtype, shape):
    fn = lib.sp_check_f32 if dtype == np.float32 else lib.sp_check_f64
    nz, ny, nx = shape
    for seed in range(3):
        rng = np.random.default_rng(seed)
        cases = [fields.gaussian_mixture(shape, 3, seed=seed, noise=0.05), rng.standard_normal(shape),
                 rng.integers(0, 3, shape), rng.integers(0, 2, shape) * 1e30, np.zeros(shape),
                 np.where(rng.random(shape) < 0.5, -0.0, 0.0), rng.integers(-2, 3, shape) * 5e-324]  # -0, subnormals
        for f in cases:
            tiny = dtype == np.float32 and np.abs(f).max() < 1e-300 and f.any()
            f = np.ascontiguousarray(f / 5e-324 * 1.4e-45 if tiny else f, dtype=dtype)
            assert fn(f.ctypes.data, nx, ny, nz) == 0
