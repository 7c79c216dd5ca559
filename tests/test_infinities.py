"""Star codes of fields with infinities, built for the host. Infinities order like any other values, so
the codes are those of the field with each infinity replaced by a finite value beyond all others; a
+inf vertex at the grid's boundary must not be tied with neighbours that do not exist."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "dmtz_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("inf") / "libinfcheck.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I" + CSRC, "-o", so,
                           os.path.join(HERE, "native", "infcheck.cpp")])
    L = ctypes.CDLL(so)
    for fn in (L.ic_check_f32, L.ic_check_f64):
        fn.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_int64] * 3
        fn.restype = ctypes.c_int64
    return L


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(2, 2, 3), (3, 5, 4), (9, 8, 11)])
@pytest.mark.parametrize("share", [0.05, 0.5, 1.0])
def test_codes_of_infinite_values(lib, dtype, shape, share):
    nz, ny, nx = shape
    for seed in range(3):
        rng = np.random.default_rng(seed)
        f = rng.standard_normal(shape).astype(dtype)
        at = rng.random(shape) < share
        f[at] = rng.choice([np.inf, -np.inf], size=int(at.sum()))
        finite = np.ascontiguousarray(np.clip(f, -1e3, 1e3), dtype=dtype)
        fn = lib.ic_check_f32 if dtype == np.float32 else lib.ic_check_f64
        assert fn(f.ctypes.data, finite.ctypes.data, nx, ny, nz) == 0
