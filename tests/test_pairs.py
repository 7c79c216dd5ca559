"""Pair words (pairs.h), built for the host: every tet's and vertex's pairing, the tet across every
paired face, the start tets of every triangle, and the ascending and descending walks, against the
pairing lookups and walks of gradient.h and repair.h."""
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
    so = str(tmp_path_factory.mktemp("pairs") / "libpairscheck.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I" + CSRC, "-o", so,
                           os.path.join(HERE, "native", "pairscheck.cpp")])
    L = ctypes.CDLL(so)
    for fn in (L.pc_check_f32, L.pc_check_f64):
        fn.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_int64] * 3
        fn.restype = ctypes.c_int64
    return L


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(2, 2, 3), (2, 7, 5), (9, 2, 4), (8, 9, 10), (5, 12, 7)])
def test_pair_words_equal_the_lookups(lib, dtype, shape):
    rng = np.random.default_rng(3)
    f = fields.gaussian_mixture(shape, 4, seed=1, noise=0.05).astype(dtype)
    eps, _ = fields.eps_from_rel(f, 3e-2)
    pairs = [(f, fields.quantize(f, eps)), (f, rng.standard_normal(shape).astype(dtype))]
    pairs.append((rng.integers(0, 3, shape).astype(dtype), rng.integers(0, 2, shape).astype(dtype)))  # heavy ties
    pairs.append((np.zeros(shape, dtype), -np.arange(f.size, dtype=dtype).reshape(shape)))
    fn = lib.pc_check_f32 if dtype == np.float32 else lib.pc_check_f64
    nz, ny, nx = shape
    for a, b in pairs:
        a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
        assert fn(a.ctypes.data, b.ctypes.data, nx, ny, nz) == 0
