"""Walls from the mismatched edges backwards (walls.h), built for the host, against the depth-first
search of repair.h on every f-critical face: small and thin grids, where numbers of cells of different
kinds collide, heavy ties, and decompressed fields."""
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
    so = str(tmp_path_factory.mktemp("walls") / "libwallscheck.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I" + CSRC, "-o", so,
                           os.path.join(HERE, "native", "wallscheck.cpp")])
    L = ctypes.CDLL(so)
    for fn in (L.wc_check_f32, L.wc_check_f64):
        fn.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_int64] * 3 + [ctypes.c_void_p]
    return L


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_walls_equal_the_search(lib, dtype):
    total = np.zeros(4, np.int64)
    shapes = [(2, 2, 3), (2, 2, 9), (6, 2, 3), (2, 9, 4), (5, 4, 3), (7, 6, 5), (9, 12, 10), (13, 8, 16)]
    for k, shape in enumerate(shapes):
        for seed in range(6):
            rng = np.random.default_rng([seed, k])
            f = fields.gaussian_mixture(shape, 4, seed=seed, noise=0.02).astype(dtype)
            eps, _ = fields.eps_from_rel(f, 5e-2)
            one = f.copy()
            one.flat[rng.integers(f.size)] -= 0.01  # a few mismatches: long chains
            cases = [(f, fields.quantize(f, eps)), (f, one), (f, f.copy()),
                     (rng.standard_normal(shape).astype(dtype), rng.standard_normal(shape).astype(dtype)),
                     (rng.integers(0, 4, shape).astype(dtype), rng.integers(0, 3, shape).astype(dtype))]
            for a, b in cases:
                a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
                out = np.zeros(4, np.int64)
                fn = lib.wc_check_f32 if dtype == np.float32 else lib.wc_check_f64
                fn(a.ctypes.data, b.ctypes.data, shape[2], shape[1], shape[0], out.ctypes.data)
                assert out[3] == 0, (shape, seed, out)
                total += out
    assert total[0] > 5000 and total[2] > 500
