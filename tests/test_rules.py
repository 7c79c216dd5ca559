"""The repair rules in vertex frames (rules.h), built for the host, against the rules over global ids
(repair.h) on every mismatched cell: the same edit set, or the record is handed to the general rule
with nothing emitted. Small and thin grids, where the numbers of cells of different kinds collide,
and fields with heavy ties are among the inputs."""
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
    so = str(tmp_path_factory.mktemp("rules") / "librulescheck.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I" + CSRC, "-o", so,
                           os.path.join(HERE, "native", "rulescheck.cpp")])
    L = ctypes.CDLL(so)
    for fn in (L.rc_check_f32, L.rc_check_f64):
        fn.argtypes = ([ctypes.c_void_p] * 2 + [ctypes.c_int64] * 3 + [ctypes.c_double, ctypes.c_int]
                       + [ctypes.c_void_p] * 2)
    return L


def run(lib, f, g, eps, edit_type, seed):
    f, g = np.ascontiguousarray(f), np.ascontiguousarray(g)
    counter = np.random.default_rng(seed).integers(1, 7, f.size).astype(np.uint8)
    out = np.zeros(3, np.int64)
    nz, ny, nx = f.shape
    fn = lib.rc_check_f32 if f.dtype == np.float32 else lib.rc_check_f64
    fn(f.ctypes.data, g.ctypes.data, nx, ny, nz, eps, edit_type, counter.ctypes.data, out.ctypes.data)
    return out


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("edit_type", [0, 1])
def test_rules_equal_the_general_rules(lib, dtype, edit_type):
    total = np.zeros(3, np.int64)
    shapes = [(2, 2, 3), (2, 2, 9), (6, 2, 3), (2, 9, 4), (5, 4, 3), (7, 6, 5), (9, 12, 10), (13, 8, 16)]
    for k, shape in enumerate(shapes):
        for seed in range(6):
            rng = np.random.default_rng([seed, k])
            f = fields.gaussian_mixture(shape, 4, seed=seed, noise=0.05).astype(dtype)
            eps, _ = fields.eps_from_rel(f, 5e-2)
            cases = [(f, fields.quantize(f, eps)),  # a decompressed field
                     (rng.standard_normal(shape).astype(dtype), rng.standard_normal(shape).astype(dtype)),
                     (rng.integers(0, 4, shape).astype(dtype), rng.integers(0, 3, shape).astype(dtype))]
            for a, b in cases:
                r = run(lib, a, b, eps, edit_type, seed)
                assert r[2] == 0, (shape, seed, r)
                total += r
    assert total[0] > 50000 and total[1] > 0  # the collisions are reached
