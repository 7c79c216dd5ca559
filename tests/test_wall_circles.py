"""2-saddle walls whose chain of open faces (walls.h) runs in a circle: small fields in which a vertex and a
face, and an edge and a tet, share their numbers, found among random ones (one chain in 150 thousand).
Such a chain has to be given up after a few steps and its face searched instead."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "dmtz_amd", "csrc")

# (nz, ny, nx), f, g
CIRCLES = [
    ((2, 3, 3),
     [13, 4, 17, 9, 14, 11, 2, 6, 7, 0, 16, 3, 8, 10, 15, 1, 12, 5],
     [14, 1, 7, 3, 13, 11, 2, 6, 9, 17, 16, 0, 10, 8, 15, 5, 12, 4]),
    ((2, 3, 3),
     [1, 16, 17, 0, 12, 4, 15, 8, 14, 6, 13, 3, 10, 7, 9, 2, 11, 5],
     [13, 11, 6, 8, 12, 4, 15, 1, 0, 17, 14, 3, 10, 9, 7, 2, 16, 5]),
    ((2, 3, 3),
     [2, 1, 2, 0, 2, 2, 1, 3, 2, 3, 2, 0, 1, 2, 2, 1, 2, 0],
     [2, 1, 1, 0, 2, 2, 1, 3, 2, 3, 2, 0, 2, 2, 2, 1, 2, 0]),
    ((4, 2, 3),
     [4, 12, 21, 16, 23, 5, 20, 13, 8, 17, 6, 0, 7, 22, 14, 18, 3, 9, 10, 2, 1, 11, 19, 15],
     [4, 21, 12, 16, 23, 5, 20, 13, 8, 17, 6, 0, 7, 22, 14, 18, 3, 9, 10, 2, 1, 11, 19, 15]),
    ((2, 4, 3),
     [0, 15, 8, 23, 1, 6, 10, 18, 5, 20, 12, 4, 21, 7, 14, 22, 11, 3, 19, 2, 13, 17, 9, 16],
     [0, 15, 9, 23, 1, 6, 10, 19, 5, 20, 12, 2, 21, 7, 14, 22, 11, 3, 18, 4, 13, 17, 8, 16]),
    ((2, 4, 3),
     [3, 2, 0, 1, 0, 2, 2, 2, 2, 2, 1, 0, 3, 1, 2, 1, 1, 1, 1, 1, 2, 0, 1, 1],
     [3, 2, 0, 1, 0, 2, 2, 2, 2, 2, 1, 0, 3, 1, 2, 1, 0, 1, 1, 1, 2, 1, 1, 1]),
    ((2, 6, 3),
     [12, 28, 27, 8, 7, 4, 26, 20, 3, 23, 5, 29, 1, 11, 31, 13, 22, 25, 34, 35, 0, 16, 18, 30, 32, 21, 2, 6, 24, 19, 14, 15, 17, 10, 33, 9],
     [15, 28, 12, 8, 7, 4, 26, 20, 34, 23, 5, 29, 1, 11, 31, 13, 22, 25, 3, 35, 0, 16, 18, 30, 32, 21, 2, 6, 24, 19, 14, 27, 17, 10, 33, 9]),
    ((2, 6, 3),
     [29, 6, 16, 28, 5, 25, 22, 31, 21, 15, 27, 12, 30, 14, 0, 32, 19, 11, 8, 4, 17, 3, 35, 33, 26, 1, 24, 20, 10, 2, 13, 23, 7, 34, 9, 18],
     [21, 27, 16, 28, 2, 25, 10, 31, 29, 8, 6, 5, 30, 7, 20, 33, 15, 11, 19, 0, 17, 3, 35, 13, 26, 1, 34, 24, 4, 12, 32, 23, 14, 22, 9, 18]),
]


def pairs(dtype):
    for shape, f, g in CIRCLES:
        yield np.array(f, dtype).reshape(shape), np.array(g, dtype).reshape(shape)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("circles") / "libcirclecheck.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I" + CSRC, "-o", so,
                           os.path.join(HERE, "native", "circlecheck.cpp")])
    L = ctypes.CDLL(so)
    for fn in (L.wc_follow_f32, L.wc_follow_f64):
        fn.argtypes = [ctypes.c_void_p] * 2 + [ctypes.c_int64] * 3 + [ctypes.c_void_p]
    return L


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_circles_are_given_up(lib, dtype):
    for f, g in pairs(dtype):
        out = np.zeros(4, np.int64)
        fn = lib.wc_follow_f32 if dtype == np.float32 else lib.wc_follow_f64
        fn(f.ctypes.data, g.ctypes.data, f.shape[2], f.shape[1], f.shape[0], out.ctypes.data)
        chains, circles, steps, wrong = out.tolist()
        assert wrong == 0 and chains >= circles > 0
        # a circle of at most all faces (fewer than 12 per vertex) is found within four times its length
        assert steps <= 48 * f.size


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_circles_are_searched_on_the_gpu(oracle, dev, dtype):
    import dmtz_amd

    for k, (f, g) in enumerate(pairs(dtype)):
        print("circle", k, f.shape, f.dtype, flush=True)
        fl = dict(preserve_vpath=1, preserve_geometry=1, preserve_connectors=1)
        want = oracle.paths(f, g, oracle.flags(**fl))
        got = dmtz_amd.walls(f, g, 100.0, 100.0, dmtz_amd.CorrectionFlags(), ctx=dev, with_targets=True)
        assert sorted(zip(got["face"].tolist(), got["edge"].tolist())) == \
            sorted(zip(want["wall"].tolist(), want["wall_rec"].tolist()))
        assert len(got["face"]) > 0
        want_t, n = oracle.wall_targets(f, g, 100.0, 100.0, oracle.flags(**fl))
        assert n == len(got["face"])
        assert (got["targets"] == want_t).all()
