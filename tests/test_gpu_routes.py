"""The routes that a correction takes by the size of the grid and of its lists, each on small inputs.

Small grids re-evaluate every star after an edit, large ones only the stars around the edited vertices;
the dense classification runs a thread per vertex on small grids and over bit planes on large ones; short edit
sets are listed, long ones marked; ascending paths are listed unless they are too many; a large level of the
wall checks has a launch of its own. The sizes at which a route changes are the
context's (dmtz_amd/csrc/testing.h), so that these tests can move them:

  - the bit planes' codes, masks and tile counts against the thread per vertex, word for word, over
    ragged grids, 64-vertex steps that carry along one to three axes, ties, zeros of both signs,
    subnormals and infinities;
  - whole corrections over dirty lists, float32 and float64, bit-exact with the oracle, with edit sets
    listed and with edit sets marked;
  - separatrix checks that walk the ascending paths instead of listing them;
  - whole corrections of grids just above the sizes of the rules as they are, bit-exact with the oracle;
  - the wall lists with every level in a launch of its own, and with every level in one block;
  - the wall lists from a queue that has to grow, and without memory for one, where all walls are searched;
    the memory that a wall check keeps.
"""
import ctypes

import numpy as np
import pytest

import corpus
import dmtz_amd
from dmtz_amd import _native, fields

pytestmark = pytest.mark.gpu

NEVER = 1 << 32


class Limits:
    """The context's sizes within a with block; those not named stay the library's own."""
    NAMES = ("plane_min", "code_small", "target_dense", "path_steps", "wall_level", "wall_queue")

    def __init__(self, ctx, **values):
        assert set(values) <= set(self.NAMES)
        self.ctx, self.values = ctx, [values.get(n, -1) for n in self.NAMES]

    def _set(self, values):
        fn = _native.lib().dmtz_testing_limits
        fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
        fn.restype = None
        fn(self.ctx.handle, (ctypes.c_int64 * len(values))(*values))

    def __enter__(self):
        self._set(self.values)

    def __exit__(self, *a):
        self._set([-1] * len(self.NAMES))


def _state(ctx, n):
    """What the last call left on the device: star codes, f-critical and mismatch masks, tile counts."""
    out = [np.zeros(4 * n, np.uint64), np.zeros(4 * n, np.uint64), np.zeros(n, np.uint64), np.zeros(n, np.uint32),
           np.zeros(n, np.uint64), np.zeros(n, np.uint32), np.zeros((n + 2047) // 2048, np.uint32)]
    fn = _native.lib().dmtz_testing_state
    fn.argtypes = [ctypes.c_void_p, ctypes.c_int64] + [ctypes.c_void_p] * 7
    fn.restype = ctypes.c_int
    assert fn(ctx.handle, n, *[a.ctypes.data for a in out]) == 0
    return dict(zip(("code_f", "code_g", "critf_lo", "critf_hi", "mm_lo", "mm_hi", "tile_nz"), out))


def _plane_fields(shape, dtype, rng):
    """(name, f, g) pairs."""
    tiny = np.finfo(dtype).smallest_subnormal
    rand = lambda: rng.standard_normal(shape).astype(dtype)  # noqa: E731
    yield "random", rand(), rand()
    yield "ties", rng.integers(0, 3, shape).astype(dtype), rng.integers(0, 2, shape).astype(dtype)
    yield "zeros", np.where(rng.random(shape) < 0.5, -0.0, 0.0).astype(dtype), np.zeros(shape, dtype)
    yield "subnormals", (rng.integers(-2, 3, shape).astype(dtype) * tiny).astype(dtype), rand()
    yield "large", (rng.integers(-2, 3, shape) * (np.finfo(dtype).max / 2)).astype(dtype), rand()
    f, g = rng.integers(0, 5, shape).astype(dtype), rng.integers(0, 5, shape).astype(dtype)
    for a in (f, g):
        at = rng.random(shape) < 0.1
        a[at] = rng.choice([np.inf, -np.inf], size=int(at.sum()))
    yield "infinities", f, g


PLANE_SHAPES = [(2, 2, 3), (700, 2, 3), (2, 350, 3), (9, 21, 13), (3, 11, 64), (5, 7, 65), (2, 3, 500), (8, 16, 16),
                (87500, 2, 3), (41, 113, 127)]  # the last two are above the library's own size


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", PLANE_SHAPES, ids=["x".join(map(str, s)) for s in PLANE_SHAPES])
def test_planes_equal_a_thread_per_vertex(dev, dtype, shape):
    n = int(np.prod(shape))
    own = -1 if n >= 1 << 19 else 0
    for name, f, g in _plane_fields(shape, dtype, np.random.default_rng(11)):
        print("planes", shape, dtype.__name__, name, flush=True)
        with Limits(dev, plane_min=own):
            t0, c0 = dmtz_amd.targets(f, g, 1.0, 10.0, dmtz_amd.CorrectionFlags(), ctx=dev)
            a = _state(dev, n)
        with Limits(dev, plane_min=NEVER):
            t1, c1 = dmtz_amd.targets(f, g, 1.0, 10.0, dmtz_amd.CorrectionFlags(), ctx=dev)
            b = _state(dev, n)
        for key in a:
            assert np.array_equal(a[key], b[key]), (name, key, np.nonzero(a[key] != b[key])[0][:5])
        assert c0 == c1 and np.array_equal(t0, t1)
        nz = np.zeros(((n + 2047) // 2048) * 2048, bool)
        nz[:n] = (a["mm_lo"] != 0) | (a["mm_hi"] != 0)
        assert np.array_equal(a["tile_nz"], nz.reshape(-1, 2048).sum(1))


def _compare_run(oracle, dev, f, g, eps, rng, fl):
    want = oracle.correct(f, g, eps, rng, oracle.flags(**fl))
    got = dmtz_amd.correct(f, g, eps, rng, dmtz_amd.CorrectionFlags(**fl), ctx=dev, return_counter=True)
    assert got.status == want["status"]
    assert got.sweeps == want["sweeps"] and got.counts == want["counts"]
    assert (got.trajectory == want["traj"]).all()
    assert (got.counter == want["counter"]).all()
    assert got.g.tobytes() == want["g"].tobytes()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("planes,marks", [(0, 0), (NEVER, 0), (NEVER, NEVER)], ids=["planes", "listed", "marked"])
@pytest.mark.parametrize("name,fl", corpus.FLAG_CASES, ids=[c[0] for c in corpus.FLAG_CASES])
def test_corrections_over_dirty_lists(oracle, dev, dtype, planes, marks, name, fl):
    for inp, f, g, eps, rng in corpus.gm_inputs() + corpus.fbm_inputs():
        print("lists", name, inp, f.shape, dtype.__name__, flush=True)
        with Limits(dev, plane_min=planes, code_small=0, target_dense=marks):
            _compare_run(oracle, dev, f.astype(dtype), g.astype(dtype), eps, rng, fl)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("name,fl", corpus.WALL_CASES, ids=[c[0] for c in corpus.WALL_CASES])
def test_wall_corrections_over_dirty_lists(oracle, dev, dtype, name, fl):
    for inp, f, g, eps, rng in corpus.gm_inputs():
        print("lists", name, inp, f.shape, dtype.__name__, flush=True)
        with Limits(dev, code_small=0):
            _compare_run(oracle, dev, f.astype(dtype), g.astype(dtype), eps, rng, dict(fl, max_sweeps=300))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_geometry_checks_that_walk(oracle, dev, dtype):
    fl = dict(preserve_vpath=1, preserve_geometry=1)
    for name, f, g, eps, rng in corpus.path_inputs(oracle):
        f, g = f.astype(dtype), g.astype(dtype)
        print("walked", name, dtype.__name__, flush=True)
        want = oracle.paths(f, g, oracle.flags(**fl))
        with Limits(dev, path_steps=0):
            got = dmtz_amd.paths(f, g, dmtz_amd.CorrectionFlags(**fl), ctx=dev)
            for a, b in (("ds", "ds_rec"), ("as_", "as_rec")):
                assert sorted(zip(got[a].tolist(), got[b].tolist())) == sorted(zip(want[a].tolist(), want[b].tolist()))
            _compare_run(oracle, dev, f, g, eps, rng, fl)


@pytest.mark.timeout(300)
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape,mode", [((41, 43, 45), "geometry"), ((41, 43, 45), "connectivity"),
                                        ((41, 43, 45), "walls"), ((2, 180, 200), "geometry"),
                                        ((2, 180, 200), "walls"), ((64, 91, 97), "geometry")])
def test_corrections_above_the_rules_sizes(oracle, dev, dtype, shape, mode):
    """79 335 and 72 000 vertices: dirty lists; 564 928: bit planes."""
    fl = dict(preserve_vpath=1, preserve_geometry=int(mode != "connectivity"), preserve_connectors=int(mode == "walls"),
              max_sweeps=40)
    f = fields.gaussian_mixture(shape, 8, seed=3, noise=0.01).astype(dtype)
    eps, rng = fields.eps_from_rel(f, 1e-3)
    print("above", shape, dtype.__name__, mode, flush=True)
    _compare_run(oracle, dev, f, fields.quantize(f, eps), eps, rng, fl)


def _wall_set(r):
    return sorted(zip(r["face"].tolist(), r["edge"].tolist()))


def test_wall_levels(oracle, dev):
    fl = oracle.flags(preserve_vpath=1, preserve_geometry=1, preserve_connectors=1)
    for name, f, g, eps, rng in corpus.wall_inputs(oracle):
        print("wall levels", name, f.shape, flush=True)
        want = oracle.paths(f, g, fl)
        want = sorted(zip(want["wall"].tolist(), want["wall_rec"].tolist()))
        for level in (1, NEVER):
            with Limits(dev, wall_level=level):
                assert _wall_set(dmtz_amd.walls(f, g, eps, rng, ctx=dev)) == want
    # levels above the library's own size, and all of them in one block
    r = np.random.default_rng(6)
    f = r.standard_normal((40, 41, 42)).astype(np.float32)
    g = (f + 0.3 * r.standard_normal(f.shape)).astype(np.float32)
    print("wall levels", f.shape, flush=True)
    want = oracle.paths(f, g, fl)
    want = sorted(zip(want["wall"].tolist(), want["wall_rec"].tolist()))
    assert len(want) > 16384
    for level in (-1, NEVER):
        with Limits(dev, wall_level=level):
            assert _wall_set(dmtz_amd.walls(f, g, 1.0, 1.0, ctx=dev)) == want


def _wall_pairs():
    """Noise, whose mismatched edges open most faces; a smooth field with a few vertices lowered, whose walls
    are large: some outgrow the first two tiers of the search's visited sets."""
    r = np.random.default_rng(6)
    f = r.standard_normal((40, 41, 42)).astype(np.float32)
    yield "noise", f, (f + 0.3 * r.standard_normal(f.shape)).astype(np.float32)
    f = fields.gaussian_mixture((64, 60, 62), 6, seed=2, noise=0.0)
    g = f.copy()
    g.flat[r.integers(0, f.size, 40)] -= np.float32(0.05)
    yield "smooth", f, g


@pytest.mark.parametrize("level", [-1, 1, NEVER])
@pytest.mark.parametrize("queue", [1, 1 << 60], ids=["grows", "no_memory"])
def test_wall_queue(oracle, queue, level):
    fl = oracle.flags(preserve_vpath=1, preserve_geometry=1, preserve_connectors=1)
    with dmtz_amd.Context(0) as ctx:  # a context of its own: a queue is kept once it has grown
        for name, f, g in _wall_pairs():
            print("wall queue", queue, level, name, flush=True)
            want = oracle.paths(f, g, fl)
            want = sorted(zip(want["wall"].tolist(), want["wall_rec"].tolist()))
            assert len(want) > 0
            with Limits(ctx, wall_queue=queue, wall_level=level):
                for _ in range(2):
                    assert _wall_set(dmtz_amd.walls(f, g, 1.0, 1.0, ctx=ctx)) == want
            assert ctx.error() == ""  # the search is no error


def test_wall_memory():
    """A check that opens few faces keeps at most 16 bytes a vertex for them, not room for all 12 faces."""
    import torch

    f = fields.fbm((160, 160, 160), seed=3)
    eps, rng = fields.eps_from_rel(f, 1e-3)
    fl = dmtz_amd.CorrectionFlags(preserve_vpath=1, preserve_geometry=1, max_sweeps=200)
    with dmtz_amd.Context(0) as ctx:
        g = dmtz_amd.correct(f, fields.quantize(f, eps), eps, rng, fl, ctx=ctx).g
        dmtz_amd.paths(f, g, dmtz_amd.CorrectionFlags(preserve_geometry=0), ctx=ctx)  # what the checks share
        free = torch.cuda.mem_get_info()[0]
        print("wall memory", f.shape, flush=True)
        assert len(dmtz_amd.walls(f, g, eps, rng, fl, ctx=ctx)["face"]) > 0
        kept = free - torch.cuda.mem_get_info()[0]
        print("kept", kept / f.size, "bytes a vertex", flush=True)
        assert kept <= 16 * f.size
