"""Loads and unloads of particles: plain and staged copies (16 MiB in all),
zones checked on the host or the device (131072 particles), every grid type."""
import ctypes as C
import threading

import numpy as np
import pytest

from galaxy_amd import GalhipError
from galaxy_amd.lib15 import P2DEnsemble, P2DGrid, P3DGrid

pytestmark = pytest.mark.gpu

# plain / device check / staged from 838861 FP32 particles / several rounds of the chunks
SIZES = [1, 131071, 131072, 838860, 838861, 1500007]


def _grid(precision="fp32"):
    return P2DGrid(60, 128, hash_=1, softl=2.0, nzones=2, nstep=(1, 2), zbr=(0.0, 5.0), pmass=1e-7,
                   precision=precision)


def _set(n, dtype, seed, cols=4):
    rng = np.random.default_rng(seed)
    a = [(rng.random(n) * 6 - 3).astype(dtype) for _ in range(cols)]
    return a + [rng.integers(1, 4, n).astype(np.int32)]


def _same(out, ref, names):
    for k, v in zip(names, ref):
        np.testing.assert_array_equal(out[k], v)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n", SIZES)
def test_round_trip(n, precision):
    g = _grid(precision)
    ref = _set(n, g.dtype, n)
    for _ in range(2):                       # the kept buffer the second time
        g.restrt(*ref)
        _same(g.unload(), ref, ("x", "y", "vx", "vy", "iz"))
        assert g.noff == int((ref[4] == 3).sum())


@pytest.mark.parametrize("n", [131073, 700001])
def test_round_trip_p3d(n):
    g = P3DGrid(20, 32, 11, dzg=0.5, hash_=1, softl=3.0, nzones=2, nstep=(1, 2), zbr=(0.0, 5.0),
                pmass=1e-7)
    ref = _set(n, g.dtype, n, 6)
    g.restrt(*ref)
    _same(g.unload(), ref, ("x", "y", "z", "vx", "vy", "vz", "iz"))


@pytest.mark.parametrize("counts", [(3, 0, 100), (0, 131072, 5, 900000), (70001, 70002, 0)])
def test_round_trip_ensemble(counts):
    e = P2DEnsemble(len(counts), 60, 128, hash_=1, softl=2.0, nzones=1, pmass=[1e-6] * len(counts))
    mem = [_set(k, e.dtype, k + 1) for k in counts]
    for m in mem:
        m[4] = np.minimum(m[4], 2)
    e.restrt(mem)
    for o, m, k in zip(e.unload(), mem, range(len(counts))):
        _same(o, m, ("x", "y", "vx", "vy", "iz"))
    assert list(e.noff) == [int((m[4] == 2).sum()) for m in mem]


@pytest.mark.parametrize("n", [1000, 131072, 1500007])
def test_bad_zone(n):
    g = _grid()
    ref = _set(n, g.dtype, 5)
    g.restrt(*ref)
    bad = ref[4].copy()
    bad[[n // 2, n - 1]] = (0, 260)
    with pytest.raises(GalhipError, match="particle %d has zone 0 outside 1..3" % (n // 2)):
        g.restrt(*ref[:4], bad)
    _same(g.unload(), ref, ("x", "y", "vx", "vy", "iz"))


def test_some_columns():
    n = 1500007
    g = _grid()
    ref = _set(n, g.dtype, 6)
    g.restrt(*ref)
    y, iz = np.empty(n, np.float32), np.empty(n, np.int32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    assert g._lib.galhip_unload(g._h, None, p(y), None, None, p(iz)) == 0
    np.testing.assert_array_equal(y, ref[1])
    np.testing.assert_array_equal(iz, ref[4])


def test_threads():
    bad = []

    def work(seed):
        g = _grid()
        for k in range(3):
            ref = _set(900000 + 1000 * seed, g.dtype, seed + k)
            g.restrt(*ref)
            out = g.unload()
            if not all((out[q] == r).all() for q, r in zip(("x", "y", "vx", "vy", "iz"), ref)):
                bad.append((seed, k))
        g.close()

    ts = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
