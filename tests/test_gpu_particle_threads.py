"""Loads, unloads and closes of contexts in several threads at once, which share
the pinned chunks of staged copies: every thread's own error or wrong value fails
the test, and every round of every thread has to have been done."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from galaxy_amd.lib15 import P2DGrid

pytestmark = pytest.mark.gpu
THREADS, ROUNDS = 4, 3


def _work(seed):
    done = 0
    for k in range(ROUNDS):
        g = P2DGrid(60, 128, hash_=1, softl=2.0, nzones=2, nstep=(1, 2), zbr=(0.0, 5.0), pmass=1e-7)
        rng = np.random.default_rng(10 * seed + k)
        n = 900_000 + 1000 * seed
        ref = [(rng.random(n) * 6 - 3).astype(g.dtype) for _ in range(4)]
        ref.append(rng.integers(1, 4, n).astype(np.int32))
        g.restrt(*ref)
        out = g.unload()
        for q, r in zip(("x", "y", "vx", "vy", "iz"), ref):
            np.testing.assert_array_equal(out[q], r)
        g.close()
        done += 1
    return done


def test_threads():
    with ThreadPoolExecutor(THREADS) as ex:
        done = [f.result() for f in [ex.submit(_work, s) for s in range(THREADS)]]
    assert done == [ROUNDS] * THREADS
