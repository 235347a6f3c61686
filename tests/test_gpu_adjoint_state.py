"""adj_record / adj_restore: the state's arrays in one launch, at sizes whose
bytes are and are not multiples of 16 and about a block's chunk; the adjoints
carried over a change of the storage order."""
import numpy as np
import pytest

from tests._model import gpu_model
from tests.test_gpu_adjoint import W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 1023, 4096, 4097, 70_001])
def test_record_restore(n, precision):
    g = gpu_model(W, precision, n=n, seed=3)
    g.masset()
    g.set_sort_interval(2)
    g.run(3)
    ref, mass, order = g.unload(), g.get_mass(), g.get_order()
    g.adj_record(2)
    g.run(5)
    last, lmass = g.unload(), g.get_mass()
    for _ in range(2):
        g.adj_restore(2)
        for k, v in g.unload().items():
            np.testing.assert_array_equal(v, ref[k])
        for a, b in zip(g.get_mass(), mass):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(g.get_order(), order)
        g.set_sort_interval(0)
        g.run(5)
        for k, v in g.unload().items():
            np.testing.assert_array_equal(v, last[k])
        for a, b in zip(g.get_mass(), lmass):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n", [1, 257, 70_001])
def test_adjoints_follow_the_order(n):
    """An adjoint step after a re-sort gives the adjoints of the step without
    it: each particle's are its own (sums over particles in another order:
    1e-12 of the largest)."""
    rng = np.random.default_rng(n)
    lam = rng.standard_normal((4, n))
    got = []
    for sort in (False, True):
        g = gpu_model(W, "fp64", n=n, seed=3)
        g.masset()
        g.set_sort_interval(0)
        g.run(4)
        g.adj_set(lam)
        if sort:
            g.sort()
        g.findf(False)
        g.adj_step()
        got.append(g.adj_get())
    assert np.abs(got[0] - got[1]).max() <= 1e-12 * np.abs(got[0]).max()
