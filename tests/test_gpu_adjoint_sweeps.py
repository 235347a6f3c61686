"""Adjoint sweeps one after another in a context: each starts from empty grid
sums, whatever the one before it was (a field transpose, a sweep broken off after
a step, other adjoints), and gives what a fresh context gives.  Sums over
particles in another order: 1e-12 of the largest."""
import numpy as np
import pytest

from tests._model import gpu_model
from tests.test_gpu_adjoint import W

pytestmark = pytest.mark.gpu


def _ready(n):
    g = gpu_model(W, "fp64", n=n, seed=3)
    g.masset()
    g.set_sort_interval(0)
    g.run(2)
    g.findf(False)
    return g


def _sweep(g, lam):
    g.adj_set(lam)
    for _ in range(2):
        g.adj_step()
    return g.adj_get(), g.adj_get_par()


@pytest.mark.parametrize("n", [257, 20_000])
@pytest.mark.parametrize("before", ["field", "step", "seed"])
def test_sweep_starts_afresh(n, before):
    print("[case] sweeps", n, before, flush=True)
    rng = np.random.default_rng(n)
    lam = rng.standard_normal((4, n))
    ref, par = _sweep(_ready(n), lam)
    g = _ready(n)
    if before == "field":
        g.adj_field(1e6 * rng.standard_normal((2, g.mesh)))
    elif before == "step":
        g.adj_set(1e6 * rng.standard_normal((4, n)))
        g.adj_step()
    else:
        g.adj_seed_a2(1.0, 0.0, 50.0)
        g.adj_step()
    got, gpar = _sweep(g, lam)
    assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
    assert np.abs(np.subtract(gpar, par)).max() <= 1e-12 * max(np.abs(par).max(), 1.0)
