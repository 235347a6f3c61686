"""The push count of galhip_get_profile: every push launched since profiling
was enabled, over particle counts about a block's and a context's stripes,
started again by a load, and not taken back when a recorded state is."""
import numpy as np
import pytest

from galaxy_amd.lib15 import P2DEnsemble, P2DGrid, P3DGrid

pytestmark = pytest.mark.gpu


def _ring(n, dim, dtype):
    """n particles at rest on a ring well inside the grid."""
    a = 2 * np.pi * np.arange(n) / max(n, 1)
    p = [2 * np.cos(a), 2 * np.sin(a)] + [np.zeros(n)] * (2 * dim - 2)
    return [v.astype(dtype) for v in p] + [np.ones(n, np.int32)]


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 257, 70_001])
def test_load_starts_the_count(n, dim, prec):
    print("[case] push count", n, dim, prec, flush=True)
    if dim == 2:
        g = P2DGrid(60, 128, hash_=1, softl=2.0, pmass=1e-9, precision=prec)
    else:
        g = P3DGrid(20, 32, 11, dzg=0.5, hash_=1, softl=3.0, pmass=1e-9, precision=prec)
    g.greenm()
    for k in (2, 3):
        g.restrt(*_ring(n, dim, g.dtype))
        g.masset()
        g.set_profile(True)
        g.run(k)
        assert g.get_profile()[1:] == (k, k * n)
        g.run(1)
        assert g.get_profile()[1:] == (k + 1, (k + 1) * n)
        g.set_profile(False)


def test_ensemble_load():
    n = [5, 0, 3000]
    e = P2DEnsemble(3, 60, 128, hash_=1, softl=2.0, pmass=[1e-9] * 3)
    e.greenm()
    for k in (1, 4):
        e.restrt([_ring(m, 2, e.dtype) for m in n])
        e.masset()
        e.set_profile(True)
        e.run(k)
        assert e.get_profile()[1:] == (k, k * sum(n))
        e.set_profile(False)


def test_restored_state_keeps_the_count():
    n = 500
    g = P2DGrid(60, 128, hash_=1, softl=2.0, pmass=1e-9)
    g.greenm()
    g.restrt(*_ring(n, 2, g.dtype))
    g.masset()
    g.adj_record(0)
    g.set_profile(True)
    g.run(3)
    g.adj_restore(0)
    assert g.get_profile()[1:] == (3, 3 * n)
    g.run(2)
    assert g.get_profile()[1:] == (5, 5 * n)
