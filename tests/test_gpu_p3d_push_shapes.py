"""The 3-D push and mass assignment where their launch shape changes: the
quadratic scheme's blocks of 256 particles, the linear scheme's of 512, and two
particles per thread above 5e6 in FP32.

Small counts against the oracle, bit-exact in FP32 as in test_gpu_p3d.py.  The
large count: 5e6 particles (one per thread) and the same with one more off the
grid (two per thread) are the same disc, with the same fixed-point scale, so every
result is the same bits."""
import numpy as np
import pytest

from galaxy_amd import configs
from galaxy_amd.lib15 import P3DGrid
from tests.test_gpu_p3d import PRECS, chain3, models, o3  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,op", PRECS)
@pytest.mark.parametrize("jmass,n", [(2, 1), (2, 512), (2, 1025), (3, 1), (3, 255), (3, 256),
                                     (3, 257), (3, 513)])
def test_step_chain(o3, prec, op, jmass, n):  # noqa: F811
    print("[case] p3d shapes", prec, jmass, n, flush=True)
    m, g = models(o3, prec, op, n=n, jmass=jmass)
    chain3(m, g, 4, prec == "fp32")


@pytest.mark.parametrize("sort", [0, 2])
def test_two_per_thread(sort):
    n = 5_000_000
    w = configs.Workload3("p3d-two", nr=50, na=96, hash=4, n=n, steps=1, dt=0.05, nstep=(1, 2),
                          zbr_model=(0.0, 1.5), ngz=31, dz_model=0.08, eps_model=0.2, seed=8)
    kw = configs.grid_kwargs3(w)
    out = []
    p = None
    for extra in (0, 1):
        print("[case] p3d two per thread", sort, n + extra, flush=True)
        g = P3DGrid(precision="fp32", **kw)
        g.greenm()
        if p is None:
            p = configs.particles3(w, None, None, g.rgrid)
        q = p
        if extra:
            last = [10.0 * g.rgrid, 0.0, 0.0, 0.0, 0.0, 0.0]
            q = [np.append(a, np.asarray(v, a.dtype)) for a, v in zip(p[:6], last)]
            q.append(np.append(p[6], np.int32(3)).astype(np.int32))
        g.restrt(*q)
        g.masset()
        m0 = g.get_mass()
        g.set_sort_interval(sort)
        g.run(4)
        out.append((m0, g.get_mass(), g.unload(), g.noff))
        g.close()
    (a0, a1, ap, an), (b0, b1, bp, bn) = out
    for a, b in ((a0, b0), (a1, b1)):
        assert a[4] == b[4]
        for u, v in zip(a[:4], b[:4]):
            np.testing.assert_array_equal(u, v)
    for k in ap:
        np.testing.assert_array_equal(ap[k], bp[k][:n])
    assert bn == an + 1
