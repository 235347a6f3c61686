"""The push and the mass assignment where their launch shape changes: one and
four particles per thread (FP32 above 1.5e6 particles), counts about a
block, blocks whose window has to be clipped many times over.

The step chain against the oracle is bit-exact (integer mass sums, FP32
arithmetic reproduced), as in test_gpu_parity.py.  The mass sums a run's
pushes leave (positions through the push's short logarithm and angle) equal
those masset forms afresh from the same positions by the general routines,
bit for bit, with the ring ranges."""
import numpy as np
import pytest

from galaxy_amd import configs
from tests._model import SMALL, gpu_model, oracle_model
from tests.test_gpu_parity import _chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1_500_000, 1_500_001])
def test_step_chain_large(orc, n):
    print("[case] step chain", n, flush=True)
    m, parts = oracle_model(orc, prec="f", n=n)
    _chain(m, gpu_model(precision="fp32", n=n, parts=parts), 3, True)


def _check(g, steps):
    for _ in range(3):
        g.run(steps)
        mfx, _, jr, kr, _ = g.get_mass()
        g.masset()
        ref = g.get_mass()
        assert np.array_equal(mfx, ref[0])
        assert np.array_equal(jr, ref[2]) and np.array_equal(kr, ref[3])


@pytest.mark.parametrize("n,nr,na", [(1, 64, 128), (255, 64, 128), (257, 64, 128),
                                     (1025, 300, 512), (40_000, 300, 512),
                                     (1_500_001, 64, 128), (1_600_123, 420, 600)])
@pytest.mark.parametrize("prec,comp", [("fp32", False), ("fp64", False), ("fp32", True)])
def test_run_masses_equal_masset(n, nr, na, prec, comp):
    """One zone, re-sorted never: the blocks' particles spread over many cells."""
    print("[case] masses", n, nr, na, prec, comp, flush=True)
    w = configs.Workload("p2d-shapes", nr=nr, na=na, hash=4, n=n, steps=1, dt=0.05, seed=7)
    g = configs.make_grid(w, precision=prec, compensated=comp)
    _check(g, 6)
    g.close()


@pytest.mark.parametrize("n,nr,na,ngz", [(1, 24, 64, 16), (511, 24, 64, 16), (513, 64, 128, 45),
                                          (30_000, 90, 128, 61), (600_123, 40, 90, 31)])
@pytest.mark.parametrize("prec,jmass", [("fp32", 2), ("fp64", 2), ("fp32", 3)])
def test_run_masses_equal_masset_p3d(n, nr, na, ngz, prec, jmass):
    from galaxy_amd.lib15 import P3DGrid
    print("[case] masses p3d", n, nr, na, ngz, prec, jmass, flush=True)
    w = configs.Workload3("p3d-shapes", nr=nr, na=na, hash=2, n=n, steps=1, dt=0.05, ngz=ngz,
                          dz_model=0.08, eps_model=0.2, seed=8)
    g = P3DGrid(precision=prec, jmass=jmass, **configs.grid_kwargs3(w))
    g.greenm()
    g.restrt(*configs.particles3(w, None, None, g.rgrid))
    g.masset()
    _check(g, 4)
    g.close()


def test_ensemble_equals_lone_discs_across_shapes():
    """Three members of 6e5 particles (four per thread together) against the
    same discs alone (one per thread)."""
    from galaxy_amd.lib15 import P2DEnsemble
    n = [600_000, 600_001, 400_000]
    w = [configs.Workload("m%d" % i, nr=64, na=128, hash=8, n=k, steps=1, dt=0.05, seed=20 + i)
         for i, k in enumerate(n)]
    kw = configs.grid_kwargs(w[0])
    kw.pop("pmass")
    E = P2DEnsemble(3, pmass=[configs.grid_kwargs(v)["pmass"] for v in w], **kw)
    E.greenm()
    E.set_fixforce(*configs.fixforce(w[0], E.rgrid))
    E.restrt([configs.particles(v, None, None, E.rgrid) for v in w])
    E.masset()
    E.run(8)
    members = E.unload()
    for i, v in enumerate(w):
        print("[case] member", i, flush=True)
        g = configs.make_grid(v)
        g.run(8)
        o = g.unload()
        for k in ("x", "y", "vx", "vy", "iz"):
            assert np.array_equal(members[i][k], o[k]), k
        for a, b in zip(E.get_mass(i), g.get_mass()):
            assert np.array_equal(a, b)
        g.close()
    E.close()
