"""galhip_lgspia without pitches (np 1 and 2), where a wavefront sums a run of
harmonics: runs of one to sixteen, full and short last ones, one and several
groups of wavefronts, on both grids.  Against the oracle at the bar of the other
lgspia tests (1e-12 absolute on coefficients of modulus <= 1; both FP64, z^m by
products grows the rounding by about m <= 512 units of 1.1e-16)."""
import numpy as np
import pytest

from galaxy_amd import configs
from galaxy_amd.lib15 import P3DGrid
from tests._model import SMALL, gpu_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("np_,nm,n", [
    (1, 1, 1), (2, 1, 64), (1, 2, 65), (1, 16, 500), (2, 16, 513), (1, 17, 3001), (2, 33, 3001),
    (1, 128, 4097), (1, 129, 4097), (2, 256, 2000), (1, 511, 700)])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_harmonics(orc, np_, nm, n, prec):
    print("[case] lgspia harmonics", np_, nm, n, prec, flush=True)
    g = gpu_model(precision=prec, n=n)
    out = g.unload()
    ls = SMALL.lscale()
    c, s = orc.lgspia(out["x"], out["y"], out["iz"], SMALL.nzones, True, 1, np_, nm, ls)
    got = g.lgspia(np_, nm, ls)
    g.close()
    assert np.abs(got[0] - c).max() <= 1e-12
    assert np.abs(got[1] - s).max() <= 1e-12


def test_p3d(orc):
    w = configs.Workload3("p3d-lgspia", nr=24, na=64, hash=4, n=3000, steps=1, dt=0.05, ngz=16,
                          dz_model=0.1, eps_model=0.2, seed=5)
    g = P3DGrid(precision="fp32", **configs.grid_kwargs3(w))
    g.restrt(*configs.particles3(w, None, None, g.rgrid))
    out = g.unload()
    off = bool(configs.grid_kwargs3(w).get("offanal"))
    c, s = orc.lgspia(out["x"], out["y"], out["iz"], 1, off, 1, 2, 40, w.lscale())
    got = g.lgspia(2, 40, w.lscale())
    assert np.abs(got[0] - c).max() <= 1e-12
    assert np.abs(got[1] - s).max() <= 1e-12
