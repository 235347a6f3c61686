"""galhip_integrals at particle counts about one block's share of the sums
(8 particles for each of 256 threads; 512 on the 3-D grid), one zone,
velocities not centred, against numpy's FP64 sums of the unloaded particles.
Bar: 1e-13 of the sum of the terms' magnitudes (n <= 4097 terms, each added
with an error of 1.1e-16 of a partial sum, in runs of at most 8 + 6 + 8)."""
import numpy as np
import pytest

from galaxy_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 2047, 2048, 2049, 4095, 4097])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_integrals_units(n, dim, prec):
    print("[case] integrals", n, dim, prec, flush=True)
    kw = dict(nr=24, na=64, hash=4, n=n, steps=1, dt=0.05, eps_model=0.2, seed=5)
    if dim == 3:
        w = configs.Workload3("p3d-integrals", ngz=16, dz_model=0.1, **kw)
        g = configs.make_grid3(w, precision=prec, green=False)
    else:
        w = configs.Workload("p2d-integrals", **kw)
        g = configs.make_grid(w, precision=prec, green=False)
    got = g.integrals(centred=False)
    o = {k: v.astype(np.float64) for k, v in g.unload().items()}
    g.close()
    pm = configs.grid_kwargs(w)["pmass"]
    names = "xyz"[:dim]
    v2 = sum(o["v" + q] ** 2 for q in names)
    lz = o["x"] * o["vy"] - o["y"] * o["vx"]

    def check(value, terms):
        assert abs(value - pm * terms.sum()) <= 1e-13 * pm * max(np.abs(terms).sum(), 1e-300)

    check(got["mass"], np.ones(n))
    check(got["ke"], 0.5 * v2)
    check(got["lz"], lz)
    for k, q in enumerate(names):
        check(got["momentum"][k], o["v" + q])
        check(got["cm"][k] * got["mass"], o[q])
