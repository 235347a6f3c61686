"""galhip_lgspia where its work split changes: pitch offsets per wavefront
(4, 8 and 12 sums, one and several runs per harmonic), wavefront groups per
block, particle counts about one tile, and the largest coefficient count.
Against the oracle at the bar of the other lgspia tests: 1e-12 absolute on
coefficients of modulus <= 1 (both FP64; w^k by repeated products grows the
rounding by about k <= 255 units of 1.1e-16)."""
import numpy as np
import pytest

from tests._model import SMALL, gpu_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("np_,nm,n", [
    (2, 1, 1), (3, 1, 63), (9, 1, 65), (11, 2, 500), (17, 8, 513), (19, 3, 4097),
    (25, 6, 3001), (26, 6, 3001), (27, 6, 3001), (51, 9, 2000), (64, 8, 2000), (511, 1, 1000),
    (1, 512, 1000)])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_lgspia_units(orc, np_, nm, n, prec):
    print("[case] lgspia", np_, nm, n, prec, flush=True)
    g = gpu_model(precision=prec, n=n)
    out = g.unload()
    ls = SMALL.lscale()
    c, s = orc.lgspia(out["x"], out["y"], out["iz"], SMALL.nzones, True, 1, np_, nm, ls)
    got = g.lgspia(np_, nm, ls)
    g.close()
    assert np.abs(got[0] - c).max() <= 1e-12
    assert np.abs(got[1] - s).max() <= 1e-12
