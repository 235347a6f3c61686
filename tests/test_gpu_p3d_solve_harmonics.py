"""The 3-D solve by its harmonics per pass (3, 5, 7 and 9, one and several
passes), with the first harmonic skipped, sectors and the Nyquist harmonic, about
the lines where a wavefront takes one plane instead of two and where each pass
gets wavefronts of its own, and where the vertical transforms take one column a
block.

Tolerances: those of test_gpu_p3d.py for the same comparison (1e-10 and 1e-5
of the component's largest value; the transforms sum at most 200 terms; the
combined masses the same floats, 1e-12 of the largest in FP64, where they are
fixed-point sums here and floating ones in the oracle)."""
import numpy as np
import pytest

from tests.test_gpu_p3d import PRECS, _close, _same, models, o3  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,op", PRECS)
@pytest.mark.parametrize("nr,na,ngz,hash_,nsect,skip", [
    (25, 64, 79, 2, 1, (0,)), (25, 64, 80, 6, 1, ()), (40, 96, 50, 12, 1, (0, 3)),
    (50, 96, 59, 9, 2, ()), (50, 96, 60, 4, 1, (0,)), (60, 90, 51, 6, 1, ()),
    (60, 90, 51, 8, 1, ()), (60, 90, 51, 11, 1, (0,)), (60, 30, 51, 15, 1, ()),
    (60, 90, 51, 16, 2, (0,)), (25, 30, 20, 15, 1, (0,)), (24, 64, 16, 0, 1, (0,))])
def test_field(o3, prec, op, nr, na, ngz, hash_, nsect, skip):  # noqa: F811
    print("[case] p3d harmonics", prec, nr, na, ngz, hash_, nsect, skip, flush=True)
    # a quarter of the outermost cell at least: the set-up refuses a fifth
    al = 2 * np.pi / na
    softl = max(0.3, 0.25 * al * np.exp(al * (nr - 1)))
    m, g = models(o3, prec, op, n=5000, fixed=False, nr=nr, na=na, ngz=ngz, hash_=hash_,
                  nsect=nsect, skip=skip, softl=softl)
    m.masset()
    g.masset()
    tol = 1e-10 if prec == "fp64" else 1e-5
    for lpot in (True, False):
        m.findf(lpot)
        g.findf(lpot)
        f = g.get_field().astype(np.float64)
        for t in range(4):
            sc = np.abs(m.fld[t]).max()
            assert np.abs(f[t] - m.fld[t]).max() <= tol * sc, (lpot, t)
    if prec == "fp32":
        _same(g.get_rho(), m.rho.astype(np.float32), "rho")
    else:
        _close(g.get_rho(), m.rho, 1e-12 * np.abs(m.rho).max(), "rho")
