"""The 3-D solve where its launch shapes change: 1, 3 and 9 component columns a
block (contexts of fewer than 3, fewer than 9 and more columns, few and many
rings), more than one pass of nine harmonics, planes and spokes about and off
the multiples of a wavefront, the Nyquist harmonic's single column.

Tolerances: those of test_gpu_p3d.py for the same comparison (1e-10 and 1e-5
of the component's largest value; the transforms sum at most 256 terms)."""
import numpy as np
import pytest

from tests.test_gpu_p3d import PRECS, models, o3  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,op", PRECS)
@pytest.mark.parametrize("nr,na,ngz,hash_", [
    (24, 64, 16, 0), (24, 64, 17, 1), (24, 64, 63, 3), (24, 64, 64, 4), (24, 100, 65, 9),
    (30, 90, 9, 45), (200, 512, 7, 8)])
def test_field(o3, prec, op, nr, na, ngz, hash_):  # noqa: F811
    print("[case] p3d solve", prec, nr, na, ngz, hash_, flush=True)
    m, g = models(o3, prec, op, n=5000, nr=nr, na=na, ngz=ngz, hash_=hash_)
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
        if lpot:
            pot = f[3]
    np.testing.assert_array_equal(f[3], pot)   # kept by a solve without it
