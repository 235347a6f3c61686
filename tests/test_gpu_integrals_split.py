"""galhip_integrals where its particles per thread change (1, 2, 4 and 8 on the
2-D grid, 1 and 2 on the 3-D one), with and without a device allocation, and
of an ensemble with members on both sides of a change, against numpy's FP64
sums.  Bar: 1e-13 of the sum of the terms' magnitudes (at most 8 + 6 + 8 + 8 + 6
+ 8 additions in a row, each with an error of 1.1e-16 of a partial sum; numpy's
pairwise sums less)."""
import numpy as np
import pytest

from galaxy_amd.lib15 import P2DEnsemble, P2DGrid, P3DGrid

pytestmark = pytest.mark.gpu
PM = 1e-7


def _set(n, dim, dtype):
    rng = np.random.default_rng(n)
    a = [(rng.random(n) * 6 - 3).astype(dtype) for _ in range(2 * dim)]
    return a + [np.ones(n, np.int32)]


def _check(got, p, dim):
    o = [v.astype(np.float64) for v in p[:2 * dim]]
    pos, vel = o[:dim], o[dim:]

    def close(value, terms):
        assert abs(value - PM * terms.sum()) <= 1e-13 * PM * np.abs(terms).sum()

    close(got["mass"], np.ones(len(o[0])))
    close(got["ke"], 0.5 * sum(v * v for v in vel))
    close(got["lz"], pos[0] * vel[1] - pos[1] * vel[0])
    for k in range(dim):
        close(got["momentum"][k], vel[k])
        close(got["cm"][k] * got["mass"], pos[k])


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("dim,n", [(2, 1048575), (2, 1048576), (2, 2097151), (2, 2097153),
                                   (2, 4194303), (2, 4194305), (3, 2097151), (3, 2097153)])
def test_split(dim, n, prec):
    print("[case] integrals split", dim, n, prec, flush=True)
    kw = dict(hash_=1, softl=3.0, pmass=PM, precision=prec)
    g = P2DGrid(60, 128, **kw) if dim == 2 else P3DGrid(20, 32, 11, dzg=0.5, **kw)
    p = _set(n, dim, g.dtype)
    g.restrt(*p)
    got = g.integrals(centred=False)
    _check(got, p, dim)
    free = g.integrals(centred=False, noalloc=True)
    for k, v in got.items():
        np.testing.assert_array_equal(np.asarray(free[k]), np.asarray(v))


def test_members():
    n = [3, 1048577, 0, 70_000]
    e = P2DEnsemble(4, 60, 128, hash_=1, softl=3.0, pmass=[PM] * 4)
    mem = [_set(k, 2, e.dtype) for k in n]
    e.restrt(mem)
    got = e.integrals(centred=False)
    for i in (0, 1, 3):
        _check(got[i], mem[i], 2)
