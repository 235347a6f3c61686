"""Ensembles with enough rings that the solve takes several at a time: every
member bit-identical to the same disc alone, whose solve works by blocks of
one ring.  Rings and spokes off the multiples of what a wavefront or block
takes, more than one pass of nine harmonics, the Nyquist harmonic, skipped
harmonics, empty members, three zones."""
import numpy as np
import pytest

from galaxy_amd import configs
from galaxy_amd.lib15 import P2DEnsemble, P2DGrid
from tests.test_gpu_ensemble import _same

pytestmark = pytest.mark.gpu


def _set_up(w, nmem, prec, mode, skip):
    kw = configs.grid_kwargs(w, 1)
    pm = kw.pop("pmass")
    if skip:
        kw["skip"] = skip
    counts = [0 if i % 7 == 3 else 150 + 97 * i for i in range(nmem)]
    pmass = [pm / max(n, 1) for n in counts]
    e = P2DEnsemble(nmem, pmass=pmass, precision=prec, **kw)
    parts = []
    for i, n in enumerate(counts):
        p = configs.particles(w, max(n, 1), 100 + i, e.rgrid)
        parts.append(tuple(np.ascontiguousarray(a[:n], np.int32 if k == 4 else e.dtype)
                           for k, a in enumerate(p)))
    ff = configs.fixforce(w, e.rgrid)

    def start(g, p):
        g.greenm()
        g.set_fixforce(*ff)
        if mode:
            g.set_contraction("mfma", 0)
        g.restrt(*p)
        g.masset()
        g.set_sort_interval(3)
        return g

    start(e, (parts,))
    lone = {i: start(P2DGrid(pmass=pmass[i], precision=prec, **kw), parts[i])
            for i in (0, 3, nmem // 2, nmem - 1)}
    return e, lone


@pytest.mark.parametrize("prec,mode", [("fp32", 0), ("fp32", 1), ("fp64", 0)])
@pytest.mark.parametrize("nr,na,hash_,nmem,skip", [
    (66, 130, 8, 24, ()), (67, 128, 17, 30, (2, 5)), (50, 90, 45, 38, ())])
def test_members_equal_lone_discs(prec, mode, nr, na, hash_, nmem, skip):
    print("[case] rows", prec, mode, nr, na, hash_, nmem, flush=True)
    w = configs.Workload("rows", nr=nr, na=na, hash=hash_, n=1, steps=1, dt=0.05, nstep=(1, 2, 4),
                         zbr_model=(0.0, 1.5, 3.5), seed=11)
    e, lone = _set_up(w, nmem, prec, mode, skip)
    for lpot in (True, False):
        e.findf(lpot)
        for i, g in lone.items():
            g.findf(lpot)
            _same(e.get_field(i), g.get_field(), "field %d" % i)
            assert e.ranges(i) == g.ranges()
    e.run(5)
    out = e.unload()
    for i, g in lone.items():
        g.run(5)
        ref = g.unload()
        for k in ref:
            _same(out[i][k], ref[k], "%s %d" % (k, i))
        for a, b in zip(e.get_mass(i)[:4], g.get_mass()[:4]):
            _same(a, b, "mass %d" % i)
