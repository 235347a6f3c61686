"""Ensembles about the line where the analysis takes several rings a wavefront,
by the harmonics of its passes (3, 5, 7, 9 and several passes): every member
bit-identical to the same disc alone, whose analysis works by rings."""
import pytest

from galaxy_amd import configs
from tests.test_gpu_ensemble import _same
from tests.test_gpu_ensemble_rows import _set_up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("nr,na,hash_,nmem", [
    (60, 128, 0, 15), (60, 128, 0, 16), (60, 130, 2, 16), (61, 128, 4, 18), (66, 128, 6, 19),
    (50, 90, 9, 26), (67, 128, 12, 26), (50, 90, 45, 82)])
def test_members_equal_lone_discs(prec, nr, na, hash_, nmem):
    print("[case] harmonics", prec, nr, na, hash_, nmem, flush=True)
    w = configs.Workload("harm", nr=nr, na=na, hash=hash_, n=1, steps=1, dt=0.05, nstep=(1, 2, 4),
                         zbr_model=(0.0, 1.5, 3.5), seed=11)
    e, lone = _set_up(w, nmem, prec, 0, ())
    for lpot in (True, False):
        e.findf(lpot)
        for i, g in lone.items():
            g.findf(lpot)
            _same(e.get_field(i), g.get_field(), "field %d" % i)
            assert e.ranges(i) == g.ranges()
