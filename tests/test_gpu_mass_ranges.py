"""galhip_set_mass / galhip_get_mass: the ring ranges of one and of the most
zones, set alone or together, on both grids; an ensemble's members, whose
ranges lie in rows longer than one grid's."""
import numpy as np
import pytest

from galaxy_amd.lib15 import P2DEnsemble, P2DGrid, P3DGrid

pytestmark = pytest.mark.gpu

NZ = [1, 3, 10]


def _zones(nz):
    return dict(nzones=nz, nstep=(1,) * nz, zbr=tuple(0.5 * i for i in range(nz)), pmass=1e-6)


def _grid(dim, nz):
    if dim == 2:
        return P2DGrid(60, 128, hash_=1, softl=2.0, **_zones(nz))
    return P3DGrid(20, 32, 11, dzg=0.5, hash_=1, softl=3.0, **_zones(nz))


@pytest.mark.parametrize("nz", NZ)
@pytest.mark.parametrize("dim", [2, 3])
def test_set_get(dim, nz):
    print("[case] ranges", dim, nz, flush=True)
    g = _grid(dim, nz)
    jr = np.arange(3, 3 + nz, dtype=np.int32)
    kr = np.arange(7, 7 + nz, dtype=np.int32)
    g.set_mass(jrad=jr, krad=kr)
    for a, b in ((jr + 1, None), (None, kr + 2)):
        got = g.get_mass()
        np.testing.assert_array_equal(got[2], jr)
        np.testing.assert_array_equal(got[3], kr)
        g.set_mass(jrad=a, krad=b)
        jr, kr = (jr if a is None else a), (kr if b is None else b)
    got = g.get_mass()
    np.testing.assert_array_equal(got[2], jr)
    np.testing.assert_array_equal(got[3], kr)


@pytest.mark.parametrize("nmem", [1, 3, 4, 70])
def test_members(nmem):
    """Each member's ranges are those of its one particle."""
    print("[case] member ranges", nmem, flush=True)
    e = P2DEnsemble(nmem, 60, 128, hash_=1, softl=2.0, nzones=2, nstep=(1, 2), zbr=(0.0, 5.0),
                    pmass=[1e-6] * nmem)
    g = P2DGrid(60, 128, hash_=1, softl=2.0, nzones=2, nstep=(1, 2), zbr=(0.0, 5.0), pmass=1e-6)
    mem = []
    for i in range(nmem):
        r = 0.3 + 0.1 * i
        mem.append([np.array([v], np.float32) for v in (r, 0.0, 0.0, 0.0)] +
                   [np.array([1 + (r > 5.0)], np.int32)])
    e.restrt(mem)
    e.masset()
    for i, m in enumerate(mem):
        g.restrt(*m)
        g.masset()
        got, ref = e.get_mass(i), g.get_mass()
        np.testing.assert_array_equal(got[2], ref[2])
        np.testing.assert_array_equal(got[3], ref[3])
