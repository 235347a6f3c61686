"""FP64 discs above 1.5e6 particles take two particles per thread when they are
never sorted again and one when they are: the arithmetic is the same, and so are
all results' bits.  The counts' last blocks hold one particle, one more than half
a block and a whole block."""
import numpy as np
import pytest

from galaxy_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1_500_161, 1_500_417, 1_500_672])
def test_same_bits(n):
    print("[case] fp64 unsorted", n, flush=True)
    w = configs.Workload("p2d-unsorted", nr=64, na=128, hash=4, n=n, steps=1, dt=0.05,
                         nstep=(1, 2, 4), zbr_model=(0.0, 1.5, 3.5), seed=7)
    out = []
    for sort in (0, 3):
        g = configs.make_grid(w, precision="fp64")
        g.set_sort_interval(sort)
        g.masset()
        m0 = g.get_mass()
        g.run(8)
        out.append((m0, g.get_mass(), g.unload(), g.noff))
        g.close()
    (a0, a1, ap, an), (b0, b1, bp, bn) = out
    for a, b in ((a0, b0), (a1, b1)):
        for u, v in zip(a, b):
            np.testing.assert_array_equal(u, v)
    for k in ap:
        np.testing.assert_array_equal(ap[k], bp[k])
    assert an == bn
