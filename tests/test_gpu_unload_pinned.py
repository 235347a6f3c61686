"""Unloads into pinned arrays, alone and among pageable ones, on both sides of
the size from which pageable memory is written through chunks of its own."""
import ctypes as C

import numpy as np
import pytest

from galaxy_amd.lib15 import P2DGrid, P3DGrid

pytestmark = pytest.mark.gpu


class _Pinned:
    """An array in memory of hipHostMalloc, by the runtime that libgalhip loads."""

    def __init__(self, lib, n, dtype):
        self.lib, self.p = lib, C.c_void_p()
        size = n * np.dtype(dtype).itemsize
        assert lib.hipHostMalloc(C.byref(self.p), C.c_size_t(size), C.c_uint(0)) == 0
        buf = (C.c_char * size).from_address(self.p.value)
        self.a = np.frombuffer(buf, dtype)

    def close(self):
        self.a = None
        assert self.lib.hipHostFree(self.p) == 0


@pytest.mark.parametrize("mask", [0b1111111, 0b0000001, 0b1010100, 0b0111111])
@pytest.mark.parametrize("dim,n,prec", [(2, 1000, "fp32"), (2, 1_500_007, "fp32"),
                                        (2, 700_001, "fp64"), (3, 800_001, "fp32")])
def test_pinned(dim, n, prec, mask):
    print("[case] pinned", dim, n, prec, bin(mask), flush=True)
    kw = dict(hash_=1, softl=3.0, pmass=1e-7, precision=prec)
    g = P2DGrid(60, 128, **kw) if dim == 2 else P3DGrid(20, 32, 11, dzg=0.5, **kw)
    rng = np.random.default_rng(n)
    ref = [(rng.random(n) * 6 - 3).astype(g.dtype) for _ in range(2 * dim)]
    ref.append(rng.integers(1, 3, n).astype(np.int32))
    g.restrt(*ref)
    pin = [_Pinned(g._lib, n, r.dtype) if mask >> k & 1 else None for k, r in enumerate(ref)]
    dst = [p.a if p else np.empty(n, r.dtype) for p, r in zip(pin, ref)]
    f = g._lib.galhip_unload if dim == 2 else g._lib.galhip_unload3
    for _ in range(2):
        for d in dst:
            d[:] = 0
        assert f(g._h, *[d.ctypes.data_as(C.c_void_p) for d in dst]) == 0
        for d, r in zip(dst, ref):
            np.testing.assert_array_equal(d, r)
    del d, dst
    for p in pin:
        if p:
            p.close()
