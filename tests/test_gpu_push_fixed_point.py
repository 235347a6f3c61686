"""Fixed-point weights of the deposits on both sides of the line between the
fused rounding and the general one (8191 particles: 49 bits), and at the
smallest and an ordinary count: the step chain against the oracle is bit-exact
in FP32 (integer mass sums included), as in test_gpu_parity.py."""
import pytest

from tests._model import gpu_model, oracle_model
from tests.test_gpu_parity import _chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 8190, 8191, 8192, 40_000])
def test_step_chain(orc, n):
    print("[case] fixed point", n, flush=True)
    m, parts = oracle_model(orc, prec="f", n=n)
    _chain(m, gpu_model(precision="fp32", n=n, parts=parts), 4, True)
