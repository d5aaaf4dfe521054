"""Root mean square errors of sums over k against float64 of the same operands, relative to the results': no larger than those of other orders
that the same sums have been in."""
import numpy as np
import pytest

from coeus_amd import _lib
from gpu_util import Weight, dev

pytestmark = pytest.mark.gpu


def _rms(got, want):
    return np.sqrt(((got - want) ** 2).mean() / (want ** 2).mean())


# Limits: blocks of 32 in order over eight waves (2048) or sixteen (8192), the waves' sums in order, and 1.5 % for other inputs
@pytest.mark.parametrize("dtype,k,n,limit", [(_lib.W_Q4_0, 2048, 8192, 7.95e-8), (_lib.W_Q8_0, 2048, 8192, 8.35e-8), (_lib.W_Q4_0, 2048, 6144, 7.95e-8),
                                             (_lib.W_Q4_0, 8192, 512, 1.075e-7)])
@pytest.mark.parametrize("rows", [8, 16])
def test_decode_rows_on_quantised_weights(dtype, k, n, limit, rows):
    wt = Weight(dtype, seed=10, shape=(k, n))
    x = np.random.default_rng(k).standard_normal((rows, k)).astype(np.float32)
    want = x.astype(np.float16).astype(np.float64) @ wt.dequantize().astype(np.float64)
    assert _rms(wt.gemv(dev(x)), want) <= limit
