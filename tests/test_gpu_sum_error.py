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


# Limits: 256x256 tiles with the shares of k that they take there (8, 8, 8, 3, 8, 5, 3), one sum per 16 of k, and 2 % for other inputs
@pytest.mark.parametrize("dtype,m,k,n,limit", [(_lib.W_BF16, 700, 5632, 2048, 1.62e-7), (_lib.W_BF16, 300, 4096, 4096, 1.40e-7), (_lib.W_BF16, 201, 2048, 2048, 1.04e-7),
                                               (_lib.W_BF16, 512, 768, 768, 9.45e-8), (_lib.W_Q8_0, 300, 4096, 4096, 1.59e-7), (_lib.W_BF16, 65, 4096, 12288, 1.72e-7),
                                               (_lib.W_BF16, 2036, 4096, 2560, 2.28e-7)])
def test_prompts_of_few_tiles(orc, dtype, m, k, n, limit):
    wt = Weight(dtype, seed=5, shape=(k, n))
    a = np.random.default_rng(m + k).standard_normal((m, k)).astype(np.float32)
    rows = np.arange(0, m, m // 24)
    ar, wd = a[rows], wt.dequantize()
    ar, wd = (orc.bf16_round(ar), wd) if dtype == _lib.W_BF16 else (ar.astype(np.float16), wd.astype(np.float16))
    want = ar.astype(np.float64) @ wd.astype(np.float64)
    assert _rms(wt.gemm(dev(a))[rows], want) <= limit


# Limits: waves of bf16 rows sixteen a workgroup, of f32 rows in four parts of k, chains from a wave's first pair to its last, and 2 % for other inputs
@pytest.mark.parametrize("dtype,k,n,rows,limit", [(_lib.W_BF16, 11008, 4096, 8, 2.08e-7), (_lib.W_BF16, 4224, 6176, 8, 1.32e-7), (_lib.W_BF16, 4096, 4096, 8, 1.30e-7),
                                                  (_lib.W_BF16, 2816, 4096, 4, 1.17e-7), (_lib.W_BF16, 2560, 12352, 8, 1.12e-7), (_lib.W_F32, 5632, 8192, 4, 1.29e-7),
                                                  (_lib.W_F32, 4096, 8192, 8, 1.62e-7)])
def test_decode_rows_on_dense_weights(dtype, k, n, rows, limit):
    wt = Weight(dtype, seed=3, shape=(k, n))
    x = np.random.default_rng(k).standard_normal((rows, k)).astype(np.float32)
    want = x.astype(np.float64) @ wt.dequantize().astype(np.float64)
    assert _rms(wt.gemv(dev(x)), want) <= limit
