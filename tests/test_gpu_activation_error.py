"""SiLU gates and GELU of the matmuls whose f32 results callers see: float64 of the same pre-activation, in roundings of the result.  One
product a dot product, so that the pre-activation is known to the bit."""
import numpy as np
import pytest

from coeus_amd import _lib
from gpu_util import Weight, dev

pytestmark = pytest.mark.gpu
UNIT = 2.0 ** -24


def _case(dtype, k, rows, gated, f16_weights):
    rng = np.random.default_rng(rows + k)
    n = 8192
    pre = (rng.uniform(-4, 4, n) * rng.choice([1, 1, .1, 3.9], n)).astype(np.float32)
    w = np.zeros((k, 2 * n), np.float32)
    if gated:
        w[0, 0::2], w[32, 1::2] = pre, 1
    else:
        w[0] = np.concatenate([pre, -pre])
    x = np.zeros((rows, k), np.float32)
    x[:, 0], x[:, 32] = np.round(rng.uniform(.5, 1.5, rows) * 128) / 128, 1  # (8 bits: exact in f16 and bf16)
    wt = Weight(dtype, w)
    wd = wt.dequantize()
    if f16_weights:
        wd = wd.astype(np.float16).astype(np.float32)
    z = (x[:, :1].astype(np.float64) * wd[:1]).astype(np.float32).astype(np.float64)
    return wt, x, z, wd[32, 1::2].astype(np.float64)


def _check(got, want, x, limits):
    for lo, hi, units in limits:
        at = (x > lo) & (x <= hi)
        worst = (np.abs(got - want)[at] / np.abs(want[at])).max() / UNIT
        assert worst <= units, (lo, hi, worst)


# e^-x: 1 ulp of exp2 (2 units) for its part e / (1 + e) of the sum, its argument to 1 unit; the division 1 unit, the product with the other
# half 1 unit
SILU = [(-16, 0, 5.0), (0, 16, 4.0)]
# the same without the product; behind the rounding of the argument s (3 units of it, |s| e / (1 + e) of the result): 9 + 4 units in
# all between -1 and -0.1, 40 |x| beyond, none of it near 0
GELU = [(-4, -2, 100.0), (-1, -.1, 8.0), (-.1, .1, 2.5), (.1, 16, 2.5)]


def _silu_and_gelu(dtype, k, rows, call, f16_weights=False):
    wt, x, z, up = _case(dtype, k, rows, True, f16_weights)
    g = z[:, 0::2]
    _check(getattr(wt, call)(dev(x), epilogue=_lib.EPI_SILU_GATE), g / (1 + np.exp(-g)) * up, g, SILU)
    wt, x, z, _ = _case(dtype, k, rows, False, f16_weights)
    with np.errstate(over="ignore"):  # 0.5 z (1 + tanh(u)) = z / (1 + e^-2u)
        want = z / (1 + np.exp(-2 * 0.7978845608028654 * z * (1 + 0.044715 * z * z)))
    _check(getattr(wt, call)(dev(x), epilogue=_lib.EPI_GELU), want, z, GELU)


@pytest.mark.parametrize("dtype", [_lib.W_Q8_0, _lib.W_Q4_0])
@pytest.mark.parametrize("rows", [5, 8, 16])
def test_decode_rows_on_quantised_weights(dtype, rows):
    _silu_and_gelu(dtype, 64, rows, "gemv")


# tiles of 128 rows by 64 columns; few slices of k, and many
@pytest.mark.parametrize("dtype", [_lib.W_BF16, _lib.W_Q8_0])
@pytest.mark.parametrize("k,rows", [(64, 65), (64, 300), (4096, 100)])
def test_prompts_of_few_tiles(dtype, k, rows):
    _silu_and_gelu(dtype, k, rows, "gemm", f16_weights=dtype == _lib.W_Q8_0)
