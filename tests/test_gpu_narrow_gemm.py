"""The prompt matmul of few tiles (128 or 256 rows by 64 to 128 columns, shares of k): float64 of the same 16-bit operands, at the
edges of the tiles, of the rings of slices and of the shares."""
import numpy as np
import pytest

from coeus_amd import _lib
from gpu_util import Weight, dev, oracle_roundtrip

pytestmark = pytest.mark.gpu


def _bf16(x):
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)


# 64 - 6 x 64 of k: fewer slices than the rings hold, as many, one more; 65 - 520 rows and 128 - 3100 columns: inside, on and
# behind the edges of 128 and 256 rows and of 64, 96 and 128 columns; long k on few tiles: shares
@pytest.mark.parametrize("m,k,n", [(65, 64, 128), (128, 128, 130), (129, 192, 190), (127, 256, 194), (200, 320, 1000), (256, 384, 256),
                                   (257, 448, 514), (300, 768, 2304), (512, 3072, 768), (201, 4096, 4098), (257, 1024, 7000),
                                   (520, 2048, 3100), (201, 1024, 22016), (1019, 704, 2048), (700, 2048, 8192)])
@pytest.mark.parametrize("dtype", [_lib.W_BF16, _lib.W_Q8_0])
def test_matches_float64(orc, dtype, m, k, n):
    rng = np.random.default_rng(m + k + n)
    w = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    a = rng.standard_normal((m, k)).astype(np.float32)
    bias, res = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    wt, wd = Weight(dtype, w), oracle_roundtrip(orc, dtype, w)
    if dtype == _lib.W_BF16:
        ar = _bf16(a)
    else:  # the matrix cores take f16 of the activations and of the dequantised weights
        ar, wd = a.astype(np.float16).astype(np.float32), wd.astype(np.float16).astype(np.float32)
    rows = np.unique(np.concatenate([np.arange(0, m, 37), [m - 1, min(m - 1, 127), min(m - 1, 128), min(m - 1, 255), min(m - 1, 256)]]))
    x, wd = ar[rows].astype(np.float64), wd.astype(np.float64)
    pre, mag = x @ wd, np.abs(x) @ np.abs(wd)
    # f32 sums over k of exact products, in any order: k roundings of at most 2^-24 of the magnitudes
    lim = (k + 4) * 2.0 ** -24 * mag + 1e-30
    assert (np.abs(wt.gemm(dev(a))[rows] - pre) <= lim).all()
    # the activation: 2^-20 of its value for exp2, reciprocal and their arguments (slope at most 1.13)
    pb = pre + bias
    want = 0.5 * pb * (1 + np.tanh(0.7978845608028654 * (pb + 0.044715 * pb ** 3)))
    got = wt.gemm(dev(a), bias=dev(bias), residual=dev(res), epilogue=_lib.EPI_GELU)[rows]
    assert (np.abs(got - want - res[rows]) <= 1.2 * lim + 2.0 ** -18 * (np.abs(pb) + np.abs(res[rows]))).all()
    g, u = pre[:, 0::2], pre[:, 1::2]
    want = g / (1 + np.exp(-g)) * u
    got = wt.gemm(dev(a), epilogue=_lib.EPI_SILU_GATE)[rows]
    assert (np.abs(got - want) <= 1.1 * (lim[:, 0::2] * np.abs(u) + lim[:, 1::2] * (np.abs(g) + lim[:, 0::2])) + 2.0 ** -18 * np.abs(g * u)).all()
