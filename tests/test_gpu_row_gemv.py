"""The decode matmul of one plain row (two weight rows a wave): float64 of the same values, at the edges of the lanes' eight elements, of
the steps of 512, of the two and four steps in flight, of a wave's two rows and a workgroup's eight."""
import numpy as np
import pytest

from coeus_amd import _lib
from gpu_util import Weight, dev, oracle_roundtrip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [_lib.W_F32, _lib.W_BF16])
@pytest.mark.parametrize("k,n", [(8, 1), (64, 3), (504, 18), (512, 4), (520, 37), (768, 8195), (1024, 2306), (1032, 7), (1536, 2048), (2048, 2050),
                                 (2056, 9), (4096, 66), (4104, 2049), (5632, 130), (11008, 33),
                                 # (where other kernels take the row: the matrix cores, a wave per row)
                                 (64, 16390), (512, 16384), (10240, 2054), (1536, 2306), (768, 20002), (1032, 8194),
                                 # two weight rows a wave again
                                 (520, 32002), (1544, 16386), (2056, 16386), (3080, 2042)])
@pytest.mark.parametrize("gated", [False, True])
def test_matches_float64(orc, dtype, k, n, gated):
    if gated:
        n = 2 * n
    rng = np.random.default_rng(k + n)
    w = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    x = rng.standard_normal((1, k)).astype(np.float32)
    bias, res = rng.standard_normal(n).astype(np.float32), rng.standard_normal((1, n // 2 if gated else n)).astype(np.float32)
    wt, wd = Weight(dtype, w), oracle_roundtrip(orc, dtype, w).astype(np.float64)
    pre = x.astype(np.float64) @ wd + bias
    # f32 sums over k in any order
    e = (k + 4) * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(wd) + np.abs(bias))
    if gated:
        g, u = pre[:, 0::2], pre[:, 1::2]
        got, want = wt.gemv(dev(x), bias=dev(bias), residual=dev(res), epilogue=_lib.EPI_SILU_GATE), g / (1 + np.exp(-g)) * u + res
        e = 1.1 * (e[:, 0::2] * np.abs(u) + e[:, 1::2] * (np.abs(g) + e[:, 0::2])) + 2.0 ** -20 * (np.abs(g * u) + np.abs(want)) + 1e-6
    else:
        got, want = wt.gemv(dev(x), bias=dev(bias), residual=dev(res)), pre + res
        e = e + 2.0 ** -23 * np.abs(want)
    assert (np.abs(got - want) <= e).all()


# A weight row a wave: one, two, three, four and six steps in flight, with shares that end inside a step and inside a trip, both sides of 1024 rows
@pytest.mark.parametrize("dtype", [_lib.W_F32, _lib.W_BF16])
@pytest.mark.parametrize("k,n", [(512, 768), (776, 3), (1288, 1030), (1544, 1024), (2560, 1025), (2568, 5), (3072, 1024), (3080, 1001), (4608, 6), (5640, 1023), (16384, 4097)])
def test_a_weight_row_a_wave(orc, dtype, k, n):
    test_matches_float64(orc, dtype, k, n, False)
