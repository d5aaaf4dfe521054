"""The decode matmul of several rows on dense weights (matrix cores; with bf16 weights the activations as three bf16
each) against a float64 product of the same weights and activations."""
import numpy as np
import pytest

from coeus_amd import _lib
from gpu_util import Weight, dev, oracle_roundtrip

pytestmark = pytest.mark.gpu


def bound(x, w, k):
    """Worst case of f32 sums in any order: three terms per k, each sum rounded once (2^-24), of the magnitudes."""
    return 3 * k * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(w)) + 1e-30


# one pair of chunks for one wave; waves with unequal shares; shares of 1, 2, 3, 4 and more pairs; weight rows that
# do not fill a tile; more tiles than workgroups (16 * 4096 rows)
@pytest.mark.parametrize("k,n", [(64, 1), (64, 16), (192, 33), (320, 50), (768, 130), (1024, 17), (2048, 70), (2112, 40), (3072, 31),
                                 (4096, 48), (5632, 20), (11008, 18), (128, 65552), (1024, 5003)])
@pytest.mark.parametrize("batch", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("dtype", [_lib.W_BF16, _lib.W_F32])
def test_rows_match_float64(orc, dtype, k, n, batch):
    rng = np.random.default_rng(k + 31 * n + batch)
    w = (rng.standard_normal((k, n)) * 0.02).astype(np.float32)
    # magnitudes over forty binary orders: every piece of an activation counts
    x = (rng.standard_normal((batch, k)) * np.exp2(rng.integers(-20, 20, (batch, k)))).astype(np.float32)
    wt = Weight(dtype, w)
    wd = oracle_roundtrip(orc, dtype, w).astype(np.float64)
    want = x.astype(np.float64) @ wd
    assert (np.abs(wt.gemv(dev(x)) - want) <= bound(x, wd, k)).all()
    if dtype == _lib.W_F32:  # a short prompt takes the same kernel
        assert (np.abs(wt.gemm(dev(x)) - want) <= bound(x, wd, k)).all()


@pytest.mark.parametrize("batch", [2, 5, 16])
def test_gated_pairs_and_bias(orc, batch):
    rng = np.random.default_rng(batch)
    k, n_eff = 1088, 601
    w = (rng.standard_normal((k, 2 * n_eff)) * 0.05).astype(np.float32)
    x = rng.standard_normal((batch, k)).astype(np.float32)
    bias = (rng.standard_normal(2 * n_eff) * 0.1).astype(np.float32)
    wd = oracle_roundtrip(orc, _lib.W_BF16, w).astype(np.float64)
    pre = x.astype(np.float64) @ wd + bias
    g, u = pre[:, 0::2], pre[:, 1::2]
    y = Weight(_lib.W_BF16, w).gemv(dev(x), bias=dev(bias), epilogue=_lib.EPI_SILU_GATE)
    e = bound(x, wd, k) + 2.0 ** -22 * np.abs(pre)
    # |d silu| <= 1.1; plus a few roundings of the gate's own arithmetic
    want = g / (1 + np.exp(-g)) * u
    assert (np.abs(y - want) <= 1.1 * (e[:, 0::2] * np.abs(u) + e[:, 1::2] * np.abs(g)) + 2.0 ** -20 * np.abs(want) + 1e-6).all()


@pytest.mark.parametrize("batch", [2, 16])
@pytest.mark.parametrize("dtype", [_lib.W_BF16, _lib.W_F32])
def test_infinities_and_nan_stay_in_their_row(orc, dtype, batch):
    rng = np.random.default_rng(batch)
    k, n = 256, 40
    w = (rng.standard_normal((k, n)) * 0.02).astype(np.float32)
    x = rng.standard_normal((batch, k)).astype(np.float32)
    x[0, 7] = np.inf
    x[1, 70] = np.nan
    wd = oracle_roundtrip(orc, dtype, w).astype(np.float64)
    y = Weight(dtype, w).gemv(dev(x))
    assert np.array_equal(y[0], np.sign(wd[7]) * np.inf) and np.isnan(y[1]).all()
    assert (np.abs(y[2:] - x[2:].astype(np.float64) @ wd) <= bound(x[2:], wd, k)).all()
