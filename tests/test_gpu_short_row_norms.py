"""The decode matmul of 2 to 16 bf16 rows behind a folded norm where a row has no more pairs of chunks than sixteen waves:
one pair for each wave, so that a wave may have to normalise several rows.  float64 of the same values, from one pair to
sixteen, with fewer and more rows than waves."""
import ctypes as C

import numpy as np
import pytest

from coeus_amd import _lib
from coeus_amd.device import DeviceArray
from coeus_amd.plugin import _check
from gpu_util import Weight, dev, oracle_roundtrip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [_lib.NORM_LAYERNORM, _lib.NORM_RMSNORM])
@pytest.mark.parametrize("batch,k,n", [
    (2, 64, 18), (16, 64, 34), (7, 448, 40), (8, 448, 4200), (16, 576, 18),
    (3, 768, 2304), (12, 768, 50), (13, 768, 34), (16, 832, 2), (4, 960, 66), (8, 1024, 18)])
def test_matches_float64(orc, batch, k, n, kind):
    rng = np.random.default_rng(k + n + batch)
    w = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    h = (rng.standard_normal((batch, k)) * 3 + 1).astype(np.float32)
    scale, nbias = rng.uniform(0.5, 1.5, k).astype(np.float32), rng.standard_normal(k).astype(np.float32)
    wt, wd = Weight(_lib.W_BF16, w), oracle_roundtrip(orc, _lib.W_BF16, w).astype(np.float64)
    x = h.astype(np.float64)
    if kind == _lib.NORM_LAYERNORM:
        x = x - x.mean(1, keepdims=True)
    x = x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5) * scale + (nbias if kind == _lib.NORM_LAYERNORM else 0)
    pre = x @ wd
    # f32 sums over k of the magnitudes, and the norm's own few roundings of the row
    e = (3 * k + 40) * 2.0 ** -24 * (np.abs(x) @ np.abs(wd))
    hd, sd, nd = dev(h), dev(scale), dev(nbias)
    for gated in (False, True):
        y, fused = DeviceArray((batch, n // 2 if gated else n)), C.c_int()
        _check(_lib.load().coeus_op_norm_gemv(wt.h, hd.ptr, batch, kind, sd.ptr, nd.ptr, C.c_float(1e-5), None, None,
                                              _lib.EPI_SILU_GATE if gated else 0, y.ptr, C.byref(fused), None))
        want, lim = pre, e
        if gated:
            g, u = pre[:, 0::2], pre[:, 1::2]
            want = g / (1 + np.exp(-g)) * u
            lim = 1.1 * (e[:, 0::2] * np.abs(u) + e[:, 1::2] * np.abs(g)) + 2.0 ** -20 * np.abs(want) + 1e-6
        assert fused.value == 1 and (np.abs(y.to_host() - want) <= lim).all(), gated
