"""The decode matmul of one row behind a norm (the row in a wave's registers): float64 of the same values, at the edges
of the lanes' eight elements, of the two 512-wide steps and of the four weight rows of a wave."""
import ctypes as C

import numpy as np
import pytest

from coeus_amd import _lib
from coeus_amd.device import DeviceArray
from coeus_amd.plugin import _check
from gpu_util import Weight, dev, oracle_roundtrip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [_lib.W_F32, _lib.W_BF16])
@pytest.mark.parametrize("kind", [_lib.NORM_LAYERNORM, _lib.NORM_RMSNORM])
@pytest.mark.parametrize("k,n", [(8, 1), (64, 3), (504, 18), (512, 4), (520, 37), (768, 2304), (1016, 5), (1024, 1030)])
@pytest.mark.parametrize("gated,shift", [(False, 0), (True, 0), (False, 1)])
def test_matches_float64(orc, dtype, kind, k, n, gated, shift):
    if gated:
        n = 2 * n
    rng = np.random.default_rng(k + n + kind)
    w = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    h = (rng.standard_normal(k) * 3 + 1).astype(np.float32)
    scale = rng.uniform(0.5, 1.5, k).astype(np.float32)
    nbias = rng.standard_normal(k).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    wt, wd = Weight(dtype, w), oracle_roundtrip(orc, dtype, w).astype(np.float64)
    x = h.astype(np.float64)
    if kind == _lib.NORM_LAYERNORM:
        d = x - x.mean()
        x = d / np.sqrt(np.mean(d * d) + 1e-5) * scale + nbias
    else:
        x = x / np.sqrt(np.mean(x * x) + 1e-5) * scale
    pre = x @ wd + bias
    # a row that starts off a 16-byte boundary takes the general kernel
    hd, sd, nd, bd = dev(np.concatenate([np.zeros(shift, np.float32), h])), dev(scale), dev(nbias), dev(bias)
    y = DeviceArray((n // 2 if gated else n,), np.float32)
    _check(_lib.load().coeus_op_norm_gemv(wt.h, hd.ptr + 4 * shift, 1, kind, sd.ptr, nd.ptr, C.c_float(1e-5), bd.ptr, None,
                                          _lib.EPI_SILU_GATE if gated else 0, y.ptr, None, None))
    got = y.to_host()
    # f32 sums over k of the magnitudes, and the norm's own few roundings of the row
    e = (3 * k + 40) * 2.0 ** -24 * (np.abs(x) @ np.abs(wd) + np.abs(bias))
    if gated:
        g, u = pre[0::2], pre[1::2]
        want = g / (1 + np.exp(-g)) * u
        e = 1.1 * (e[0::2] * np.abs(u) + e[1::2] * np.abs(g)) + 2.0 ** -20 * np.abs(want) + 1e-6
    else:
        want = pre
    assert (np.abs(got - want) <= e).all()
