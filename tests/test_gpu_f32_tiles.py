"""The f32 prompt matmul at the edges of its tiles, of a slice of k and of its shares, against float64."""
import ctypes as C

import numpy as np
import pytest

from coeus_amd import _lib
from coeus_amd.device import DeviceArray, synchronize
from coeus_amd.plugin import _check
from gpu_util import Weight, dev

pytestmark = pytest.mark.gpu

# A sum is at most 64 products long before it is added to those before it (up to 64 more sums for k <= 4096, then 8 waves' and 8 shares' sums): 160 roundings.
ROUNDINGS = 160 * 2.0 ** -24


def planned(k, n, m):
    out = _lib.CMatmulPlan()
    _check(_lib.load().coeus_plan_matmul(_lib.W_F32, k, n, m, 1, C.byref(out)))
    return out.tile_rows, out.tile_cols, out.waves, out.shares


# (tile rows, tile columns, waves, split): each kernel, with rows, columns and k at and beside its multiples
@pytest.mark.parametrize("k,n,m,expected", [
    (768, 768, 128, (32, 32, 8, False)), (4, 40, 17, (32, 32, 8, False)), (772, 201, 65, (32, 32, None, None)), (3072, 97, 33, (32, 32, None, True)),
    (768, 2304, 256, (32, 32, 4, False)), (3072, 768, 128, (32, 32, 4, True)), (836, 2305, 255, (32, 32, 4, False)),
    (768, 2304, 512, (64, 32, 8, False)), (3072, 768, 500, (64, 32, 8, True)), (764, 3071, 495, (64, 32, 8, False)),
    (768, 3072, 1024, (64, 64, 8, False)), (2052, 2050, 1001, (64, 64, 8, None)),
    (768, 20010, 1000, (128, 64, 8, False)), (60, 50257, 641, (64, 64, 8, False)), (284, 50257, 1000, (128, 64, 8, False)),
])
def test_products(k, n, m, expected):
    got = planned(k, n, m)
    assert all(e is None or e == g for e, g in zip(expected, got[:3] + (got[3] > 1,))), got
    rng = np.random.default_rng(k + n + m)
    w, a = Weight(_lib.W_F32, seed=7, shape=(k, n)), rng.standard_normal((m, k)).astype(np.float32)
    wt = w.dequantize().astype(np.float64)
    rows = np.unique(np.r_[0:min(m, 40), max(0, m - 40):m, rng.integers(0, m, 40)])
    out = w.gemm(dev(a))[rows]
    exact, size = a[rows].astype(np.float64) @ wt, np.abs(a[rows]).astype(np.float64) @ np.abs(wt)
    assert np.all(np.abs(out - exact) <= ROUNDINGS * size + 1e-30)


@pytest.mark.parametrize("k,n,m", [(100, 96, 33), (3072, 768, 70), (768, 2304, 512), (768, 3072, 1000)])
def test_epilogues(k, n, m):
    rng = np.random.default_rng(5)
    w, a = Weight(_lib.W_F32, seed=9, shape=(k, n)), rng.standard_normal((m, k)).astype(np.float32)
    d, b, r = dev(a), rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    exact, size = a.astype(np.float64) @ w.dequantize(), np.abs(a).astype(np.float64) @ np.abs(w.dequantize())
    out = w.gemm(d, bias=dev(b), residual=dev(r))
    assert np.all(np.abs(out - (exact + b + r)) <= ROUNDINGS * (size + np.abs(b) + np.abs(r)))
    g, u = exact[:, 0::2], exact[:, 1::2]
    out = w.gemm(d, epilogue=_lib.EPI_SILU_GATE)
    s = g / (1 + np.exp(-g))  # |silu'| < 1.1; 32 more roundings for exp, the quotient and the product
    assert np.all(np.abs(out - s * u) <= ROUNDINGS * (1.1 * size[:, 0::2] * np.abs(u) + np.abs(s) * size[:, 1::2]) + 32 * 2.0 ** -24 * np.abs(s * u) + 1e-12)


@pytest.mark.parametrize("k,n,m", [(100, 96, 33), (3072, 768, 70), (772, 2304, 515), (284, 50257, 1000)])
def test_what_is_not_finite_stays_in_its_row(k, n, m):
    rng = np.random.default_rng(6)
    w, a = Weight(_lib.W_F32, seed=9, shape=(k, n)), rng.standard_normal((m, k)).astype(np.float32)
    clean = w.gemm(dev(a))
    a[m - 1, k - 1], a[3, k - 2] = np.inf, np.nan
    out = w.gemm(dev(a))
    last = w.dequantize()[k - 1]
    assert np.array_equal(out[m - 1], np.where(last > 0, np.inf, -np.inf).astype(np.float32)) and np.all(np.isnan(out[3]))
    keep = np.setdiff1d(np.arange(m), [3, m - 1])
    assert np.array_equal(out[keep], clean[keep])


def test_rows_between_pieces():
    """An input that starts between two 16-byte pieces is multiplied like one that does not."""
    k, n, m = 768, 96, 40
    rng = np.random.default_rng(8)
    w, a = Weight(_lib.W_F32, seed=9, shape=(k, n)), rng.standard_normal((m, k)).astype(np.float32)
    exact, size = a.astype(np.float64) @ w.dequantize(), np.abs(a).astype(np.float64) @ np.abs(w.dequantize())
    shifted = dev(np.r_[np.float32(0), a.ravel()])
    out = DeviceArray((m, n), np.float32)
    _check(_lib.load().coeus_op_gemm(w.h, C.c_void_p(C.cast(shifted.ptr, C.c_void_p).value + 4), m, None, None, _lib.EPI_NONE, out.ptr, None))
    synchronize()
    out = out.to_host()
    assert np.all(np.abs(out - exact) <= 256 * 2.0 ** -24 * size)  # (sums of up to 192 products in each of four waves)
