"""The f32 prompt matmul at the edges of its tiles, of a slice of k, of its shares and of 16-byte pieces of what it reads and writes, against float64."""
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


# outputs that whole groups of four fill and that they do not (a row of 2050 weight rows gives 1025 gated ones); one share and several; all from 17 rows on
@pytest.mark.parametrize("k,n,m", [(100, 98, 33), (3072, 104, 40), (768, 2050, 300), (772, 2304, 257)])
@pytest.mark.parametrize("epilogue", [_lib.EPI_NONE, _lib.EPI_GELU, _lib.EPI_SILU_GATE])
@pytest.mark.parametrize("off", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (3, 2, 1)])
def test_epilogues_between_pieces(k, n, m, epilogue, off):
    """Results, bias and residual that start between two 16-byte pieces (by `off` floats), with every activation."""
    rng = np.random.default_rng(n + m)
    gated = epilogue == _lib.EPI_SILU_GATE
    w, a = Weight(_lib.W_F32, seed=9, shape=(k, n)), rng.standard_normal((m, k)).astype(np.float32)
    b, r = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n // 2 if gated else n)).astype(np.float32)
    at = lambda x, o: dev(np.r_[np.zeros(o, np.float32), x.ravel()])  # noqa: E731
    da, out, db, dr = dev(a), at(np.full(r.size + 4, 7, np.float32), off[0]), at(b, off[1]), at(r, off[2])
    ptr = lambda x, o: C.c_void_p(C.cast(x.ptr, C.c_void_p).value + 4 * o)  # noqa: E731
    _check(_lib.load().coeus_op_gemm(w.h, da.ptr, m, ptr(db, off[1]), ptr(dr, off[2]), epilogue, ptr(out, off[0]), None))
    synchronize()
    got = out.to_host()
    assert not got[:off[0]].any() and np.all(got[off[0] + r.size:] == 7)
    got = got[off[0]:off[0] + r.size].reshape(r.shape)
    size, pb = ROUNDINGS * (np.abs(a).astype(np.float64) @ np.abs(w.dequantize()) + np.abs(b)), a.astype(np.float64) @ w.dequantize() + b
    # GELU has slopes of up to 1.13, SiLU of 1.1; some 16 roundings each of their own, the residual one
    if gated:
        g, u = pb[:, 0::2], pb[:, 1::2]
        s = g / (1 + np.exp(-g))
        want, bound = s * u, 1.1 * size[:, 0::2] * np.abs(u) + np.abs(s) * size[:, 1::2] + 2.0 ** -20 * np.abs(s * u) + 1e-6
    elif epilogue == _lib.EPI_GELU:
        want, bound = 0.5 * pb * (1 + np.tanh(0.7978845608028654 * pb * (1 + 0.044715 * pb * pb))), 1.2 * size + 2.0 ** -20 * (1 + np.abs(pb))
    else:
        want, bound = pb, size
    assert np.all(np.abs(got - (want + r)) <= bound + 2.0 ** -23 * (np.abs(want) + np.abs(r)))
