"""The 16-bit prompt matmul on 256x256 tiles: one to nine slices of k, shares of k, the gated epilogues to 32 and to 16 bits; float64 of the same
operands, each launch's kernel asserted, so that a change of the rules does not empty a test."""
import ctypes as C

import numpy as np
import pytest

from coeus_amd import _lib
from coeus_amd.device import DeviceArray, synchronize
from coeus_amd.plugin import _check
from gpu_util import Weight, dev, rel_err
from test_matmul_plan import plan

pytestmark = pytest.mark.gpu


def _operands(orc, dtype, a, wd):
    if dtype == _lib.W_BF16:
        return orc.bf16_round(a).astype(np.float64), wd.astype(np.float64)
    return a.astype(np.float16).astype(np.float64), wd.astype(np.float16).astype(np.float64)


def _gelu(x):
    return 0.5 * x * (1 + np.tanh(0.7978845608028654 * x * (1 + 0.044715 * x * x)))


def _plain_gelu_gated(orc, dtype, m, k, n, rows):
    rng = np.random.default_rng(k + m)
    wt = Weight(dtype, seed=7, shape=(k, n))
    a = rng.standard_normal((m, k)).astype(np.float32)
    bias, res = (rng.standard_normal(n) * 0.1).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    ar, wd = _operands(orc, dtype, a[rows], wt.dequantize())
    pre = ar @ wd
    da = dev(a)
    # (the bar of the other prompt matmul tests: f32 sums over k)
    assert rel_err(wt.gemm(da)[rows], pre) < 2e-5
    assert rel_err(wt.gemm(da, bias=dev(bias), residual=dev(res), epilogue=_lib.EPI_GELU)[rows], _gelu(pre + bias) + res[rows]) < 2e-5
    g, u = pre[:, 0::2], pre[:, 1::2]
    assert rel_err(wt.gemm(da, epilogue=_lib.EPI_SILU_GATE)[rows], g / (1 + np.exp(-g)) * u) < 2e-5


# 20 x 20 tiles, the last ones' rows and columns past the end; the pipeline keeps three A slices and two W slices in flight: fewer, as many, more
@pytest.mark.parametrize("dtype", [_lib.W_BF16, _lib.W_Q8_0])
@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 576])
def test_slices(orc, dtype, k):
    p = plan(dtype, k, 5100, 5000, 1)
    assert (p.kernel, p.shares, p.tail_shares) == (b"gemm_h256k64_kernel", 1, 1)
    _plain_gelu_gated(orc, dtype, 5000, k, 5100, np.unique(np.r_[0:5000:331, 31, 32, 127, 128, 255, 256, 4863, 4864, 4991, 4992, 4999]))


@pytest.mark.parametrize("dtype", [_lib.W_BF16, _lib.W_Q8_0])
def test_shares_of_k(orc, dtype):
    p = plan(dtype, 11008, 4096, 300, 1)
    assert p.kernel == b"gemm_h256k64_kernel" and p.shares >= 4
    _plain_gelu_gated(orc, dtype, 300, 11008, 4096, np.unique(np.r_[0:300:23, 255, 256, 299]))


def _gemm16(wt, da, epilogue, limit, bf16, ld):
    m, n_eff = da.shape[0], wt.n // 2
    out = DeviceArray((m, ld), np.uint16)
    _check(_lib.load().coeus_op_gemm16(wt.h, da.ptr, m, epilogue, limit, bf16, ld, out.ptr, None))
    synchronize()
    return out.to_host()[:, :n_eff]


# 20 x 20 tiles, rows that end inside a block of 32; all columns inside (5120), or the last tile's past the end.  Rows of a multiple of 8 values are
# stored from the accumulators, others through LDS: the same bits
@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("epilogue", [_lib.EPI_SILU_GATE, _lib.EPI_CLAMP_GATE])
@pytest.mark.parametrize("k,n", [(64, 5120), (192, 5120), (128, 5036)])
def test_gates_to_16_bits(orc, bf16, epilogue, k, n):
    m, limit = 4999, 1.3
    assert plan(_lib.W_BF16, k, n, m, 1).kernel == b"gemm_h256k64_kernel"
    rng = np.random.default_rng(k + n)
    wt = Weight(_lib.W_BF16, (rng.standard_normal((k, n)) * 2 / np.sqrt(k)).astype(np.float32))
    a = orc.bf16_round(rng.standard_normal((m, k)).astype(np.float32))
    da = dev(a)
    z = a.astype(np.float64) @ wt.dequantize().astype(np.float64)
    g, u = z[:, 0::2], z[:, 1::2]
    if epilogue == _lib.EPI_CLAMP_GATE:
        g, u = np.minimum(g, limit), np.clip(u, -limit, limit)
        want = g / (1 + np.exp(-1.702 * g)) * (u + 1)
    else:
        want = g / (1 + np.exp(-g)) * u
    bits = _gemm16(wt, da, epilogue, limit, bf16, n // 2 + (-(n // 2)) % 8)
    got = (bits.astype(np.uint32) << 16).view(np.float32) if bf16 else bits.view(np.float16)
    # half a unit of 8 or 11 bits (2^-8 or 2^-11 of a value just above a power of two), and the f32 value's own error: sums of k products of size
    # 4 / k, slopes of at most 2.5
    assert (np.abs(got.astype(np.float64) - want) <= np.abs(want) * 2.0 ** (-8 if bf16 else -11) + 1e-5).all()
    assert np.array_equal(_gemm16(wt, da, epilogue, limit, bf16, n // 2 + 4 + (-(n // 2)) % 8), bits)
    f32 = DeviceArray((m, n // 2), np.float32)
    if epilogue == _lib.EPI_SILU_GATE:
        _check(_lib.load().coeus_op_gemm(wt.h, da.ptr, m, None, None, epilogue, f32.ptr, None))
    else:
        _check(_lib.load().coeus_op_matmul_limited(wt.h, da.ptr, m, 1, epilogue, limit, f32.ptr, None))
    synchronize()
    v = f32.to_host()
    assert np.abs(v - want).max() <= 1e-5 * np.abs(want).max()
    # (f16: one instruction multiplies and rounds, which is another value where the product in f32 lies on the middle between two: one in 2^13)
    rounded = (orc.bf16_round(v).view(np.uint32) >> 16).astype(np.uint16) if bf16 else v.astype(np.float16).view(np.uint16)
    assert (bits != rounded).mean() <= (0 if bf16 else 2.0 ** -12) and np.abs(bits.astype(int) - rounded).max() <= 1


def test_gemm16_refuses():
    wt = Weight(_lib.W_BF16, seed=1, shape=(64, 128))
    lib, buf = _lib.load(), DeviceArray((128, 128), np.float32)
    for epilogue, limit, ld in [(0, 0, 127), (_lib.EPI_SILU_GATE, 0, 63), (_lib.EPI_CLAMP_GATE, 0.0, 64), (9, 1.0, 128)]:
        assert lib.coeus_op_gemm16(wt.h, buf.ptr, 8, epilogue, limit, 1, ld, buf.ptr, None) != 0
