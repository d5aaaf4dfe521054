"""The prompt matmul on up to 16 rows of 16-bit operands, which takes the decode step's kernels: float64 of the rounded operands, at
the edges of the padded row counts, of a tile's 16 outputs, of whole chunks of k, and of the shares that bf16 tiles are dealt in; and the stacks
that do not take them."""
import numpy as np
import pytest

from coeus_amd import PLUGINS, LayeredConfig, _lib
from gpu_util import Weight, dev, oracle_roundtrip
from test_matmul_plan import plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("dtype,k,n", [
    (_lib.W_BF16, 64, 2), (_lib.W_BF16, 192, 34), (_lib.W_BF16, 768, 2304), (_lib.W_BF16, 1024, 1022), (_lib.W_BF16, 2112, 4130), (_lib.W_BF16, 3072, 768),
    (_lib.W_BF16, 5632, 2048), (_lib.W_BF16, 4096, 4610), (_lib.W_Q8_0, 128, 18), (_lib.W_Q8_0, 768, 2302), (_lib.W_Q8_0, 1152, 4100), (_lib.W_Q8_0, 3072, 770),
    (_lib.W_Q4_0, 128, 4098), (_lib.W_Q4_0, 1280, 130), (_lib.W_Q4_0, 2048, 8190), (_lib.W_Q4_0, 8192, 258)])
def test_matches_float64(orc, dtype, k, n, rows):
    rng = np.random.default_rng(k + n + rows)
    w = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    a = rng.standard_normal((rows, k)).astype(np.float32)
    bias, res = (rng.standard_normal(s).astype(np.float32) for s in (n, (rows, n)))
    wt, wd = Weight(dtype, w), oracle_roundtrip(orc, dtype, w)
    bf = dtype == _lib.W_BF16
    assert plan(dtype, k, n, rows, 1).kernel == (b"gemv_mfma_kernel" if bf else b"gemv_rows_kernel")
    ar, wr = (x.astype(np.float64) for x in ((orc.bf16_round(a), wd) if bf else (a.astype(np.float16), wd.astype(np.float16))))
    pre = ar @ wr
    e = (k + 20) * 2.0 ** -24 * (np.abs(ar) @ np.abs(wr))  # f32 sums over k of the magnitudes
    da = dev(a)
    got = wt.gemm(da)
    assert (np.abs(got - pre) <= e).all() and np.array_equal(got, wt.gemm(da))
    # a GELU has slopes of up to 1.13 and three roundings of its own, bias and residual one each
    pb = pre + bias
    want = 0.5 * pb * (1 + np.tanh(0.7978845608028654 * pb * (1 + 0.044715 * pb * pb))) + res
    got = wt.gemm(da, bias=dev(bias), residual=dev(res), epilogue=_lib.EPI_GELU)
    assert (np.abs(got - want) <= 1.2 * e + 2.0 ** -20 * (1 + np.abs(pb) + np.abs(res))).all()
    g, u = pre[:, 0::2], pre[:, 1::2]
    want = g / (1 + np.exp(-g)) * u
    got = wt.gemm(da, epilogue=_lib.EPI_SILU_GATE)
    assert (np.abs(got - want) <= 1.1 * (e[:, 0::2] * np.abs(u) + e[:, 1::2] * np.abs(g)) + 2.0 ** -20 * np.abs(want) + 1e-6).all()


def test_rows_do_not_meet(orc):
    """A row that is not finite leaves the others as they were."""
    rng = np.random.default_rng(0)
    for dtype in (_lib.W_BF16, _lib.W_Q4_0):
        wt = Weight(dtype, (rng.standard_normal((1024, 520)) * 0.05).astype(np.float32))
        a = rng.standard_normal((5, 1024)).astype(np.float32)
        clean = wt.gemm(dev(a))
        a[2, 7] = np.inf
        got = wt.gemm(dev(a))
        assert np.array_equal(np.delete(got, 2, 0), np.delete(clean, 2, 0)) and not np.isfinite(got[2]).any()


def stack(mixer, attention):
    mlp = {"kind": "dense", "ff": 512}
    layers = [dict(mixer, mlp=mlp), dict(attention, mlp=mlp)]
    cfg = {"architecture": "Bofirax", "vocab": 300, "width": 1024, "norm": {"eps": 1e-5}, "layers": layers}
    return PLUGINS["layered_model"].create_builder().build(LayeredConfig(cfg, max_seq_len=32, max_batch=1), seed=5)


@pytest.mark.parametrize("rows", [2, 5, 16])
def test_stacks_with_a_delta_rule_keep_the_longer_prompts_sums(rows):
    """Such a stack's rows are, bit for bit, those of a prompt of one token more than the decode step's kernels take; one without it has other sums."""
    latent = {"type": "latent_attention", "mixer": dict(heads=4, dim=128, vdim=128, q_rank=192, kv_rank=128, scale=128 ** -0.5, mask={"size": 32})}
    delta = {"type": "delta", "mixer": dict(heads=4, kv_heads=2, dim=128, vdim=128, conv=4)}
    ids = np.random.default_rng(1).integers(0, 300, (1, 17), dtype=np.uint64)
    for mixer, same in ((delta, True), (latent, False)):
        model = stack(mixer, latent)
        few, more = (model.session(batch=1, max_ctx=32).feed(ids[:, :n], want=(0,), want_residuals=True)[1] for n in (rows, 17))
        assert np.array_equal(few, more[:, :rows]) == same
