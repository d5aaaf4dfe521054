"""The decode matmul of several rows on dense weights (matrix cores; with bf16 weights the activations as three bf16
each) against a float64 product of the same weights and activations."""
import ctypes as C

import numpy as np
import pytest

import layered_util as L
from coeus_amd import PLUGINS, Transformer250MConfig, _lib, load_model
from coeus_amd.device import DeviceArray
from coeus_amd.plugin import _check
from gpu_util import Weight, dev, oracle_roundtrip

pytestmark = pytest.mark.gpu


def bound(x, w, k):
    """Worst case of f32 sums in any order: three terms per k, each sum rounded once (2^-24), of the magnitudes."""
    return 3 * k * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(w)) + 1e-30


# one pair of chunks for one wave; waves with unequal shares; shares of 1, 2, 3, 4 and more pairs; weight rows that
# do not fill a tile; more tiles than workgroups (16 * 4096 rows); both sides of the lines up to which one, two and three rows
# stay with a wave per weight row
@pytest.mark.parametrize("k,n", [(64, 1), (64, 16), (192, 33), (320, 50), (768, 130), (1024, 17), (2048, 70), (2112, 40), (3072, 31),
                                 (4096, 48), (5632, 20), (11008, 18), (128, 65552), (1024, 5003),
                                 (256, 1000), (1024, 1024), (1088, 1040), (1024, 2056), (4608, 33), (5184, 33), (16384, 18)])
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


# Tiles of 4 and 8 weight rows whose lines are parts of k: tiles that end inside the matrix, one pair a wave, shares of one, two and more pairs,
# several tiles a workgroup, gated pairs, and one more row of weights or 64 of k than the rule allows
@pytest.mark.parametrize("k,n", [(128, 5), (768, 6), (1024, 1022), (1280, 1024), (2816, 1030), (3072, 7), (4096, 4098), (5632, 2046), (6144, 4100), (8192, 1026), (4160, 1000), (2176, 4102), (2560, 8210)])
@pytest.mark.parametrize("batch", [2, 3, 4, 5, 8])
@pytest.mark.parametrize("dtype", [_lib.W_BF16, _lib.W_F32])
def test_parts_of_k(orc, dtype, k, n, batch):
    rng = np.random.default_rng(k + 31 * n + batch)
    w = (rng.standard_normal((k, n)) * 0.02).astype(np.float32)
    x = (rng.standard_normal((batch, k)) * np.exp2(rng.integers(-20, 20, (batch, k)))).astype(np.float32)
    wt, wd = Weight(dtype, w), oracle_roundtrip(orc, dtype, w).astype(np.float64)
    assert (np.abs(wt.gemv(dev(x)) - x.astype(np.float64) @ wd) <= bound(x, wd, k)).all()
    if n % 2 == 0:
        x = rng.standard_normal((batch, k)).astype(np.float32)
        pre, e = x.astype(np.float64) @ wd, bound(x, wd, k)
        g, u = pre[:, 0::2], pre[:, 1::2]
        want = g / (1 + np.exp(-g)) * u
        lim = 1.1 * (e[:, 0::2] * np.abs(u) + e[:, 1::2] * np.abs(g)) + 2.0 ** -20 * np.abs(want) + 1e-6
        assert (np.abs(wt.gemv(dev(x), epilogue=_lib.EPI_SILU_GATE) - want) <= lim).all()


# Long rows in shares that differ by a pair: eight waves of several tiles a workgroup, twelve where rows are 32 KiB apart
@pytest.mark.parametrize("dtype,k,n", [(_lib.W_F32, 4128, 5130), (_lib.W_F32, 8192, 2070), (_lib.W_BF16, 2112, 5130), (_lib.W_BF16, 16384, 2070), (_lib.W_F32, 16384, 2050)])
@pytest.mark.parametrize("batch", [1, 2, 4, 8, 16])
def test_waves_of_long_rows(orc, dtype, k, n, batch):
    rng = np.random.default_rng(k + batch)
    w = (rng.standard_normal((k, n), np.float32) * np.float32(0.02))
    x = (rng.standard_normal((batch, k)) * np.exp2(rng.integers(-20, 20, (batch, k)))).astype(np.float32)
    wt, wd = Weight(dtype, w), oracle_roundtrip(orc, dtype, w).astype(np.float64)
    assert (np.abs(wt.gemv(dev(x)) - x.astype(np.float64) @ wd) <= bound(x, wd, k)).all()


@pytest.mark.parametrize("dtype,rows", [(_lib.W_F32, 2), (_lib.W_F32, 5), (_lib.W_F32, 16), (_lib.W_F32, 17), (_lib.W_BF16, 5)])
def test_timed_matmul_is_the_one_that_runs(dtype, rows):
    """What the repeated, timed launches leave is the bits of the plain call: the same kernel, in the same order of sums."""
    rng = np.random.default_rng(rows)
    w = Weight(dtype, (rng.standard_normal((3072, 768)) * 0.02).astype(np.float32))
    x, y, ms = dev(rng.standard_normal((rows, 3072)).astype(np.float32)), DeviceArray((rows, 768)).zero_(), C.c_float()
    _check(_lib.load().coeus_op_gemm_timed(w.h, x.ptr, rows, 0, y.ptr, 3, C.byref(ms), None))
    assert ms.value > 0 and np.array_equal(y.to_host(), w.gemm(x))


# A norm in front: the shortest rows that give each of 16 waves a pair of chunks, the longest whose staging fits for 2, 4, 8 and 16 rows,
# both sides of the lengths at which the staging changes (1024, 2048), shares of up to 8 pairs, and three in flight (a share of
# three, more than 256 tiles)
@pytest.mark.parametrize("kind", [_lib.NORM_LAYERNORM, _lib.NORM_RMSNORM])
@pytest.mark.parametrize("dtype,batch,k,n", [
    (_lib.W_F32, 16, 512, 18), (_lib.W_F32, 9, 768, 34), (_lib.W_F32, 16, 864, 50), (_lib.W_F32, 8, 1024, 18), (_lib.W_F32, 5, 1056, 40),
    (_lib.W_F32, 8, 1600, 34), (_lib.W_F32, 4, 2048, 18), (_lib.W_F32, 3, 2080, 40), (_lib.W_F32, 4, 2688, 18), (_lib.W_F32, 2, 4064, 34),
    (_lib.W_F32, 2, 1536, 4200), (_lib.W_F32, 6, 1504, 4106), (_lib.W_BF16, 8, 1024, 34), (_lib.W_BF16, 5, 1600, 18), (_lib.W_BF16, 4, 2112, 40),
    (_lib.W_BF16, 3, 2688, 18), (_lib.W_BF16, 2, 2048, 34), (_lib.W_BF16, 2, 2112, 4200), (_lib.W_BF16, 2, 4032, 4106)])
def test_norm_in_front(orc, dtype, batch, k, n, kind):
    rng = np.random.default_rng(k + n + kind)
    w = (rng.standard_normal((k, n)) * 0.05).astype(np.float32)
    h = (rng.standard_normal((batch, k)) * 3 + 1).astype(np.float32)
    scale, nbias = rng.uniform(0.5, 1.5, k).astype(np.float32), rng.standard_normal(k).astype(np.float32)
    wt, wd = Weight(dtype, w), oracle_roundtrip(orc, dtype, w).astype(np.float64)
    x = h.astype(np.float64)
    if kind == _lib.NORM_LAYERNORM:
        x = x - x.mean(1, keepdims=True)
    x = x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5) * scale + (nbias if kind == _lib.NORM_LAYERNORM else 0)
    pre = x @ wd
    # f32 sums over k of the magnitudes, and the norm's own few roundings of the row
    e = (3 * k + 40) * 2.0 ** -24 * (np.abs(x) @ np.abs(wd))
    sd, nd = dev(scale), dev(nbias)
    for shift, gated in ((0, False), (0, True), (1, False)):  # (rows off a 16-byte boundary take the general kernel)
        hd, y, fused = dev(np.concatenate([np.zeros(shift, np.float32), h.ravel()])), DeviceArray((batch, n // 2 if gated else n)), C.c_int()
        _check(_lib.load().coeus_op_norm_gemv(wt.h, hd.ptr + 4 * shift, batch, kind, sd.ptr, nd.ptr, C.c_float(1e-5), None, None,
                                              _lib.EPI_SILU_GATE if gated else 0, y.ptr, C.byref(fused), None))
        want, lim = pre, e
        if gated:
            g, u = pre[:, 0::2], pre[:, 1::2]
            want = g / (1 + np.exp(-g)) * u
            lim = 1.1 * (e[:, 0::2] * np.abs(u) + e[:, 1::2] * np.abs(g)) + 2.0 ** -20 * np.abs(want) + 1e-6
        assert fused.value == 1 and (np.abs(y.to_host() - want) <= lim).all(), (shift, gated)


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


@pytest.mark.parametrize("batch,k,n", [(1, 4096, 40), (1, 1024, 16400), (2, 256, 40), (5, 1024, 33), (16, 2048, 70)])
@pytest.mark.parametrize("dtype", [_lib.W_BF16, _lib.W_F32])
def test_infinite_weights(orc, dtype, batch, k, n):
    rng = np.random.default_rng(k + batch)
    w = (rng.standard_normal((k, n)) * 0.02).astype(np.float32)
    x = rng.standard_normal((batch, k)).astype(np.float32)
    x[:, 1] = 1.0  # (one bf16: its other two pieces are zero)
    w[1, 3], w[k - 1, 7], w[5, n - 1] = np.inf, -np.inf, np.inf
    w[9, 11] = 3.4e38  # rounds to an infinite bf16
    wd = oracle_roundtrip(orc, dtype, w).astype(np.float64)
    want = x.astype(np.float64) @ np.where(np.isinf(wd), 0, wd)
    bad = np.isinf(wd).any(0)
    for r, c in np.argwhere(np.isinf(wd)):
        want[:, c] = wd[r, c] * np.sign(x[:, r])
    got = Weight(dtype, w).gemv(dev(x))
    assert np.array_equal(got[:, bad], want[:, bad].astype(np.float32))
    ok = np.setdiff1d(np.flatnonzero(~bad), [11])
    assert (np.abs(got[:, ok] - want[:, ok]) <= bound(x, np.where(np.isinf(wd), 0, wd), k)[:, ok]).all()


def test_infinite_weights_of_models(orc, tmp_path):
    """Columns of the output projection with an infinite value each: infinite logits (capped ones: the cap), not NaN.  One
    activation in 256 has a third bf16 that is zero; here 1120 and 3200 of them meet an infinity."""
    rng = np.random.default_rng(3)
    kw = dict(hidden_dim=1024, num_layers=1, num_heads=16, intermediate_dim=320, vocab_size=90, max_seq_len=16, norm_scope="token", weight_dtype="bf16",
              kv_dtype="bf16", max_batch=16)
    oc = orc.config_from_kwargs(kw)
    params = orc.init_seeded(oc, 5)
    out = params[orc.layout(oc).output_proj_offset:][:1024 * 90].reshape(1024, 90)
    out[np.arange(20, 90) * 2, np.arange(20, 90)] = np.inf
    s = PLUGINS["transformer_model"].create_builder().build(Transformer250MConfig(**kw), parameters=params).session(batch=16, max_ctx=16)
    ids = rng.integers(0, 90, (16, 4), dtype=np.uint64)
    s.prefill(ids)
    y = s.decode(ids[:, 0])
    assert np.isinf(y[:, 20:]).all() and np.isfinite(y[:, :20]).all()

    cfg = L.CONFIGS["hyper_wide"]
    w = L.weights(cfg, 6)
    w["head"][np.arange(200), np.arange(200) % 128] = np.inf
    model = load_model(L.write_folder(str(tmp_path / "m"), cfg, w), max_seq_len=16, max_batch=16)
    s = model.session(batch=16, max_ctx=16)
    ids = rng.integers(0, 200, (16, 4), dtype=np.uint64)
    s.prefill(ids)
    y = s.decode(ids[:, 0])
    assert (np.abs(y) == 8.0).all()
