"""Prompts of 2 - 16 rows on f32 weights (the decode matmul with the norms folded in, per row or over all rows, and the
cache rows from its epilogue) against the float64 model."""
import numpy as np
import pytest

import f64_model
from coeus_amd import Transformer250MConfig, TransformerModelPlugin

pytestmark = pytest.mark.gpu


def build(orc, **kw):
    kw = {"num_layers": 2, "num_heads": 16, "intermediate_dim": 608, **kw}
    cfg = Transformer250MConfig(vocab_size=150, max_seq_len=40, **kw)
    oc = orc.config_from_kwargs({k: getattr(cfg, k) for k in ("vocab_size", "max_seq_len", *kw)})
    params = orc.init_seeded(oc, 11)
    return TransformerModelPlugin().create_builder().build(cfg, parameters=params), oc, params


# 512: one chunk pair per wave; 768, 1024: registers of a wave full or not; 1088, 2080: the next size of the staging, and
# rows too long for it
@pytest.mark.parametrize("hidden", [512, 768, 1024, 1088, 2080])
@pytest.mark.parametrize("scope", ["sequence", "token"])
def test_forward_matches_float64(orc, hidden, scope):
    model, oc, params = build(orc, hidden_dim=hidden, norm_scope=scope)
    rng = np.random.default_rng(hidden)
    for rows in (2, 3, 4, 5, 8, 9, 16, 17):
        ids = rng.integers(0, 150, rows, dtype=np.uint64)
        want = f64_model.forward_all(oc, params, ids)
        got = model.forward_all(ids)
        # f32 sums of up to 2080 terms over two layers; the sinusoidal table's f32 angles (1e-6 at these positions)
        assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max(), rows


@pytest.mark.parametrize("batch,n", [(1, 7), (3, 5), (16, 1), (2, 8)])
@pytest.mark.parametrize("kv", ["f32", "bf16"])
def test_session_cache_rows(orc, batch, n, kv):
    """The rows that the epilogue wrote are read by the steps behind the prompt; a second prompt starts behind the first."""
    model, oc, params = build(orc, hidden_dim=512, norm_scope="token", max_batch=16, kv_dtype=kv)
    ids = np.random.default_rng(batch).integers(0, 150, (batch, 2 * n + 1), dtype=np.uint64)
    s = model.session(batch=batch, max_ctx=36)
    s.prefill(ids[:, :n], want_logits=False)
    s.prefill(ids[:, n:2 * n], want_logits=False)
    got = s.decode(ids[:, 2 * n])
    tol = 2e-5 if kv == "f32" else 2e-2  # (bf16 keys and values: 2^-9 each)
    for b in range(batch):
        want = f64_model.forward_all(oc, params, ids[b])[-1]
        assert np.abs(got[b] - want).max() <= tol * np.abs(want).max(), b


# biases of a layer whose lengths are no multiple of four: behind them no vector starts on 16 bytes unless it is padded
@pytest.mark.parametrize("scope", ["sequence", "token"])
@pytest.mark.parametrize("kw", [dict(intermediate_dim=770), dict(intermediate_dim=609), dict(intermediate_dim=609, activation="silu_gated"),
                                dict(num_heads=3, head_dim=21), dict(num_heads=3, head_dim=21, intermediate_dim=611, use_bias=False)])
def test_vectors_behind_odd_lengths(orc, kw, scope):
    model, oc, params = build(orc, hidden_dim=512, num_layers=3, norm_scope=scope, **kw)
    rng = np.random.default_rng(len(kw))
    for rows in (1, 2, 5, 16, 17):
        ids = rng.integers(0, 150, rows, dtype=np.uint64)
        want = f64_model.forward_all(oc, params, ids)
        got = model.forward_all(ids)
        assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max(), rows  # (as above)


@pytest.mark.parametrize("hidden,rows", [(512, 2), (768, 5), (1024, 16), (1088, 9), (2048, 4), (2080, 2), (2080, 4)])
def test_whole_slice_far_from_zero(orc, hidden, rows):
    """Statistics over all rows of values 2000 standard deviations from zero.  Attention adds nothing here, so the norm in
    front of the feed-forward sees exactly the embedded rows; what comes behind is large against them and keeps its digits."""
    cfg = dict(hidden_dim=hidden, num_layers=1, use_bias=False)
    _, oc, params = build(orc, **cfg)
    rng = np.random.default_rng(hidden + rows)
    first, stride, rel = f64_model.offsets(oc)
    params = params.copy()

    def part(name, shape=None):
        at, size = rel[name]
        a = params[first + at:first + at + size]
        return a.reshape(shape) if shape else a

    table = params[:150 * hidden].reshape(150, hidden)
    table[:] = 1000 + 0.5 * rng.standard_normal(table.shape)
    part("wo")[:] = 0
    part("w_down")[:] = 1e5 * rng.standard_normal(part("w_down").size)
    model = TransformerModelPlugin().create_builder().build(
        Transformer250MConfig(vocab_size=150, max_seq_len=40, num_heads=16, intermediate_dim=608, **cfg), parameters=params)
    ids = rng.integers(0, 150, rows, dtype=np.uint64)
    x = (table[ids.astype(int)] + orc.positional_encoding(40, hidden)[:rows]).astype(np.float64)
    eps = np.float64(np.float32(oc.layer_norm_eps))

    def norm(x, scale, bias):
        # (the mean is rounded to f32 before it is subtracted, as where the norm is a launch of its own)
        return scale * (x - np.float64(np.float32(x.mean()))) / np.sqrt(x.var() + eps) + bias

    up = norm(x, part("ln2_s"), part("ln2_b")) @ part("w_up", (hidden, 608)).astype(np.float64)
    x = x + f64_model.gelu(up) @ part("w_down", (608, hidden)).astype(np.float64)
    at = first + stride
    x = norm(x, params[at:at + hidden], params[at + hidden:at + 2 * hidden])
    want = x @ params[at + 2 * hidden:at + 2 * hidden + 150 * hidden].reshape(hidden, 150).astype(np.float64)
    # a mean that is off by one f32 step (6e-5 of values that spread by 0.5) moves every normalised value by 1.2e-4;
    # f32 sums of the matmuls: a few 1e-7
    assert np.abs(model.forward_all(ids) - want).max() <= 5e-6 * np.abs(want).max()


# Attention of 1 - 15 new rows per sequence, a workgroup per row and head: alone, behind cached keys on both sides of one trip of the waves (64 and 128
# keys of 64 in f32 and 16 bits, 32 and 64 of 128) and of many
@pytest.mark.parametrize("heads,hd", [(2, 64), (3, 128)])
@pytest.mark.parametrize("kv", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("first,n,batch", [(0, 1, 2), (0, 2, 1), (0, 15, 3), (17, 15, 1), (18, 15, 2), (50, 14, 1), (58, 7, 1), (114, 14, 2), (115, 14, 1), (300, 9, 1)])
def test_few_rows_behind_cached_keys(orc, heads, hd, kv, first, n, batch):
    kw = dict(hidden_dim=heads * hd, num_layers=2, num_heads=heads, intermediate_dim=4 * hd, vocab_size=130, max_seq_len=first + n, norm_scope="token")
    oc = orc.config_from_kwargs(kw)
    params = orc.init_seeded(oc, n)
    model = TransformerModelPlugin().create_builder().build(Transformer250MConfig(**kw, kv_dtype=kv, max_batch=3), parameters=params)
    ids = np.random.default_rng(n + hd).integers(0, 130, (batch, first + n), dtype=np.uint64)
    s = model.session(batch=batch, max_ctx=first + n)
    if first:
        s.prefill(ids[:, :first], want_logits=False)
    got = s.prefill(ids[:, first:])
    tol = {"f32": 2e-5, "bf16": 2e-2, "f16": 3e-3}[kv]  # (f32 sums over two layers; keys and values of 2^-9 and 2^-12 each)
    for b in range(batch):
        want = f64_model.forward_all(oc, params, ids[b])[-1]
        assert np.abs(got[b] - want).max() <= tol * np.abs(want).max(), b
