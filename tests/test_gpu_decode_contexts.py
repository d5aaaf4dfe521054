"""Decode attention (split context): a session's step logits against the prompt pass over the same tokens, at contexts
around the kernel's tiles and splits."""
import numpy as np
import pytest

import f64_model
from coeus_amd import Transformer250MConfig, TransformerModelPlugin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,hd", [(2, 64), (3, 128)])
@pytest.mark.parametrize("max_ctx", [140, 520, 1300, 2300])
@pytest.mark.parametrize("kv", ["f32", "f16", "bf16"])
def test_steps_match_prompt_pass(heads, hd, max_ctx, kv):
    cfg = Transformer250MConfig(hidden_dim=heads * hd, num_layers=2, num_heads=heads, intermediate_dim=256, vocab_size=160,
                                max_seq_len=max_ctx, norm_scope="token", max_batch=3, kv_dtype=kv)
    model = TransformerModelPlugin().create_builder().build(cfg, seed=5)
    rng = np.random.default_rng(max_ctx + hd)
    # 16-bit: 32 - 128 (16 - 64) keys of 64 (128) a wave, four or eight waves, one split or several of 64 keys and more
    for ctx in (1, 2, 31, 32, 33, 64, 127, 128, 129, 255, 257, 512, 513, 1025, 2049, max_ctx):
        if ctx > max_ctx:
            continue
        ids = rng.integers(0, cfg.vocab_size, (3, ctx), dtype=np.uint64)
        s = model.session(batch=3, max_ctx=max_ctx)
        if ctx > 1:
            s.prefill(ids[:, :-1], want_logits=False)
        got = s.decode(ids[:, -1])
        s.close()
        for b in range(3):
            want = model.forward(ids[b])
            # f32: two orders of sums over two layers, a few roundings of 2^-24 each (1e-6 measured).  16-bit caches: the
            # prompt pass also rounds queries and weights of the softmax to the cache's type, 2^-11 and 2^-8 relative
            tol = {"f32": 2e-5, "f16": 2e-3, "bf16": 1.6e-2}[kv]
            assert np.abs(got[b] - want).max() <= tol * np.abs(want).max(), (ctx, b)


@pytest.mark.parametrize("heads,hd,max_ctx", [(4, 64, 1024), (4, 64, 1025), (4, 128, 512), (8, 64, 1030), (9, 64, 1500), (9, 128, 700),
                                              (2, 64, 1000), (2, 128, 1030), (3, 64, 1025), (6, 128, 640)])
@pytest.mark.parametrize("kv", ["f32", "f16"])
def test_many_heads_match_prompt_pass(heads, hd, max_ctx, kv):
    # 16 sequences: 64 heads and up to 128 KiB of keys a head whole, 64 - 128 heads split beyond that, more than 128 whole;
    # 32 heads in four splits up to 1024 keys (f32: eight) and eight beyond, 48 in four, 96 in two
    cfg = Transformer250MConfig(hidden_dim=heads * hd, num_layers=1, num_heads=heads, intermediate_dim=256, vocab_size=160,
                                max_seq_len=max_ctx, norm_scope="token", max_batch=16, kv_dtype=kv)
    model = TransformerModelPlugin().create_builder().build(cfg, seed=6)
    ids = np.random.default_rng(max_ctx).integers(0, cfg.vocab_size, (16, max_ctx), dtype=np.uint64)
    s = model.session(batch=16, max_ctx=max_ctx)
    s.prefill(ids[:, :-1], want_logits=False)
    got = s.decode(ids[:, -1])
    s.close()
    tol = {"f32": 2e-5, "f16": 2e-3}[kv]  # as above
    for b in (0, 7, 15):
        want = model.forward(ids[b])
        assert np.abs(got[b] - want).max() <= tol * np.abs(want).max(), b


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("ctx", [130, 300, 700])
def test_keys_that_score_minus_infinity(orc, hd, ctx):
    """Keys 64 on, up to the last, overflow to a score of -inf against the last query: they weigh nothing, also where a wave or
    a split has only such keys.  The others' scores are finite and far apart."""
    H, V = 2 * hd, 60
    kw = dict(hidden_dim=H, num_layers=1, num_heads=2, intermediate_dim=64, vocab_size=V, max_seq_len=ctx, norm_scope="token", use_bias=False)
    oc = orc.config_from_kwargs(kw)
    params = orc.init_seeded(oc, 9)
    rng = np.random.default_rng(ctx)
    table = params[:V * H].reshape(V, H)
    table[:] = rng.standard_normal((V, H))
    table[:, 0], table[:30, 1], table[30:, 1] = 10.0, 0.1 * table[:30, 1], -1000.0
    first, _, rel = f64_model.offsets(oc)
    for name, row, scale in (("wq", 0, 1e20), ("wk", 1, 2e17)):
        w = params[first + rel[name][0]:first + rel[name][0] + H * H].reshape(H, H)
        w[:], w[row, 0], w[row, hd] = 0, scale, scale  # the first element of each head
    ids = np.concatenate([rng.integers(0, 30, 64), rng.integers(30, V, ctx - 65), rng.integers(0, 30, 1)]).astype(np.uint64)
    model = TransformerModelPlugin().create_builder().build(Transformer250MConfig(**kw), parameters=params)
    s = model.session(batch=1, max_ctx=ctx)
    s.prefill(ids[None, :-1], want_logits=False)
    got, want = s.decode(ids[-1:])[0], f64_model.forward_all(oc, params, ids)[-1]
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()  # (f32, as above)
