"""Prompts of fewer than 16 rows, whose attention writes the output projection's 16-bit rows itself: the same logits as the same
tokens one step at a time, for both 16-bit row types, both 16-bit caches and both head sizes."""
import numpy as np
import pytest

from coeus_amd import PLUGINS, Transformer250MConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weights", ["bf16", "q8_0"])
@pytest.mark.parametrize("cache", ["f16", "bf16"])
@pytest.mark.parametrize("heads", [2, 4])
@pytest.mark.parametrize("batch,n", [(1, 2), (3, 5), (1, 15), (16, 15)])
def test_as_step_by_step(weights, cache, heads, batch, n):
    cfg = Transformer250MConfig(hidden_dim=256, num_layers=2, num_heads=heads, intermediate_dim=512, vocab_size=300, max_seq_len=40, norm_scope="token",
                                weight_dtype=weights, kv_dtype=cache, max_batch=16)
    model = PLUGINS["transformer_model"].create_builder().build(cfg, seed=3)
    ids = np.random.default_rng(n).integers(0, 300, (batch, n), dtype=np.uint64)
    whole, steps = model.session(batch=batch, max_ctx=32), model.session(batch=batch, max_ctx=32)
    got = whole.prefill(ids)
    want = steps.prefill(ids[:, :1])
    for i in range(1, n):
        want = steps.decode(ids[:, i].copy())
    # the prompt rounds its activations, and quantised weights, to 16 bits (2^-9 for bf16, 2^-12 for f16, a dozen roundings over two layers)
    assert np.linalg.norm(got - want) < (12 * 2.0 ** -9 if weights == "bf16" else 12 * 2.0 ** -11) * np.linalg.norm(want)
    # and what it left in the cache serves the next step alike
    a, b = whole.decode(ids[:, 0].copy()), steps.decode(ids[:, 0].copy())
    assert np.linalg.norm(a - b) < (12 * 2.0 ** -9 if weights == "bf16" else 12 * 2.0 ** -11) * np.linalg.norm(b)
