"""f32 prompts of few workgroups: attention of 32 queries whose waves share the keys, cache rows from the q|k|v epilogue, norms over the
whole slice; float64 of the same model at the edges of the tiles and of the waves' turns, in one piece and in two."""
import numpy as np
import pytest

import f64_model
from coeus_amd import Transformer250MConfig, TransformerModelPlugin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,hd", [(2, 64), (3, 128)])
@pytest.mark.parametrize("scope", ["token", "sequence"])
@pytest.mark.parametrize("n,first", [(17, 0), (31, 0), (32, 0), (33, 0), (64, 30), (65, 33), (129, 100), (161, 20), (290, 129)])
def test_matches_float64(orc, heads, hd, scope, n, first):
    first = 0 if scope == "sequence" else first  # (a norm over the whole slice has no cache)
    kw = dict(hidden_dim=heads * hd, num_layers=2, num_heads=heads, intermediate_dim=4 * hd, vocab_size=130, max_seq_len=n, norm_scope=scope)
    oc = orc.config_from_kwargs(kw)
    params = orc.init_seeded(oc, n)
    ids = np.random.default_rng(n + hd).integers(0, 130, n, dtype=np.uint64)
    want = f64_model.forward_all(oc, params, ids)
    model = TransformerModelPlugin().create_builder().build(Transformer250MConfig(**kw), parameters=params)
    got = model.forward_all(ids)
    # f32: sums of up to 4 hd terms over two layers, a few roundings of 2^-24 each (2e-6 measured)
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()
    if first:
        s = model.session(batch=1, max_ctx=n)
        s.prefill(ids[None, :first], want_logits=False)
        last = s.prefill(ids[None, first:])[0]
        assert np.abs(last - want[-1]).max() <= 2e-5 * np.abs(want[-1]).max()
