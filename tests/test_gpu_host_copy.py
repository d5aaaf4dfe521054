"""Logits on their way to the caller: sizes around the pinned slots (1 MiB, four of them) and results that start in the
middle of a page, against the same rows fetched one at a time."""
import ctypes as C

import numpy as np
import pytest

from coeus_amd import Transformer250MConfig, TransformerModelPlugin, _lib
from coeus_amd.plugin import _check

pytestmark = pytest.mark.gpu


# 4 * vocab bytes a row: 4096 in all; one slot, and one value more; four slots; nine and a bit
@pytest.mark.parametrize("vocab,rows", [(512, 2), (1024, 256), (1025, 256), (4096, 256), (9001, 270), (513, 2)])
def test_every_row_arrives(vocab, rows):
    cfg = Transformer250MConfig(hidden_dim=32, num_layers=1, num_heads=2, intermediate_dim=64, vocab_size=vocab, max_seq_len=rows,
                                norm_scope="token")
    model = TransformerModelPlugin().create_builder().build(cfg, seed=3)
    ids = np.random.default_rng(vocab).integers(0, vocab, rows, dtype=np.uint64)
    want = model.forward_all(ids)
    buf = np.full(rows * vocab + 40, 7.0, dtype=np.float32)  # (17 floats in: not at a page's or a line's start)
    _check(_lib.load().coeus_model_forward_all(model._h, ids.ctypes.data, rows, buf.ctypes.data + 17 * 4))
    assert np.array_equal(buf[17:17 + rows * vocab].reshape(rows, vocab), want)
    assert (buf[:17] == 7.0).all() and (buf[17 + rows * vocab:] == 7.0).all()
    per = (1 << 20) // (4 * vocab)  # rows of a slot
    for r in sorted({0, rows - 1, *[i for k in range(1, 11) for i in (per * k - 1, per * k, per * k + 1) if 0 <= i < rows]}):
        one = model.forward(ids[:r + 1])  # per-token norms: a row does not see what follows it
        assert np.abs(one - want[r]).max() <= 2e-5 * np.abs(want[r]).max(), r
    s = model.session(batch=1, max_ctx=rows)
    if rows > 2:
        s.prefill(ids[:-1].reshape(1, -1), want_logits=False)
        last = s.decode(ids[-1:])[0]
        assert np.abs(last - want[-1]).max() <= 2e-5 * np.abs(want[-1]).max()
