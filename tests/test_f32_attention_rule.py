"""f32 prompt attention on both sides of every line between its kernels (a query a workgroup, 32, or 128): float64, several sequences, keys
before the prompt, and scores that are infinite or no number."""
import numpy as np
import pytest

import f64_model
from coeus_amd import Transformer250MConfig, TransformerModelPlugin, _lib
from coeus_amd.device import DeviceArray, synchronize
from coeus_amd.plugin import _check
from gpu_util import dev

gpu = pytest.mark.gpu


# The launches that were slower with 32 queries (us, 128 / 32): heads of 128 in 256 workgroups of short walks, 28.4 / 42.7 at 256 heads of 128 rows, and with
# one tile of keys
@pytest.mark.parametrize("batch,rows,cached,heads,hd,queries", [
    (1, 16, 0, 32, 128, 128), (1, 32, 0, 1, 128, 128), (8, 32, 0, 32, 128, 128), (1, 33, 0, 32, 128, 32), (1, 17, 16, 32, 128, 32), (1, 17, 15, 32, 128, 128),
    (1, 128, 0, 256, 128, 128), (2, 128, 0, 128, 128, 128), (1, 256, 0, 128, 128, 128), (1, 512, 0, 64, 128, 128), (1, 128, 0, 128, 128, 32), (1, 512, 0, 32, 128, 32),
    (1, 768, 0, 32, 128, 32), (1, 1024, 0, 32, 128, 32), (1, 767, 0, 32, 128, 128), (1, 1025, 0, 32, 128, 128), (1, 16, 0, 12, 64, 32), (1, 4096, 0, 12, 64, 32),
    (8, 512, 0, 12, 64, 32), (8, 513, 0, 12, 64, 128), (1, 15, 0, 12, 64, 1), (8, 1, 900, 32, 128, 1), (1, 15, 0, 4, 96, 4), (1, 40, 0, 4, 96, 4)])
def test_plan(batch, rows, cached, heads, hd, queries):
    assert _lib.load().coeus_plan_attention_f32(batch, rows, cached, heads, hd) == queries


def _attention(qkv, heads, hd):
    out = DeviceArray((qkv.shape[0], heads * hd), np.float32)
    dq = dev(qkv)
    _check(_lib.load().coeus_op_attention(dq.ptr, qkv.shape[0], heads, hd, out.ptr, None))
    synchronize()
    return out.to_host()


def _float64(qkv, heads, hd, h):
    inner = heads * hd
    q, k, v = (qkv[:, i * inner + h * hd:i * inner + (h + 1) * hd].astype(np.float64) for i in range(3))
    s = np.where(np.tril(np.ones((len(qkv), len(qkv)), bool)), q @ k.T / np.sqrt(hd), -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    return (p / p.sum(-1, keepdims=True)) @ v


# workgroups of 128 queries: heads of 64 384 | 388, 386, 392; of 128 one tile of keys | two, 128 | 129, 128 | 130, 252 | 258 of 768 rows, 240 of 700
@gpu
@pytest.mark.parametrize("rows,heads,hd", [(400, 96, 64), (400, 97, 64), (129, 193, 64), (1000, 49, 64), (32, 5, 128), (33, 5, 128), (100, 128, 128),
                                           (128, 129, 128), (256, 64, 128), (130, 65, 128), (768, 42, 128), (768, 43, 128), (700, 40, 128)])
def test_both_sides(rows, heads, hd):
    qkv = np.random.default_rng(rows + heads).standard_normal((rows, 3 * heads * hd)).astype(np.float32)
    out = _attention(qkv, heads, hd)
    for h in range(0, heads, max(1, heads // 7)):
        want = _float64(qkv, heads, hd, h)
        # f32: sums of hd products and of up to 1000 probabilities, exp2 to 1 ulp of arguments below 16
        assert np.abs(out[:, h * hd:(h + 1) * hd] - want).max() <= 1e-5 * np.abs(want).max(), h


@gpu
@pytest.mark.parametrize("rows,heads,hd", [(150, 3, 64), (150, 3, 128), (150, 200, 64), (150, 70, 128)])
def test_scores_that_are_infinite_or_no_number(rows, heads, hd):
    """A key whose score is -inf weighs nothing, wherever it stands behind the first tile; +inf and NaN make the queries that see the key NaN, and
    no others."""
    rng = np.random.default_rng(rows)
    inner = heads * hd
    qkv = rng.standard_normal((rows, 3 * inner)).astype(np.float32)
    qkv[:, :inner:hd] = 1e20  # (dimension 0 of every head; keys hold nothing there but the ones below)
    qkv[:, inner:2 * inner:hd] = 0
    clean = qkv.copy()
    for j in (37, 64, 65, 70, 95, 130):
        qkv[j, inner:2 * inner:hd] = -1e30  # -1e50: -inf
    want = {h: _float64(qkv, heads, hd, h) for h in (0, heads - 1)}
    out = _attention(qkv, heads, hd)
    for h, w in want.items():
        assert np.abs(out[:, h * hd:(h + 1) * hd] - w).max() <= 1e-5 * np.abs(w).max()
    for bad in (1e30, np.nan):
        qkv = clean.copy()
        qkv[75, inner:2 * inner:hd] = bad
        out = _attention(qkv, heads, hd)
        assert np.isnan(out[75:]).all() and np.isfinite(out[:75]).all()
        w = _float64(clean[:75], heads, hd, heads - 1)
        assert np.abs(out[:75, (heads - 1) * hd:] - w).max() <= 1e-5 * np.abs(w).max()


# 16 sequences; workgroups of 128 queries 384 | 512, 128 | 256, the second piece behind the first one's keys
@gpu
@pytest.mark.parametrize("heads,hd,n,first", [(8, 64, 300, 0), (8, 64, 390, 0), (8, 64, 330, 150), (4, 128, 200, 0), (4, 128, 290, 0), (4, 128, 170, 141),
                                              (2, 128, 60, 33), (2, 128, 49, 33)])
def test_sequences_and_earlier_keys(orc, heads, hd, n, first):
    kw = dict(hidden_dim=heads * hd, num_layers=1, num_heads=heads, intermediate_dim=64, vocab_size=130, max_seq_len=n, norm_scope="token", max_batch=16)
    oc = orc.config_from_kwargs(kw)
    params = orc.init_seeded(oc, n)
    model = TransformerModelPlugin().create_builder().build(Transformer250MConfig(**kw), parameters=params)
    ids = np.random.default_rng(n).integers(0, 130, (16, n), dtype=np.uint64)
    s = model.session(batch=16, max_ctx=n)
    if first:
        s.prefill(ids[:, :first], want_logits=False)
    rows = sorted({0, 1, 15, 16, 31, 32, 33, (n - first) // 2, n - first - 1} & set(range(n - first)))
    got = np.asarray(s.feed(ids[:, first:], want=rows)).reshape(16, len(rows), 130)
    for b in range(0, 16, 3):
        want = f64_model.forward_all(oc, params, ids[b])[[first + r for r in rows]]
        # (as in the other tests of f32 prompts: sums of up to 4 hd terms, a few roundings of 2^-24 each)
        assert np.abs(got[b] - want).max() <= 2e-5 * np.abs(want).max(), b


# 1 - 15 rows, a workgroup per row and head: the lanes behind a row's last key read that key again
@gpu
@pytest.mark.parametrize("rows", [1, 2, 5, 15])
@pytest.mark.parametrize("heads,hd", [(3, 64), (2, 128)])
def test_few_rows_of_infinite_values_and_scores(rows, heads, hd):
    """An infinite value is an infinity (or, with its opposite, no number) in that dimension of the rows that see it, and nothing elsewhere; scores
    of -inf weigh nothing, +inf and NaN make the rows that see them NaN."""
    rng = np.random.default_rng(rows + hd)
    inner = heads * hd
    clean = rng.standard_normal((rows, 3 * inner)).astype(np.float32)
    clean[:, :inner:hd] = 1e20
    clean[:, inner:2 * inner:hd] = 0
    cases = []
    for j in range(rows):
        values = clean.copy()
        values[j, 2 * inner::hd] = np.inf
        values[j, 2 * inner + hd - 1::hd] = -np.inf
        if j + 1 < rows:
            values[j + 1, 2 * inner + 3::hd] = -np.inf
            values[j, 2 * inner + 3::hd] = np.inf
        cases.append(values)
        for score in (-1e30, 1e30, np.nan):
            scores = clean.copy()
            scores[j, inner:2 * inner:hd] = score
            cases.append(scores)
    for i, qkv in enumerate(cases):
        out = _attention(qkv, heads, hd)
        for h in range(heads):
            # (as f32 has them: 1e50 is infinite, and what a key weighs that nobody may see is no factor)
            want, got = np.full((rows, hd), np.nan), out[:, h * hd:(h + 1) * hd]
            for r in range(rows):
                with np.errstate(over="ignore", invalid="ignore"):
                    q, k, v = (qkv[:r + 1, at * inner + h * hd:at * inner + (h + 1) * hd].astype(np.float64) for at in range(3))
                    s = (q[r] * k).sum(-1) / np.sqrt(hd)
                    s = np.where(np.abs(s) > 3.5e38, np.copysign(np.inf, s), s)
                    p = np.exp(s - s.max())
                    want[r] = (p[:, None] * v).sum(0) / p.sum()
            odd = ~np.isfinite(want)
            assert np.array_equal(got[odd], want[odd].astype(np.float32), equal_nan=True), (i, h)
            # sums of hd products and of up to 15 probabilities, exp2 to 1 ulp of arguments below 16
            assert odd.all() or np.abs(got - want)[~odd].max() <= 1e-5 * np.abs(want[~odd]).max(), (i, h)
