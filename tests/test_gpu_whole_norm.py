"""Norms over a whole slice at the edges of the one-workgroup kernel's sizes, and short prompts on both sides of where two launches take over, against float64."""
import ctypes as C

import numpy as np
import pytest

from coeus_amd import Transformer250MConfig, _lib
from coeus_amd.device import DeviceArray, synchronize
from coeus_amd.plugin import _check
from gpu_util import dev, rel_err
from test_gpu_model import build, orc_cfg

pytestmark = pytest.mark.gpu
EPS = np.float64(np.float32(1e-5))


def norm(kind, x, scale, bias):
    rows, hidden = x.shape
    dx, ds, db, y = dev(x), dev(scale), dev(bias), DeviceArray(x.shape, np.float32)
    _check(_lib.load().coeus_op_norm(kind, 0, dx.ptr, rows, hidden, ds.ptr, None if kind else db.ptr, C.c_float(1e-5), y.ptr, None))
    synchronize()
    return y.to_host()


# one piece; a wave's, a workgroup's and one more; each number of pieces a thread; the largest slice that the operator gives one workgroup; two launches; rows without pieces
@pytest.mark.parametrize("rows,hidden", [(1, 4), (3, 84), (1, 256), (16, 256), (1025, 4), (2, 4096), (683, 12), (4, 4096), (4097, 4), (42, 768), (8191, 4), (8, 4096), (43, 768), (42, 767)])
@pytest.mark.parametrize("far", [False, True])
def test_whole_slice(rows, hidden, far):
    rng = np.random.default_rng(rows * hidden)
    x = (1000.0 + 0.5 * rng.standard_normal((rows, hidden)) if far else 2 * rng.standard_normal((rows, hidden)) + 0.5).astype(np.float32)
    scale, bias, x64 = rng.standard_normal(hidden).astype(np.float32), rng.standard_normal(hidden).astype(np.float32), x.astype(np.float64)
    mean = np.float64(np.float32(x64.mean()))  # (rounded to f32 before it is subtracted)
    # five roundings of 2^-24 each of the scaled value, one more of the sum with the bias
    t = scale * (x64 - mean) / np.sqrt(x64.var() + EPS)
    assert np.all(np.abs(norm(0, x, scale, bias) - (t + bias)) <= 2.0 ** -24 * (6 * np.abs(t) + np.abs(t + bias)) + 1e-30)
    t = scale * x64 / np.sqrt((x64 ** 2).mean() + EPS)
    assert np.all(np.abs(norm(1, x, scale, bias) - t) <= 2.0 ** -24 * 6 * np.abs(t) + 1e-30)


def test_values_that_are_not_finite():
    x, one = np.random.default_rng(2).standard_normal((20, 768)).astype(np.float32), np.ones(768, np.float32)
    for bad in (np.inf, np.nan):
        for at in ((0, 0), (19, 767)):
            y = x.copy()
            y[at] = bad
            assert np.isnan(norm(0, y, one, one)).all()
            got = norm(1, y, one, one)  # (an infinite mean square: zeros, and infinity over infinity)
            assert np.isnan(got).all() if np.isnan(bad) else np.isnan(got[at]) and np.count_nonzero(got) == 1


@pytest.mark.parametrize("n", [3, 17, 21, 22, 24, 32, 42, 43])
def test_as_a_model_runs_it(orc, n):
    """The last norm of a pass, with one workgroup or (from 22 rows of 768) two launches: blocks that add nothing in front of it, logits that are its results."""
    H = 768
    cfg = Transformer250MConfig(hidden_dim=H, num_layers=1, num_heads=12, intermediate_dim=96, vocab_size=H, max_seq_len=64)
    oc = orc_cfg(orc, cfg)
    params, at = orc.init_seeded(oc, 5), orc.layout(oc)
    rng, layer = np.random.default_rng(n), at.first_layer_offset
    put = lambda o, x: params.__setitem__(slice(o, o + x.size), x.ravel())  # noqa: E731
    for o, size in ((at.wo, H * H), (at.bo, H), (at.w_down, 96 * H), (at.b_down, H)):
        put(layer + o, np.zeros(size, np.float32))
    table, scale, bias = (rng.standard_normal(x).astype(np.float32) for x in ((H, H), H, H))
    put(at.token_embed_offset, table + np.float32(0.5))
    put(at.final_ln_offset, scale)
    put(at.final_ln_offset + H, bias)
    put(at.output_proj_offset, np.eye(H, dtype=np.float32))
    ids = orc.synth_ids(n, H, n)
    x = ((table + np.float32(0.5))[np.asarray(ids, np.int64)] + orc.positional_encoding(64, H)[:n]).astype(np.float64)
    t = scale * (x - np.float64(np.float32(x.mean()))) / np.sqrt(x.var() + EPS)
    # the roundings of test_whole_slice, and one of a sine or cosine of the positions
    bound = 2.0 ** -24 * (6 * np.abs(t) + np.abs(t + bias)) + 2.0 ** -23 * np.abs(scale) / x.std()
    assert np.all(np.abs(build(cfg, params).forward_all(ids) - (t + bias)) <= bound)


@pytest.mark.parametrize("n", [17, 21, 22, 42, 43])
def test_short_prompts(orc, n):
    cfg = Transformer250MConfig(hidden_dim=768, num_layers=1, num_heads=12, intermediate_dim=96, vocab_size=50, max_seq_len=64)
    oc = orc_cfg(orc, cfg)
    params = orc.init_seeded(oc, 5)
    ids = orc.synth_ids(n, 50, n)
    rc, _, want = orc.forward(oc, params, ids, all_rows=True)
    assert rc == 0 and rel_err(build(cfg, params).forward_all(ids), want) < 1e-3  # (the oracle's own statistics are sums in f32)
