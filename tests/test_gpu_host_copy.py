"""Logits on their way to the caller: sizes around the pieces (16 KiB) and halves (4 MiB, two of them) of the pinned memory that they go through, and
results that start in the middle of a page, against the same rows fetched one at a time."""
import ctypes as C
import resource
import time

import numpy as np
import pytest

from coeus_amd import Transformer250MConfig, TransformerModelPlugin, _lib
from coeus_amd.device import DeviceArray
from coeus_amd.plugin import _check

pytestmark = pytest.mark.gpu


# 4 * vocab bytes a row: 4096 in all (the runtime's copy) and one row more; 1 MiB and one value a row more; one half; three rounds through the halves, three threads
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
    # rows on both sides of every MiB: of pieces' and halves' ends
    per = (1 << 20) // (4 * vocab)
    for r in sorted({0, rows - 1, *[i for k in range(1, 11) for i in (per * k - 1, per * k, per * k + 1) if 0 <= i < rows]}):
        one = model.forward(ids[:r + 1])  # per-token norms: a row does not see what follows it
        assert np.abs(one - want[r]).max() <= 2e-5 * np.abs(want[r]).max(), r
    s = model.session(batch=1, max_ctx=rows)
    if rows > 2:
        s.prefill(ids[:-1].reshape(1, -1), want_logits=False)
        last = s.decode(ids[-1:])[0]
        assert np.abs(last - want[-1]).max() <= 2e-5 * np.abs(want[-1]).max()


def test_into_pinned_and_device_memory():
    """Results that the caller wants in pinned memory (seven halves' worth, and a few pieces), or on the device."""
    vocab, rows = 50257, 128
    cfg = Transformer250MConfig(hidden_dim=32, num_layers=1, num_heads=2, intermediate_dim=64, vocab_size=vocab, max_seq_len=rows,
                                norm_scope="token")
    model = TransformerModelPlugin().create_builder().build(cfg, seed=3)
    lib, hip = _lib.load(), C.CDLL("libamdhip64.so", mode=C.RTLD_GLOBAL)
    hip.hipHostMalloc.argtypes, hip.hipHostFree.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint], [C.c_void_p]
    ids = np.random.default_rng(4).integers(0, vocab, rows, dtype=np.uint64)
    for n, call, size in ((rows, lib.coeus_model_forward_all, rows * vocab), (rows, lib.coeus_model_forward, vocab)):
        want = np.empty(size, np.float32)
        _check(call(model._h, ids.ctypes.data, n, want.ctypes.data))
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), 4 * size + 4096, 0) == 0
        buf = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_float)), (size + 1024,))
        buf[:] = 7.0
        _check(call(model._h, ids.ctypes.data, n, p.value + 4 * 17))
        assert np.array_equal(buf[17:17 + size], want) and (buf[:17] == 7.0).all() and (buf[17 + size:] == 7.0).all()
        del buf
        assert hip.hipHostFree(p) == 0
        d = DeviceArray((size,), np.float32)
        _check(call(model._h, ids.ctypes.data, n, d.ptr))
        assert np.array_equal(d.to_host(), want)


# a 16 KiB piece and one value less or more; a half of 4 MiB and one more; two halves; 8 MiB (three threads) and one row more, and
# an odd number of values in five rounds
@pytest.mark.parametrize("vocab,rows", [(1365, 3), (4096, 1), (4097, 1), (1024, 1024), (1025, 1024), (2048, 1024), (2049, 1024), (4999, 877)])
def test_pieces_halves_and_threads(vocab, rows):
    cfg = Transformer250MConfig(hidden_dim=32, num_layers=1, num_heads=2, intermediate_dim=64, vocab_size=vocab, max_seq_len=rows,
                                norm_scope="token")
    model = TransformerModelPlugin().create_builder().build(cfg, seed=3)
    lib = _lib.load()
    for seed in (1, 2, 3):  # (the flags of one call are not the next one's)
        ids = np.random.default_rng(seed).integers(0, vocab, rows, dtype=np.uint64)
        d = DeviceArray((rows * vocab,), np.float32)
        _check(lib.coeus_model_forward_all(model._h, ids.ctypes.data, rows, d.ptr))
        assert np.array_equal(model.forward_all(ids).ravel(), d.to_host())


def test_long_pass_keeps_no_core_busy():
    """Results large enough for three threads behind a pass of some 100 ms: the two others sleep.  The calling thread may spin for all
    of it in the runtime (1.0 of the pass), the others for 5 ms each and their share of the copy; without sleep 3.0 in all."""
    cfg = Transformer250MConfig(hidden_dim=2048, num_layers=48, num_heads=16, intermediate_dim=8192, vocab_size=1100, max_seq_len=2048,
                                norm_scope="token")
    model = TransformerModelPlugin().create_builder().build(cfg, seed=3)
    ids = np.random.default_rng(5).integers(0, 1100, 2048, dtype=np.uint64)
    d = DeviceArray((2048 * 1100,), np.float32)
    _check(_lib.load().coeus_model_forward_all(model._h, ids.ctypes.data, 2048, d.ptr))
    out = d.to_host().reshape(2048, 1100)
    assert out.nbytes > 8 << 20  # (three rounds through two halves)
    used, took = [], []
    for _ in range(3):
        r, t = resource.getrusage(resource.RUSAGE_SELF), time.perf_counter()
        assert np.array_equal(model.forward_all(ids), out)
        took.append(time.perf_counter() - t)
        e = resource.getrusage(resource.RUSAGE_SELF)
        used.append(e.ru_utime + e.ru_stime - r.ru_utime - r.ru_stime)
    assert min(took) > 0.06, took  # (else the pass is too short to tell)
    assert min(u / t for u, t in zip(used, took)) < 1.8, (used, took)
