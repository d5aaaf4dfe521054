"""Matrix memory, prompts of one chunk: a launch that reads the state, answers and stores the state behind the prompt.  At the
edges of the 16-token tiles and of the sizes, from a state that earlier tokens left, with a value that is not finite (which the rows
in front of it must not see) or a key that is infinite, and for rows that
16-byte pieces do not lie in, in one chunk and in several."""
import ctypes as C

import numpy as np
import pytest

from coeus_amd import _lib
from coeus_amd.device import DeviceArray
from coeus_amd.plugin import _check
from gpu_util import dev
from test_gpu_zekilix import Memory, off

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4, 24, 64), (2, 128, 128), (1, 256, 256), (2, 36, 132), (3, 4, 4), (2, 128, 40)])
@pytest.mark.parametrize("n", [2, 15, 16, 17, 32, 33, 48, 49, 63, 64])
def test_behind_earlier_tokens(shape, n):
    t = Memory(*shape, batch=2, seed=n)
    p = t.inputs(3 + n + 1)
    want, S = t.want(p)
    got = np.concatenate([t.prompt(p[:, :3], 0), t.prompt(p[:, 3:3 + n], 1), t.step(p[:, 3 + n])[:, None]], axis=1)
    # (the bounds of the other tests of prompts and states: chains of f32 sums of some 64 terms)
    assert off(got, want) < 2e-5 and t.state_off(S) < 2e-5


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("n,j", [(5, 3), (30, 0), (40, 39), (64, 20)])
def test_rows_in_front_of_a_value_that_is_not_finite(bad, n, j):
    H, d, e = 2, 32, 48
    a, b = (Memory(H, d, e, batch=1, seed=n) for _ in range(2))
    p = a.inputs(n)
    clean = b.prompt(p, 1)
    p[0, j, 2 * H * d + 5] = bad
    got = a.prompt(p, 1)
    assert np.array_equal(got[:, :j], clean[:, :j])  # the same sums of the same values
    assert not np.isfinite(got[0, j:, 5]).any() and np.isfinite(got[0, :, e:]).all()  # (the other head)
    assert not np.isfinite(a.state[0].to_host()[0, 0, :, 5]).any() and np.isfinite(a.state[0].to_host()[0, :, :, 6]).all()


@pytest.mark.parametrize("n,j", [(2, 1), (5, 4), (16, 15), (17, 16), (30, 29), (30, 7), (63, 62)])
def test_infinite_key_as_token_by_token(n, j):
    H, d, e = 2, 32, 48
    a, b = (Memory(H, d, e, batch=1, seed=n) for _ in range(2))
    p = a.inputs(n)
    p[0, j, H * d + 3] = np.inf
    got, want = a.prompt(p, 1), b.prompt(p, 0)
    assert np.array_equal(np.isfinite(got), np.isfinite(want)) and np.isfinite(got[0, :j]).all()
    for x, y in zip(a.state, b.state):
        x, y = x.to_host(), y.to_host()
        assert np.array_equal(x[~np.isfinite(y)], y[~np.isfinite(y)]) and np.isfinite(x).sum() == np.isfinite(y).sum()
    assert (np.abs(a.state[0].to_host()[0, 0, 3]) == np.inf).all() and a.state[1].to_host()[0, 0, 3] == np.inf


def test_rows_off_a_16_byte_boundary():
    t = Memory(2, 32, 48, batch=1, seed=1)
    p = t.inputs(20)
    x, out = dev(np.concatenate([np.zeros(1, np.float32), p.ravel()])), DeviceArray((1, 20, 96))
    _check(_lib.load().coeus_op_memory_prompt(C.byref(t.s), C.byref(t.w), x.ptr + 4, *[a.ptr for a in t.state], 1, 20, 1, out.ptr, None))
    want, S = t.want(p)
    assert off(out.to_host(), want) < 2e-5 and t.state_off(S) < 2e-5


@pytest.mark.parametrize("shape", [(2, 32, 48), (1, 20, 8), (2, 9, 5)])
@pytest.mark.parametrize("n", [2, 48, 64, 65, 130])
def test_rows_off_a_boundary_in_chunks(shape, n):
    """The same bits as rows on a boundary, nothing behind the last row's gates read (the buffer ends there)."""
    H, d, e = shape
    a, b = (Memory(*shape, batch=2, seed=n) for _ in range(2))
    p = a.inputs(n)
    want = a.prompt(p, 1)
    x, out = dev(np.r_[np.zeros(1, np.float32), p.ravel()[:p.size - (a.ld - a.nb - 2 * H)]]), DeviceArray((2, n, H * e))
    _check(_lib.load().coeus_op_memory_prompt(C.byref(b.s), C.byref(b.w), x.ptr + 4, *[s.ptr for s in b.state], 2, n, 1, out.ptr, None))
    assert np.array_equal(out.to_host(), want)
    assert all(np.array_equal(s.to_host(), t.to_host()) for s, t in zip(a.state, b.state))
