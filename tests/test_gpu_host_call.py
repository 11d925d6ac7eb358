"""The host call on each side of its largest pinned size (16 tokens): strided rows in and out, in place, with and without the
routing, against the oracle's, and nothing written between the rows."""
import ctypes as C

import numpy as np
import pytest

from c0ven_amd import _lib
from tests import harness as h
from tests.harness import moe
from tests.test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 5, 16, 17])
def test_host_call_rows(T):
    say("host call", T)
    H, K = 512, 4
    L = h.Layer(H, 256, 32, K, moe.QT_Q4_K, moe.QT_Q8_0, seed=81, zipf=1.1)
    blk = L.block(max_tokens=20, exact_router=True)
    L.upload(blk)
    x = h.tokens(82, T, H)
    yo, io, wo = L.oracle_forward(x)
    for xs, ys, inplace, route in ((H, H, False, True), (H + 3, H + 5, False, False), (H + 4, H + 4, True, True)):
        xb = np.full((T, xs), np.float32(7.0))
        xb[:, :H] = x
        yb = xb if inplace else np.full((T, ys), np.float32(7.0))
        ids, w = np.full((T, K), -1, np.int32), np.zeros((T, K), np.float32)
        ro = _lib.MoeRouteOut(ids.ctypes.data_as(C.POINTER(C.c_int32)), w.ctypes.data_as(C.POINTER(C.c_float)))
        assert _lib.lib.moe_forward(blk.h, 0, h.ptr(xb), T, xs, h.ptr(yb), ys, C.byref(ro) if route else None) == 0
        assert np.array_equal(yb[:, :H], yo), h.max_abs(yb[:, :H], yo)
        assert (yb[:, H:] == 7.0).all()
        assert not route or (np.array_equal(ids, io) and np.array_equal(w, wo))
    blk.close()


@pytest.mark.parametrize("T", [3, 18])
def test_host_call_after_device_calls(T):
    """The routing of a host call is its own forward's, whatever buffers the forwards before it wrote theirs to."""
    say("host call after device calls", T)
    H, K = 512, 4
    L = h.Layer(H, 256, 32, K, moe.QT_Q4_K, moe.QT_Q8_0, seed=83, zipf=1.1)
    blk = L.block(max_tokens=20, exact_router=True)
    L.upload(blk)
    d = h.Dev()
    ids, w, y = d.alloc(20 * K * 4), d.alloc(20 * K * 4), d.alloc(20 * H * 4)
    for i, (a, b) in enumerate(((ids, w), (None, w), (ids, None))):
        for n in (2, 19):
            blk.forward_async(0, d.put(h.tokens(90 + i, n, H)), n, y, a, b)
        x = h.tokens(84 + i, T, H)
        yo, io, wo = L.oracle_forward(x)
        y2, i2, w2 = blk.forward(0, x)
        assert np.array_equal(y2, yo) and np.array_equal(i2, io) and np.array_equal(w2, wo)
    d.free()
    blk.close()
