"""The routing a device forward writes to the caller's ids and w (moe_forward_async, its no-alloc form and
moe_forward_hc_async): the oracle's, and nothing outside them, on each side of the decode kernel's last token count, both
prefill routers, and buffers off their word alignment (which are copied to)."""
import numpy as np
import pytest

from tests import harness as h
from tests.harness import moe
from tests.test_gpu_parity import say

pytestmark = pytest.mark.gpu

PAD = 64  # bytes watched on each side


def run(call, T, K, off):
    """ids and w of a forward into buffers `off` bytes past their alignment; the bytes around them must stay."""
    d = h.Dev()
    n = T * K * 4
    guard = np.full(n + 2 * PAD + 4, 0xA5, np.uint8)
    bufs = [d.put(guard) for _ in range(2)]
    call(bufs[0].value + PAD + off, bufs[1].value + PAD + off)
    out = []
    for b, t in zip(bufs, (np.int32, np.float32)):
        raw = d.get(b, (guard.size,), np.uint8)
        assert (raw[:PAD + off] == 0xA5).all() and (raw[PAD + off + n:] == 0xA5).all()
        out.append(np.frombuffer(raw[PAD + off:PAD + off + n].tobytes(), t).reshape(T, K))
    d.free()
    return out


@pytest.mark.parametrize("off", [0, 4, 2])
@pytest.mark.parametrize("T,exact", [(1, False), (16, False), (17, False), (17, True), (130, False)])
def test_routing_out(T, exact, off):
    say("routing out", (T, exact, off))
    H = 512
    L = h.Layer(H, 256, 32, 4, moe.QT_Q4_K, moe.QT_Q8_0, seed=77, zipf=1.1)
    blk = L.block(max_tokens=max(T, 16), exact_router=exact)
    L.upload(blk)
    x = h.tokens(78, T, H)
    _, io, wo = L.oracle_forward(x)
    d = h.Dev()
    xd, yd = d.put(x), d.alloc(x.nbytes)

    def sync(f):
        f()
        blk.check()

    calls = [blk.forward_async] + ([blk.forward_async_noalloc] if T <= 16 else [])
    for f in calls:
        ids, w = run(lambda i, v: sync(lambda: f(0, xd, T, yd, i, v)), T, 4, off)
        assert np.array_equal(ids, io)
        # The default prefill router's weights are within the block's bound; the others are the oracle's bits.
        assert np.array_equal(w, wo) if blk.bit_exact(T) else h.max_abs(w, wo) <= h.W_TOL
    d.free()
    blk.close()
