"""The certified top-k's open places: router rows that repeat (exact ties) or differ in one value's last bit, more candidates
than a wave holds, rows of one load batch and of many, and tokens so small that fp32 cannot hold their products (the k-order
chain decides), experts masked by their bias; the ids are the oracle's."""
import numpy as np
import pytest

from tests import harness as h
from tests.harness import moe
from tests.test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,E,K", [(512, 32, 4), (1536, 512, 16), (8192, 96, 1)])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -115])
def test_open_places(H, E, K, scale):
    say("open places", (H, E, K), scale)
    L = h.Layer(H, 256, E, K, moe.QT_Q8_0, moe.QT_Q8_0, has_shared=False, seed=31 + H, experts=[0])
    r = np.random.default_rng(H)
    for e in range(1, E):  # groups of up to 80 rows: repeats, or one value's last bit apart
        if e % 80:
            L.router[e] = L.router[e - 1]
            if e % 3 == 0:
                L.router[e, r.integers(H)] ^= 1
    blk = L.block(max_tokens=40)
    L.upload(blk)
    x = h.tokens(32, 40, H) * np.float32(scale)
    _, io, _ = L.oracle_route(x)  # (the experts play no part)
    _, ids, _ = blk.forward(0, x)
    blk.close()
    assert np.array_equal(ids, io)


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("E,K", [(32, 4), (512, 10)])
def test_masked_experts(E, K, exact):
    """Biases of minus infinity, of the type's lowest value and of plus infinity on some experts, and logits that are infinite."""
    say("masked experts", (E, K), exact)
    L = h.Layer(512, 256, E, K, moe.QT_Q8_0, moe.QT_Q8_0, has_shared=False, seed=91, zipf=1.1, experts=[0])
    L.bias[1::3], L.bias[2::7], L.bias[5] = -np.inf, np.finfo(np.float32).min, np.inf
    x = h.tokens(92, 40, 512)
    x[3] *= np.float32(2.0 ** 120)
    _, io, _ = L.oracle_route(x)
    blk = L.block(max_tokens=40, exact_router=exact)
    L.upload(blk)
    _, ids, _ = blk.forward(0, x)
    blk.close()
    assert np.array_equal(ids, io)
