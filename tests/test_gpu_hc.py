"""moe_forward_hc: the block with its hyper-connection mix and combine fused into the decode launch (MODEL_LAYER.md
1.1-1.2; model.cpp:1350-1416 runs them as separate kernels) against the oracle's mix, block and combine, bit for bit:
the updated streams R, y, the routing."""
import sys
import time

import numpy as np
import pytest

from tests import harness as h
from tests.harness import moe

pytestmark = pytest.mark.gpu


def say(*a):
    print("[hc]", *a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("shape", [(512, 256, 32, 4, 64), (2560, 640, 64, 8, 320)])
@pytest.mark.parametrize("types", [(moe.QT_Q4_K, moe.QT_Q8_0, moe.QT_Q8_0, moe.QT_Q8_0),
                                   (moe.QT_IQ3_XXS, moe.QT_IQ4_NL, moe.QT_Q4_K, moe.QT_IQ4_NL)])
def test_forward_hc(shape, types):
    H, F, E, K, lr = shape
    gt, dt, sgt, sdt = types
    if H % 256 or (dt == moe.QT_Q4_K and F % 256):
        pytest.skip("shape not of these types")
    say("forward_hc", shape, [moe.TYPE_NAMES[t] for t in types])
    L = h.Layer(H, F, E, K, gt, dt, sgt, sdt, seed=H + lr, zipf=1.1)
    hc = h.HcModule(H, lr, seed=11)
    blk = moe.MoeBlock(H, F, E, K, gt, dt, True, sgt, sdt, n_layer=2, max_tokens=16, hc_lr=lr)
    L.upload(blk, 1)
    hc.load(blk, 1)
    r = np.random.default_rng(H)
    for T in (1, 8, 16):
        R = r.standard_normal((T, 4, H)).astype(np.float32)
        R2, y, ids, w = blk.forward_hc(1, R)
        x, inj = hc.pre(R)
        yo, io, wo = L.oracle_forward(x)
        Ro = h.HcModule.post(R, inj, yo)
        assert np.array_equal(ids, io) and np.array_equal(w, wo), T
        assert np.array_equal(y, yo), (T, h.max_abs(y, yo))
        assert np.array_equal(R2, Ro), (T, h.max_abs(R2, Ro))
        # The plain forward on the oracle's x gives the same y (the mix is the only difference).
        y2, _, _ = blk.forward(1, x)
        assert np.array_equal(y2, yo)
    blk.close()


def test_forward_hc_requires_module():
    blk = moe.MoeBlock(512, 256, 8, 2, moe.QT_Q8_0, moe.QT_Q8_0, hc_lr=64)
    L = h.Layer(512, 256, 8, 2, moe.QT_Q8_0, moe.QT_Q8_0, seed=4)
    L.upload(blk)
    with pytest.raises(moe.MoeError):  # no moe_load_hc yet
        blk.forward_hc(0, np.zeros((1, 4, 512), np.float32))
    blk.close()
    with pytest.raises(moe.MoeError):  # hc_lr not a multiple of 8
        moe.MoeBlock(512, 256, 8, 2, moe.QT_Q8_0, moe.QT_Q8_0, hc_lr=100)


@pytest.mark.parametrize("shape", [(512, 256, 32, 4, 64), (2560, 640, 64, 8, 320)])
@pytest.mark.parametrize("fixed_order", [False, True])
def test_forward_hc_prefill(shape, fixed_order):
    """More tokens than the decode kernel takes: the mix's kernels (exact digit products within a bound, the open sums in
    the fixed order; with hc_fixed_order every down sum in the fixed order), the prefill block, the combine's kernel;
    R, y and the routing against the oracle's, bit for bit (the exact router: the oracle's weights and y)."""
    H, F, E, K, lr = shape
    say("forward_hc prefill", shape, "fixed order" if fixed_order else "bound")
    L = h.Layer(H, F, E, K, moe.QT_Q4_K, moe.QT_Q8_0, moe.QT_Q8_0, moe.QT_Q8_0, seed=H + lr + 1, zipf=1.1)
    hc = h.HcModule(H, lr, seed=12)
    blk = moe.MoeBlock(H, F, E, K, moe.QT_Q4_K, moe.QT_Q8_0, True, moe.QT_Q8_0, moe.QT_Q8_0, n_layer=1,
                       max_tokens=320, hc_lr=lr, exact_router=True, hc_fixed_order=fixed_order)
    L.upload(blk, 0)
    hc.load(blk, 0)
    r = np.random.default_rng(H + 7)
    for T in ((17, 100) if fixed_order else (17, 100, 320)):
        R = r.standard_normal((T, 4, H)).astype(np.float32)
        R2, y, ids, w = blk.forward_hc(0, R)
        x, inj = hc.pre(R)
        yo, io, wo = L.oracle_forward(x)
        Ro = h.HcModule.post(R, inj, yo)
        assert np.array_equal(ids, io) and np.array_equal(w, wo), T
        assert np.array_equal(y, yo), (T, h.max_abs(y, yo))
        assert np.array_equal(R2, Ro), (T, h.max_abs(R2, Ro))
    blk.close()


@pytest.mark.parametrize("lr,T", [(8, 17), (72, 63), (328, 65), (512, 49)])
def test_forward_hc_prefill_wide_values(lr, T):
    """The mix's digit products at their edges: ranks and tokens that end inside a 64-value chunk, a 16-row tile and a 64-row
    tile; rows and tokens whose values span 2^50 (they lose bits of their grid), whose largest value is a power of two or a
    subnormal, all-zero rows and tokens; R, y and the routing against the oracle's, bit for bit."""
    H, F, E, K = 512, 256, 32, 4
    say("forward_hc prefill wide values, rank", lr, "T", T)
    L = h.Layer(H, F, E, K, moe.QT_Q4_K, moe.QT_Q8_0, moe.QT_Q8_0, moe.QT_Q8_0, seed=lr, zipf=1.1)
    hc = h.HcModule(H, lr, seed=13)
    r = np.random.default_rng(lr + T)

    def widen(w):
        f = (w.astype(np.uint32) << 16).view(np.float32).copy()
        f[::3] *= np.exp2(-r.integers(0, 50, f[::3].shape)).astype(np.float32)  # spans 2^50
        f[1::7] = 0.0
        f[2::7] = np.where(r.random(f[2::7].shape) < 0.5, np.float32(-0.25), np.float32(2.0 ** -24))
        f[4::11, 0] = 2.0 ** -130
        f[5::11] *= np.float32(2.0 ** -120)
        return h.to_bf16(f.reshape(-1)).reshape(w.shape)

    hc.down, hc.inj, hc.up = widen(hc.down), widen(hc.inj), widen(hc.up)
    blk = moe.MoeBlock(H, F, E, K, moe.QT_Q4_K, moe.QT_Q8_0, True, moe.QT_Q8_0, moe.QT_Q8_0, n_layer=1, max_tokens=T,
                       hc_lr=lr, exact_router=True)
    L.upload(blk, 0)
    hc.load(blk, 0)
    R = r.standard_normal((T, 4, H)).astype(np.float32)
    R[::4] *= np.exp2(-r.integers(0, 50, R[::4].shape)).astype(np.float32)
    R[3] = 0.0
    R[5] = np.where(r.random((4, H)) < 0.5, np.float32(1.0), np.float32(-1.0))
    R[6, :, 1:] = 0.0
    R2, y, ids, w = blk.forward_hc(0, R)
    x, inj = hc.pre(R)
    yo, io, wo = L.oracle_forward(x)
    Ro = h.HcModule.post(R, inj, yo)
    blk.close()
    assert np.array_equal(ids, io) and np.array_equal(w, wo)
    assert np.array_equal(y, yo), h.max_abs(y, yo)
    assert np.array_equal(R2, Ro), h.max_abs(R2, Ro)


def test_forward_hc_prefill_not_finite():
    """Tokens with infinities and NaN among finite ones, and a row of W_down with an infinity: as the oracle's, NaN where it has
    one (the payload aside)."""
    H, F, E, K, lr, T = 512, 256, 32, 4, 64, 40
    say("forward_hc prefill, not finite")
    L = h.Layer(H, F, E, K, moe.QT_Q4_K, moe.QT_Q8_0, moe.QT_Q8_0, moe.QT_Q8_0, seed=3, zipf=1.1)
    hc = h.HcModule(H, lr, seed=14)
    hc.down[7, 5] = 0x7F80
    blk = moe.MoeBlock(H, F, E, K, moe.QT_Q4_K, moe.QT_Q8_0, True, moe.QT_Q8_0, moe.QT_Q8_0, n_layer=1, max_tokens=T,
                       hc_lr=lr, exact_router=True)
    L.upload(blk, 0)
    hc.load(blk, 0)
    r = np.random.default_rng(15)
    R = r.standard_normal((T, 4, H)).astype(np.float32)
    R[2, 1, 9], R[17, 0, 3], R[33, 3, 100] = np.inf, -np.inf, np.nan
    R[20, :, 5] = 0.0  # (0 times the infinite weight)
    x, inj = hc.pre(R)
    fine = np.isfinite(x).all(1)
    assert fine.sum() > 8 and not fine.all()
    R2, y, _, _ = blk.forward_hc(0, R)
    yo, _, _ = L.oracle_forward(np.where(fine[:, None], x, np.float32(0)))
    Ro = h.HcModule.post(R, inj, np.where(fine[:, None], yo, y))
    blk.close()
    assert np.array_equal(y[fine], yo[fine])
    assert np.array_equal(R2[fine], Ro[fine], equal_nan=True)


def test_forward_hc_prefill_outliers_cost():
    """A step whose tokens have a few channels thousands of times the others (values that lose bits of the digits' grid) leaves
    no more sums to the fixed-order kernels than another: it took 3.5 times as long while it did, and takes at most twice
    (the products then run on the fp64 matrix cores)."""
    H, F, E, K, lr, T = 2560, 640, 16, 2, 320, 1000
    say("forward_hc prefill outliers cost")
    L = h.Layer(H, F, E, K, moe.QT_Q4_K, moe.QT_Q8_0, moe.QT_Q8_0, moe.QT_Q8_0, seed=5, experts=[0])
    hc = h.HcModule(H, lr, seed=16)
    blk = moe.MoeBlock(H, F, E, K, moe.QT_Q4_K, moe.QT_Q8_0, True, moe.QT_Q8_0, moe.QT_Q8_0, n_layer=1, max_tokens=T, hc_lr=lr)
    L.upload(blk, 0)
    hc.load(blk, 0)
    R = np.random.default_rng(17).standard_normal((T, 4, H)).astype(np.float32)
    us = []
    for scale in (1.0, 3000.0):
        R[:, :, [11, 1500]] *= np.float32(scale)
        d = h.Dev()
        Rd, y = d.put(R), d.alloc(T * H * 4)
        best = []
        for _ in range(12):
            t0 = time.perf_counter()
            blk.forward_hc_async(0, Rd, T, y)
            blk.sync()
            best.append(time.perf_counter() - t0)
        d.free()
        us.append(min(best) * 1e6)
    blk.close()
    say("us", us)
    assert us[1] <= 2.0 * us[0], us
