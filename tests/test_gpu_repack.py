"""The device's repack of borrowed experts from the file's layout, against the oracle's compute_many bit for bit: types of every
piece form, fewer and more experts than the staging buffer holds, down rows in two regions that part inside a unit, and
rows whose last unit is not full."""
import numpy as np
import pytest

from tests import harness as h
from tests.harness import moe
from tests.test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("types", [(moe.QT_Q5_K, moe.QT_Q6_K), (moe.QT_Q6_K, moe.QT_Q5_K), (moe.QT_IQ4_XS, moe.QT_IQ4_NL),
                                   (moe.QT_IQ3_XXS, moe.QT_Q8_0), (moe.QT_IQ2_S, moe.QT_Q2_0), (moe.QT_IQ3_S, moe.QT_Q4_K)])
@pytest.mark.parametrize("n", [1, 16, 17, 40])
def test_repack_of_borrowed_experts(types, n):
    gt, dt = types
    say("repack", moe.TYPE_NAMES[gt], moe.TYPE_NAMES[dt], "experts", n)
    bv, bb = moe.BLOCK[dt]
    H, F = 512, (640 if bv < 256 else 768)
    L = h.Layer(H, F, n, 1, gt, dt, has_shared=False, seed=700 + n)
    blk = moe.MoeBlock(H, F, 64, 2, gt, dt, has_shared=False, max_tokens=64)
    if {gt, dt} & set(moe.CODEBOOK_TYPES):
        blk.set_codebooks(h.CODEBOOKS)
    T = 40 if n > 16 else 8
    x = h.tokens(701 + n, T, H)
    jobs, ojobs = [], []
    for j in range(max(n, T)):
        g, u, d = L.experts[j % n]
        nb = F // bv
        b0 = 1 + (j % n) % (nb - 1)
        rows = d.reshape(H, nb * bb)
        d2 = np.ascontiguousarray(np.concatenate([rows[:, :b0 * bb].ravel(), rows[:, b0 * bb:].ravel()]))
        jobs.append(((g, u, d2, 2, (b0, nb - b0)), j % T, 1.0))
        ojobs.append(((g, u, d), j % T, 1.0))
    y = blk.compute_many(jobs, x)
    yo = h.orc_compute_many(gt, dt, H, F, ojobs, x)
    assert np.array_equal(y, yo), h.max_abs(y, yo)
    blk.close()


def test_load_allocates_nothing():
    """A context holds all that its loads need once it is open."""
    say("loads allocate nothing")
    L = h.Layer(512, 256, 8, 2, moe.QT_Q4_K, moe.QT_Q8_0, moe.QT_Q8_0, moe.QT_Q8_0, seed=3)
    blk = L.block()
    held = blk.device_bytes()
    L.upload(blk)
    assert blk.device_bytes() == held
    blk.close()
