"""The prefill expert GEMMs over spans of one expert's positions (gate/up in two int8 planes, the q8_0 family's down),
at the edges of their position tiles and spans, against the oracle's compute_many bit for bit; every gate/up and down type
they take, rows of K that end in a partial unit, and codebooks with too many levels for the planes' digits."""
import numpy as np
import pytest

from tests import harness as h
from tests.harness import moe
from tests.test_gpu_parity import say

pytestmark = pytest.mark.gpu

# Positions an expert gets: around a position tile (16), a short span (64), a long one (128), and past two of each.
COUNTS = (1, 15, 16, 17, 63, 64, 65, 128, 129, 257)
Q8, Q4, I3, NL, XS, Q2, XX, S2 = (moe.QT_Q8_0, moe.QT_Q4_K, moe.QT_IQ3_S, moe.QT_IQ4_NL, moe.QT_IQ4_XS, moe.QT_Q2_0,
                                  moe.QT_IQ3_XXS, moe.QT_IQ2_S)


def check(gt, dt, H, F, codebooks, limit=0.0, scales=None):
    E = len(COUNTS)
    L = h.Layer(H, F, E, E, gt, dt, has_shared=False, seed=910 + gt + F, swiglu_limit=limit)
    blk = moe.MoeBlock(H, F, E, E, gt, dt, False, max_tokens=260, swiglu_limit=limit)
    if {gt, dt} & set(moe.CODEBOOK_TYPES):
        blk.set_codebooks(codebooks)
    r = np.random.default_rng(5)
    x = h.tokens(911, 260, H)
    x[3] = 0.0  # a row whose scale is zero
    if scales is not None:
        x *= np.repeat(scales[r.integers(len(scales), size=(260, H // 256))], 256, axis=1).astype(np.float32)
    # Each expert's tokens in an order of its own; a token's jobs in expert order.
    toks = [set(r.permutation(260)[:c].tolist()) for c in COUNTS]
    jobs = [(L.experts[e], t, float(r.normal())) for t in range(260) for e in range(E) if t in toks[e]]
    y = blk.compute_many(jobs, x)
    yo = h.orc_compute_many(gt, dt, H, F, jobs, x, swiglu_limit=limit)
    blk.close()
    assert np.array_equal(y, yo), h.max_abs(y, yo)


@pytest.mark.parametrize("gt,dt,H,F", [(Q4, NL, 512, 640), (I3, Q2, 512, 320), (XX, NL, 1024, 640), (S2, Q8, 512, 256),
                                       (XS, NL, 512, 448), (I3, Q4, 2560, 512), (S2, Q2, 2560, 640), (Q8, Q8, 512, 512),
                                       (Q4, Q8, 512, 960), (Q4, Q8, 512, 896), (XX, NL, 512, 896), (I3, NL, 512, 768),
                                       (S2, Q2, 512, 704)],
                         ids=lambda v: moe.TYPE_NAMES.get(v, str(v)))
def test_spans(gt, dt, H, F):
    say("spans", (moe.TYPE_NAMES[gt], moe.TYPE_NAMES[dt], H, F))
    check(gt, dt, H, F, h.CODEBOOKS)


@pytest.mark.parametrize("gt", [Q4, I3], ids=lambda v: moe.TYPE_NAMES[v])
def test_span_lists(gt):
    """The lists' order: an expert with more positions than the last class, several with as many spans as each other, rests of
    one tile, experts without positions."""
    counts = [80] * 9 + [1090, 0, 128, 128, 16, 1, 0, 65] + [144] * 4
    E, T, H, F = len(counts), 1100, 512, 256
    L = h.Layer(H, F, E, E, gt, Q8, has_shared=False, seed=77)
    say("span lists", moe.TYPE_NAMES[gt])
    blk = moe.MoeBlock(H, F, E, 15, gt, Q8, False, max_tokens=T)
    r = np.random.default_rng(6)
    x = h.tokens(78, T, H)
    room = np.full(T, 16)  # jobs a token may still take
    jobs = []
    for e, c in enumerate(counts):
        toks = r.permutation(np.flatnonzero(room))[:c]
        room[toks] -= 1
        jobs += [(L.experts[e], int(t), float(r.normal())) for t in toks]
    y = blk.compute_many(jobs, x)
    blk.close()
    yo = h.orc_compute_many(gt, Q8, H, F, jobs, x)
    assert np.array_equal(y, yo), h.max_abs(y, yo)


@pytest.mark.parametrize("spans,walk", [(80, 2), (160, 4), (320, 8)])
@pytest.mark.parametrize("dt", [Q8, NL, Q2], ids=lambda v: moe.TYPE_NAMES[v])
def test_down_walk(dt, spans, walk):
    """A work-group of the q8_0 family's down that walks several 64-row groups (their number follows from the spans and n_embd:
    pf_down.h's down_walk, restated), rows that end in half a unit, spans of one position, of several tiles and full ones."""
    H, F, E, K = 2560, 640, spans - 4, 15
    groups = lambda w: (spans + 7) // 8 * 8 * (H // 64 // w)  # noqa: E731
    assert next(w for w in (8, 4, 2, 1) if w == 1 or groups(w) >= 1536) == walk
    counts = [1] * (E - 12) + [16, 17, 33, 48, 63, 64, 64, 50, 128, 100, 65, 70]
    assert sum((c + 63) // 64 for c in counts) == spans
    say("down walk", (moe.TYPE_NAMES[dt], spans, walk))
    L = h.Layer(H, F, 4, 1, Q4, dt, has_shared=False, seed=55)
    T = 130
    blk = moe.MoeBlock(H, F, 64, K, Q4, dt, False, max_tokens=T)
    r = np.random.default_rng(spans)
    x = h.tokens(56, T, H)
    room = np.full(T, K + 1)
    jobs, ojobs = [], []
    for e, c in enumerate(counts):
        g, u, d = L.experts[e % 4]
        mine = (g.copy(), u, d)  # an expert of its own by its gate's address
        toks = np.argsort(-room + 0.5 * r.random(T))[:c]
        room[toks] -= 1
        for t in toks:
            w = float(r.normal())
            jobs.append((mine, int(t), w)), ojobs.append((L.experts[e % 4], int(t), w))
    y = blk.compute_many(jobs, x)
    blk.close()
    yo = h.orc_compute_many(Q4, dt, H, F, ojobs, x)
    assert np.array_equal(y, yo), h.max_abs(y, yo)


def test_spans_swiglu_limit():
    check(XX, NL, 512, 256, h.CODEBOOKS, limit=0.05)


@pytest.mark.parametrize("gt", [Q4, I3, XX, S2, XS], ids=lambda v: moe.TYPE_NAMES[v])
def test_spans_tiny_scales(gt):
    """Units whose activation scale makes its product with the weights' subnormal or zero beside units of ordinary size, and
    rows of nothing else."""
    say("spans, tiny scales", moe.TYPE_NAMES[gt])
    check(gt, NL, 1024, 256, h.CODEBOOKS, scales=np.exp2([0.0, 0.0, -20.0, -85.0, -95.0, -105.0, -118.0]))


@pytest.mark.parametrize("gt,dt", [(Q4, NL), (I3, Q2), (XX, Q8), (S2, NL), (XS, Q8)], ids=lambda v: moe.TYPE_NAMES[v])
def test_spans_infinite_scales(gt, dt):
    """Blocks whose scale is infinite in rows of up (the SwiGLU limit makes their values finite again) and, infinite or NaN, in
    rows of down: no other row or position sees them."""
    say("spans, infinite scales", (moe.TYPE_NAMES[gt], moe.TYPE_NAMES[dt]))
    H, F, T, E, limit = 512, 256, 70, 3, 0.05
    L = h.Layer(H, F, E, E, gt, dt, has_shared=False, seed=970 + gt, swiglu_limit=limit)
    x = h.tokens(971, T, H)
    jobs = [(L.experts[e], t, 0.5 + e) for t in range(T) for e in range(E) if (t + e) % 5]
    clean = h.orc_compute_many(gt, dt, H, F, jobs, x, swiglu_limit=limit)
    up, down = (L.experts[1][m].reshape((F, H)[m - 1], -1) for m in (1, 2))
    up[[5, 100], :2] = 0x00, 0x7C
    yo = h.orc_compute_many(gt, dt, H, F, jobs, x, swiglu_limit=limit)
    assert np.isfinite(yo).all() and not np.array_equal(yo, clean)
    down[[7, 300], :2], down[33, :2] = (0x00, 0xFC), (0x00, 0x7E)
    yo = h.orc_compute_many(gt, dt, H, F, jobs, x, swiglu_limit=limit)
    assert np.isfinite(np.delete(yo, [7, 300, 33], axis=1)).all() and np.isinf(yo[:, 7]).any() and np.isnan(yo[:, 33]).any()
    blk = moe.MoeBlock(H, F, 8, E, gt, dt, False, max_tokens=T, swiglu_limit=limit)
    if gt in moe.CODEBOOK_TYPES:
        blk.set_codebooks(h.CODEBOOKS)
    y = blk.compute_many(jobs, x)
    blk.close()
    assert np.array_equal(y, yo, equal_nan=True)


@pytest.mark.parametrize("gt", [XX, S2], ids=lambda v: moe.TYPE_NAMES[v])
def test_codebooks_past_the_levels(gt):
    """A caller's tables whose bytes take more values than the planes' digit tables hold run the general path."""
    book = h.CODEBOOKS.copy()
    n = 9216 if gt == XX else 8192
    book[n - 4:n] = (7, 9, 11, 13)
    try:
        h.oracle.orc_set_codebooks(h.ptr(book))
        moe.synth_set_codebooks(book)
        check(gt, NL, 512, 256, book)
    finally:
        h.oracle.orc_set_codebooks(h.ptr(h.CODEBOOKS))
        moe.synth_set_codebooks(h.CODEBOOKS)
