"""The work a program gives the MoE block, as measurable cases.

A serving program opens one context per model, keeps every layer's weights resident and then calls the block layer
after layer: one token (decode) or a few (speculative verify), prompts cut into chunks (prefill), with or without the
hyper-connection mix around the block, from device buffers on its stream or through the synchronous host call, and,
where experts stay in host memory, compute_many on borrowed weights. The shapes and types are those of the benchmark
configurations (2048 x 512, 512 experts, top 10; Q8_0, Q4_K, IQ3_S) and of the model file's layers (2560 x 640; IQ3_XXS,
IQ2_S, IQ3_S, IQ4_XS with IQ4_NL or Q2_0 down and a shared expert of types of its own).

A state holds its own context, with weights drawn from the seed: a pool of eight experts' matrices (N(0, 0.02), the
library's quantisers), loaded in turn as the layer's 512 experts, so that every expert has an address and bytes in
device memory of its own; the other layers hold device copies of them with routers and biases of their own. Small
calls go through several layers a pass, as a decode step does, so that weights come from memory and not from a cache.
"""
import functools
import math
import re

import numpy as np
import torch

import c0ven_amd as moe

E, K = 512, 10  # routed experts of a layer and those a token uses (every configuration's)
POOL = 8        # distinct experts' matrices drawn for a state
SIGMA = 0.02

# Type sets: routed gate and up, routed down, shared gate, shared up, shared down.
Q8 = "Q8_0 Q8_0 Q8_0 Q8_0 Q8_0"
Q4 = "Q4_K Q4_K Q4_K Q4_K Q4_K"
I3 = "IQ3_S IQ3_S IQ3_S IQ3_S IQ3_S"
MIX = "IQ3_S Q4_K Q8_0 Q8_0 Q8_0"
# Layers of the model file (tests/golden/model_layer_types.json): 0, 1 and later ones' kinds.
M_XXS = "IQ3_XXS IQ4_NL Q4_K IQ4_XS IQ4_NL"
M_2S = "IQ2_S Q2_0 IQ4_XS Q4_K IQ4_NL"
M_2N = "IQ2_S IQ4_NL Q4_K Q4_K IQ4_NL"


def _case(name, kind, T, types, layers, zipf=0.0, H=2048, F=512, lr=0, exact_router=False):
    return {"name": name, "kind": kind, "T": T, "types": types, "layers": layers, "zipf": zipf, "H": H, "F": F, "lr": lr,
            "exact_router": exact_router}


def listed():
    return [
        # One generated token through the synchronous host call, a layer of the model file: the smallest call.
        _case("host_decode_1", "host", 1, M_XXS, 1, H=2560, F=640),
        # Decode of one token, device buffers, several layers a pass.
        _case("decode_1_q8_0", "block", 1, Q8, 4),
        # Speculative verify of 8 tokens with the skewed expert use of real routing.
        _case("verify_8_q4_k", "block", 8, Q4, 4, zipf=1.1),
        # The largest batch the decode kernel takes, experts used evenly, the mixed types of the 48-layer stack.
        _case("decode_16_mixed", "block", 16, MIX, 2),
        # The model's own step: hyper-connection mix and combine around each block, a short verify.
        _case("decode_hc_3", "hc", 3, M_2S, 4, H=2560, F=640, lr=320),
        # A short prompt, just past the decode kernel, ragged.
        _case("prompt_37_q4_k", "block", 37, Q4, 1),
        # An ordinary prompt on the model file's types.
        _case("prompt_301_model", "block", 301, M_XXS, 1, zipf=1.1, H=2560, F=640),
        # A whole prefill chunk, the benchmark's configuration.
        _case("prefill_2048_q4_k", "block", 2048, Q4, 1, zipf=1.1),
        # A chunk of the 48-layer stack.
        _case("prefill_2048_mixed", "block", 2048, MIX, 1, zipf=1.1),
        # The largest chunk, the model file's smallest types.
        _case("prefill_4096_model", "block", 4096, M_2N, 1, zipf=1.1, H=2560, F=640),
        # A prompt of the model with the hyper-connection mix around the block.
        _case("prefill_hc_1000", "hc", 1000, M_XXS, 1, zipf=1.1, H=2560, F=640, lr=320),
        # Experts left in host memory, borrowed for the call: a few tokens' misses.
        _case("borrowed_4", "many", 4, M_XXS, 1, H=2560, F=640),
    ]


def draw(rng):
    """A case of the same ranges: tokens spread over the logarithm of 1..4096 (the host call to 64, borrowed experts to
    32), any of the type sets on its shapes, even or skewed expert use."""
    kind = rng.choices(["block", "hc", "host", "many"], [60, 20, 10, 10])[0]
    model = kind in ("hc", "many") or rng.random() < 0.45
    most = {"block": 4096, "hc": 2048, "host": 64, "many": 32}[kind]
    T = min(most, int(math.exp(rng.uniform(0.0, math.log(most + 1)))))
    types = rng.choice([M_XXS, M_2S, M_2N, M_XXS] if model else [Q8, Q4, I3, MIX, Q4])
    layers = 1 if kind == "many" else 4 if T <= 4 else 2 if T <= 64 else 1
    c = _case("", kind, T, types, layers, rng.choice([0.0, 1.1]), 2560 if model else 2048, 640 if model else 512,
              320 if kind == "hc" else 0, kind == "block" and T > 16 and rng.random() < 0.1)
    del c["name"]
    return c


def _types(case):
    return [moe.TYPE_IDS[t] for t in case["types"].split()]


# ---------------------------------------------------------------------------------------------------------------------
# Inputs


@functools.lru_cache(None)
def _iq3s_grid():
    """The 512 words of ggml's IQ3_S grid, from the table the library carries."""
    with open("c0ven_amd/csrc/iq3s_grid.h") as f:
        words = re.findall(r"0x([0-9a-fA-F]{8})u", f.read())
    return np.array([int(w, 16) for w in words[:512]], dtype=np.uint32)


IQ4NL = np.array([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113], dtype=np.int8)


@functools.lru_cache(None)
def _codebooks():
    """A codebook buffer with seeded stand-ins for ggml's iq2s_grid and iq3xxs_grid (a caller's tables): distinct words
    of each table's byte values."""
    r = np.random.default_rng(4242)
    buf = np.zeros(moe.QGRID_BYTES, dtype=np.uint8)
    for off, n, width, values in ((moe.QGRID_IQ2S, 1024, 8, [8, 25, 43]),
                                  (moe.QGRID_IQ3XXS, 256, 4, [4, 12, 20, 28, 36, 44, 52, 62])):
        words = set()
        while len(words) < n:
            words.add(bytes(np.array(values, dtype=np.uint8)[r.integers(0, len(values), size=width)]))
        buf[off:off + n * width] = np.frombuffer(b"".join(sorted(words)), np.uint8)
    buf[moe.QGRID_IQ3S:moe.QGRID_IQ3S + 2048] = _iq3s_grid().view(np.uint8)
    buf[moe.QGRID_KVALUES:moe.QGRID_KVALUES + 16] = IQ4NL.view(np.uint8)
    moe.synth_set_codebooks(buf)
    return buf


def _bf16(x):
    """fp32 to bf16 bits, round to nearest even."""
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def _expert(seed, stream, types, F, H):
    """Gate, up and down in the file's layout, of N(0, 0.02) values."""
    return tuple(moe.synth_matrix(seed, 4 * stream + i, t, *((F, H) if i < 2 else (H, F)), sigma=SIGMA, nthreads=16)
                 for i, t in enumerate(types))


def _weights(case, seed):
    """The pool of routed experts and the shared one."""
    gt, dt, sg, su, sd = _types(case)
    _codebooks()
    H, F = case["H"], case["F"]
    return [_expert(seed, e, (gt, gt, dt), F, H) for e in range(POOL)], _expert(seed, POOL, (sg, su, sd), F, H)


def _router(case, seed, layer):
    H = case["H"]
    w = moe.synth_normal(seed, 1000 + layer, (E + 1) * H, SIGMA, 16)
    return _bf16(w).reshape(E + 1, H), moe.zipf_bias(seed + 7 * layer, E, case["zipf"]) if case["zipf"] else None


def _hc_module(case, seed, layer):
    H, lr, base = case["H"], case["lr"], 2000 + 8 * layer
    D = 4 * H
    return ((1.0 + moe.synth_normal(seed, base, D, 0.1, 16)).astype(np.float32),
            _bf16(moe.synth_normal(seed, base + 1, lr * D, SIGMA, 16)).reshape(lr, D),
            _bf16(moe.synth_normal(seed, base + 2, 4 * D, SIGMA, 16)).reshape(4, D),
            _bf16(moe.synth_normal(seed, base + 3, D * lr, SIGMA, 16)).reshape(D, lr))


def _x(case, seed):
    """The block's input (RMSNorm-like), or the residual streams."""
    n = 4 if case["kind"] == "hc" else 1
    x = moe.synth_normal(seed, 3000, case["T"] * n * case["H"], 1.0, 16)
    return x.reshape((case["T"], n, case["H"]) if n > 1 else (case["T"], case["H"]))


def _jobs(case, seed):
    """compute_many's jobs as (expert, token, weight): K different experts a token out of a set with some overlap between
    the tokens, weights summing to one."""
    r = np.random.default_rng(seed)
    T = case["T"]
    n = min(48, 12 + 4 * (T - 1))
    jobs = []
    for t in range(T):
        w = r.exponential(size=K)
        jobs += [(int(e), t, float(v)) for e, v in zip(r.choice(n, size=K, replace=False), (w / w.sum()).astype(np.float32))]
    return n, jobs


@functools.lru_cache(None)
def _stream():
    """The program's stream."""
    return torch.cuda.Stream()


class State:
    pass


def prepare(case, seed):
    s = State()
    s.kind, s.T, s.layers = case["kind"], case["T"], case["layers"]
    T, H, F = case["T"], case["H"], case["F"]
    gt, dt, sg, su, sd = _types(case)
    pool, shared = _weights(case, seed)
    many = case["kind"] == "many"
    s.blk = moe.MoeBlock(H, F, 32 if many else E, K, gt, dt, True, sg, sd, n_layer=case["layers"], max_tokens=max(16, T),
                         hc_lr=case["lr"], sh_up_type=su, exact_router=case["exact_router"])
    if {gt, dt, sg, su, sd} & set(moe.CODEBOOK_TYPES):
        s.blk.set_codebooks(_codebooks())
    x = _x(case, seed)
    if many:
        n, jobs = _jobs(case, seed)
        experts = [tuple(m.copy() for m in pool[e % POOL]) for e in range(n)]
        s.jobs = [(experts[e], t, w) for e, t, w in jobs]
        s.x = x
        return s
    for l in range(case["layers"]):
        s.blk.load_router(l, *_router(case, seed, l))
        if case["lr"]:
            s.blk.load_hc(l, *_hc_module(case, seed, l))
    for e in range(E):
        s.blk.load_expert(0, e, *pool[e % POOL])
    s.blk.load_expert(0, E, *shared)
    for l in range(1, case["layers"]):
        s.blk.copy_experts(0, l)
    if case["kind"] == "host":
        s.x = x
        return s
    with torch.cuda.stream(_stream()):
        s.x = torch.from_numpy(x).cuda()
        s.y = torch.empty((case["layers"], T, H), device="cuda")
        s.ids = torch.empty((case["layers"], T, K), dtype=torch.int32, device="cuda")
        s.w = torch.empty((case["layers"], T, K), device="cuda")
        if case["kind"] == "hc":
            s.R = torch.empty_like(s.x)
    _stream().synchronize()
    return s


def run(s):
    if s.kind == "many":
        return {"y": s.blk.compute_many(s.jobs, s.x)}
    if s.kind == "host":
        out = [s.blk.forward(l, s.x) for l in range(s.layers)]
        return {"y": [o[0] for o in out], "ids": [o[1] for o in out], "w": [o[2] for o in out]}
    q = _stream().cuda_stream
    if s.kind == "hc":  # the residual streams start from the embedding's and pass from layer to layer
        with torch.cuda.stream(_stream()):
            s.R.copy_(s.x)
        for l in range(s.layers):
            s.blk.forward_hc_async(l, s.R.data_ptr(), s.T, s.y[l].data_ptr(), s.ids[l].data_ptr(), s.w[l].data_ptr(), q)
        return {"R": s.R, "y": s.y, "ids": s.ids, "w": s.w}
    for l in range(s.layers):
        s.blk.forward_async(l, s.x.data_ptr(), s.T, s.y[l].data_ptr(), s.ids[l].data_ptr(), s.w[l].data_ptr(), q)
    return {"y": s.y, "ids": s.ids, "w": s.w}


@functools.lru_cache(None)
def _distinct(T, zipf, H):
    """Experts that T tokens use, counted on logits of the layers' distribution (N(0, 0.02 sqrt(H)) + the bias)."""
    r = np.random.default_rng(7)
    bias = moe.zipf_bias(1, E, zipf) if zipf else np.zeros(E, np.float32)
    used = np.zeros(E, bool)
    for _ in range(T):
        used[np.argpartition(-(r.normal(size=E) * SIGMA * math.sqrt(H) + bias), K)[:K]] = True
    return int(used.sum())


def work(case):
    T, H, F, L, lr = case["T"], case["H"], case["F"], case["layers"], case["lr"]
    gt, dt, sg, su, sd = _types(case)

    def nbytes(g, u, d):
        return F * (moe.row_bytes(g, H) + moe.row_bytes(u, H)) + H * moe.row_bytes(d, F)

    if case["kind"] == "many":
        n = min(48, 12 + 4 * (T - 1))
        return {"bytes": n * nbytes(gt, gt, dt) + 8 * T * H, "flops": 6.0 * T * K * F * H}
    b = _distinct(T, case["zipf"], H) * nbytes(gt, gt, dt) + nbytes(sg, su, sd) + 2 * (E + 1) * H + 8 * T * H + 8 * T * K
    f = 6.0 * T * (K + 1) * F * H + 2.0 * T * (E + 1) * H
    if lr:
        b += 2 * 4 * H * (2 * lr + 4) + 16 * H + 2 * 16 * T * H - 4 * T * H
        f += 2.0 * T * 4 * H * (2 * lr + 4)
    return {"bytes": L * b, "flops": L * f}


def tolerance(case):
    """Against float64 sums with the formats' own roundings (bf16 operands, int8 activation codes) the outputs are off by
    what a rounding that falls to the other code leaves: up to 2.6e-4 of y for the block (a code of h), 2.3e-3 for the
    hyper-connection step (also a bf16 of the normed streams, of the low rank or of x, carried through the layers);
    about four times those."""
    return {"rel": 1e-2, "max": 0.1, "differ": 0.0} if case["lr"] else {"rel": 1e-3, "max": 0.02, "differ": 0.0}


# ---------------------------------------------------------------------------------------------------------------------
# The same values in 64 bits: the formats' decoding as their documents state it, float64 products and sums. What the
# operator itself rounds stays rounded (bf16 operands of the router and the mix, int8 activation blocks).


def _f16(b, off):
    return np.ascontiguousarray(b[:, off:off + 2]).view(np.float16).astype(np.float64)[:, 0]


def _scale_min(b):
    """Q4_K's and Q5_K's eight 6-bit scales and minima from their twelve bytes."""
    q = b.astype(np.int64)
    sc = np.concatenate([q[:, :4] & 63, (q[:, 8:12] & 15) | ((q[:, :4] >> 6) << 4)], 1)
    mn = np.concatenate([q[:, 4:8] & 63, (q[:, 8:12] >> 4) | ((q[:, 4:8] >> 6) << 4)], 1)
    return sc, mn


def _signs(bits):
    """-1 where a bit is set: bytes (n, m) to (n, 8 m)."""
    return 1 - 2 * np.unpackbits(bits, axis=1, bitorder="little").astype(np.int64)


def _decode(name, raw, cols):
    """rows x cols values of a matrix of type name in the file's layout."""
    values, size = moe.BLOCK[moe.TYPE_IDS[name]]
    b = raw.reshape(-1, size)
    n = len(b)
    if name == "Q8_0":
        v = _f16(b, 0)[:, None] * b[:, 2:].view(np.int8)
    elif name == "IQ4_NL":
        v = _f16(b, 0)[:, None] * IQ4NL[np.concatenate([b[:, 2:] & 15, b[:, 2:] >> 4], 1)]
    elif name == "Q2_0":
        q = (b[:, 2:, None] >> (2 * np.arange(4, dtype=np.uint8))) & 3
        v = _f16(b, 0)[:, None] * (q.reshape(n, 64).astype(np.int64) - 1)
    elif name == "IQ4_XS":
        h = b[:, 2].astype(np.int64) | (b[:, 3].astype(np.int64) << 8)
        lo = np.stack([b[:, 4:8] & 15, b[:, 4:8] >> 4], 2).reshape(n, 8).astype(np.int64)
        ls = (lo | (((h[:, None] >> (2 * np.arange(8))) & 3) << 4)) - 32
        q = b[:, 8:].reshape(n, 8, 16)
        v = (_f16(b, 0)[:, None] * ls)[:, :, None] * IQ4NL[np.concatenate([q & 15, q >> 4], 2)]
    elif name in ("Q4_K", "Q5_K"):
        sc, mn = _scale_min(b[:, 4:16])
        qs = b[:, 16 if name == "Q4_K" else 48:].reshape(n, 4, 32)
        q = np.stack([qs & 15, qs >> 4], 2).reshape(n, 8, 32).astype(np.int64)
        if name == "Q5_K":
            q = q | (((b[:, None, 16:48] >> np.arange(8, dtype=np.uint8)[None, :, None]) & 1).astype(np.int64) << 4)
        v = (_f16(b, 0)[:, None] * sc)[:, :, None] * q - (_f16(b, 2)[:, None] * mn)[:, :, None]
    elif name == "Q6_K":
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        lo = np.stack([ql & 15, ql >> 4], 2).reshape(n, 2, 4, 32).astype(np.int64)
        hi = ((qh >> (2 * np.arange(4, dtype=np.uint8))[None, None, :, None]) & 3).astype(np.int64)
        sc = b[:, 192:208].view(np.int8).astype(np.int64).repeat(16, 1)
        v = _f16(b, 208)[:, None] * sc * ((lo | (hi << 4)).reshape(n, 256) - 32)
    elif name == "IQ3_S":
        idx = b[:, 2:66].astype(np.int64) | (np.unpackbits(b[:, 66:74], axis=1, bitorder="little").astype(np.int64) << 8)
        g = _iq3s_grid().view(np.uint8).reshape(512, 4)[idx].reshape(n, 256).astype(np.int64) * _signs(b[:, 74:106])
        s = np.stack([b[:, 106:110] & 15, b[:, 106:110] >> 4], 2).reshape(n, 8).astype(np.int64)
        v = (_f16(b, 0)[:, None] * (1 + 2 * s))[:, :, None] * g.reshape(n, 8, 32)
    elif name == "IQ3_XXS":
        table = _codebooks()[moe.QGRID_IQ3XXS:moe.QGRID_IQ3XXS + 1024].reshape(256, 4)
        w = np.ascontiguousarray(b[:, 66:98]).view(np.uint32)
        s7 = ((w[:, :, None] >> np.array([0, 7, 14, 21], dtype=np.uint32)) & 127).astype(np.uint8).reshape(n, 32)
        s8 = s7 | (np.unpackbits(s7[:, :, None], axis=2).sum(2).astype(np.uint8) << 7)
        g = table[b[:, 2:66]].reshape(n, 256).astype(np.int64) * _signs(s8)
        v = (_f16(b, 0)[:, None] * (0.5 + (w >> 28)) * 0.5)[:, :, None] * g.reshape(n, 8, 32)
    elif name == "IQ2_S":
        table = _codebooks()[moe.QGRID_IQ2S:moe.QGRID_IQ2S + 8192].reshape(1024, 8)
        hi = ((b[:, 66:74, None] >> np.array([0, 2, 4, 6], dtype=np.uint8)) & 3).reshape(n, 32).astype(np.int64)
        g = table[b[:, 2:34].astype(np.int64) | (hi << 8)].reshape(n, 256).astype(np.int64) * _signs(b[:, 34:66])
        s = np.stack([b[:, 74:82] & 15, b[:, 74:82] >> 4], 2).reshape(n, 16).astype(np.int64)
        v = (_f16(b, 0)[:, None] * (0.5 + s) * 0.25)[:, :, None] * g.reshape(n, 16, 16)
    return torch.from_numpy(np.ascontiguousarray(v, dtype=np.float64).reshape(-1, cols)).cuda()


def _int8_blocks(x, name):
    """x through the activation blocks a weight type's products take (q8_0 of 32 values, else q8_K of 256), decoded."""
    small = name in ("Q8_0", "IQ4_NL", "Q2_0")
    n, k = x.shape
    v = x.float().reshape(n, -1, 32 if small else 256) if small or k % 256 == 0 else None
    if small:
        top = v.abs().amax(2, keepdim=True)
        q = torch.where(top > 0, torch.round(v * (127.0 / top)), torch.zeros_like(v))
        d = (top / 127.0).half()
    else:
        top = torch.gather(v, 2, v.abs().argmax(2, keepdim=True))
        i = -127.0 / top
        q = torch.where(top != 0, torch.round(i * v).clamp(max=127), torch.zeros_like(v))
        d = torch.where(top != 0, 1.0 / i, torch.zeros_like(i))
    return (q.double() * d.double()).reshape(n, k)


def _ffn(case, mats, which, x):
    """An expert's outputs for the rows x; mats decoded, which: its types' names (gate, up, down)."""
    g, u = (_int8_blocks(x, t) @ m.T for t, m in zip(which, mats[:2]))
    h = g / (1.0 + torch.exp(-g)) * u
    return _int8_blocks(h, which[2]) @ mats[2].T


def _bf16_of(x):
    return x.float().bfloat16().double()


def _bits(b):
    return torch.from_numpy((b.astype(np.uint32) << 16).view(np.float32)).double().cuda()


def exact(case, seed):
    if not torch.cuda.is_available():
        return None
    names = case["types"].split()
    H, F, T = case["H"], case["F"], case["T"]
    pool, shared = _weights(case, seed)
    routed_t, shared_t = (names[0], names[0], names[1]), (names[2], names[3], names[4])
    decode = lambda mats, ts: [_decode(t, m, H if i < 2 else F) for i, (m, t) in enumerate(zip(mats, ts))]  # noqa: E731
    pool, shared = [decode(p, routed_t) for p in pool], decode(shared, shared_t)
    x = torch.from_numpy(_x(case, seed)).double().cuda()
    if case["kind"] == "many":
        _, jobs = _jobs(case, seed)
        y = torch.zeros((T, H), dtype=torch.float64, device="cuda")
        for e, t, w in jobs:
            y[t] += w * _ffn(case, pool[e % POOL], routed_t, x[t:t + 1])[0]
        return {"y": y}
    R, ys, ws = x, [], []
    for l in range(case["layers"]):
        router, bias = _router(case, seed, l)
        if case["lr"]:
            gamma, down, inj, up = _hc_module(case, seed, l)
            n = R / torch.sqrt((R * R).mean(2, keepdim=True) + 1e-6)
            n = n * torch.from_numpy(gamma).double().cuda().reshape(1, 4, H)
            nb = _bf16_of(n).reshape(T, 4 * H)
            v = nb @ _bits(down).T / 4
            a = _bf16_of(v / (1.0 + torch.exp(-v))) @ _bits(up).T
            gate = 2.0 * torch.sigmoid(nb @ _bits(inj).T / 4)
            x = (n * torch.sigmoid(a.reshape(T, 4, H))).sum(1) / 4
        logits = _bf16_of(x) @ _bits(router).T
        gs = torch.sigmoid(logits[:, E])
        logits = logits[:, :E]
        if bias is not None:
            logits = logits + torch.from_numpy(bias).double().cuda()
        p, ids = torch.topk(torch.softmax(logits, 1), K)
        w = p / p.sum(1, keepdim=True).clamp(min=6.1035e-5)
        y = gs[:, None] * _ffn(case, shared, shared_t, x)
        for e in range(POOL):
            t, k = torch.nonzero(ids % POOL == e, as_tuple=True)
            if len(t):
                y.index_add_(0, t, w[t, k][:, None] * _ffn(case, pool[e], routed_t, x[t]))
        ys.append(y)
        ws.append(w)
        if case["lr"]:
            R = R + gate[:, :, None] * y[:, None, :]
    if case["kind"] == "host":
        return {"y": ys, "ids": None, "w": ws}
    out = {"y": torch.stack(ys), "ids": None, "w": torch.stack(ws)}
    return dict(out, R=R) if case["kind"] == "hc" else out
