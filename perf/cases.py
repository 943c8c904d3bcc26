"""Timed cases of the decode path, through the package's public entry points.

Whole calls (``Context.eval`` / ``eval_all``) run a few layers of the
architectures of ``rustfox_amd.synth`` with a reduced vocabulary; the others
are one stage of a layer through ``Gpu``: a projection, the q/k/v stage, the
gate/up stage, attention, the output head.  Weights are drawn from a pool of
quantised N(0, 0.02) (K-quants) or uniformly ternary blocks, activations are
N(0, 1) and caches N(0, 1), as in the benchmark.
Whole calls keep to a few layers: the int8 activations turn
a last-bit difference from 64-bit sums into a whole step of the quantiser,
layer after layer.

A decode streams every weight from HBM once per token, so a stage's state
holds copies of its matrices (or caches) that successive passes take in turn;
every copy has the same contents.
"""
import math
import os
import tempfile
from types import SimpleNamespace

import numpy as np
import torch

import rustfox_amd as rf
from rustfox_amd import synth

TYPES = {"F16": rf.F16, "Q4_K": rf.Q4_K, "Q6_K": rf.Q6_K, "TQ1_0": rf.TQ1_0, "TQ2_0": rf.TQ2_0}
EPS = 1e-5
POOL = 4096                 # distinct blocks a matrix is drawn from
ROTATE = 110 << 20          # bytes of matrices one state holds, so that three states exceed the caches


def listed():
    return [
        # a chat or document prompt read before the first answer token: the
        # 4B-class ternary layers, 1024 tokens on an empty cache
        dict(name="prompt-4b-1024", kind="eval", model="4b", layers=2, vocab=32768, tokens=1024,
             past=0, rows="last"),
        # the next turn of a conversation: a ragged handful of new tokens on
        # a filled cache, K-quant layers (Q4_K with Q6_K v and ffn_down)
        dict(name="prompt-8b-77", kind="eval", model="8b", layers=2, vocab=16384, tokens=77,
             past=1024, rows="last"),
        # speculative decoding: 8 drafted tokens verified in one pass, the
        # logits of every position
        dict(name="verify-27b-8", kind="eval", model="27b", layers=2, vocab=8192, tokens=8,
             past=4096, rows="all"),
        # one answer token sampled on the host: the 4B-class layers on a
        # 2048-row cache
        dict(name="step-4b", kind="eval", model="4b", layers=4, vocab=32768, tokens=1, past=2048,
             rows="last"),
        # the smallest model's step: bound by launches and latency
        dict(name="step-tiny", kind="eval", model="tiny-512", layers=6, vocab=32000, tokens=1,
             past=32, rows="last"),
        # the benchmark's roofline projection, one token
        dict(name="gemv-tq1-1", kind="gemv", type="TQ1_0", cols=4096, rows=14336, tokens=1),
        # the 8B-class ffn_down of one token
        dict(name="gemv-q6k-1", kind="gemv", type="Q6_K", cols=14336, rows=4096, tokens=1),
        # an 8B-class projection of a verify pass or a prompt's tail
        dict(name="gemv-q4k-8", kind="gemv", type="Q4_K", cols=4096, rows=14336, tokens=8),
        # the 4B-class output head over four drafted tokens
        dict(name="head-f16-4", kind="gemv", type="F16", cols=2560, rows=151936, tokens=4),
        # the 27B-class norm + gate/up + SwiGLU of a verify pass
        dict(name="gate-up-tq2-8", kind="gate_up", type="TQ2_0", cols=5376, rows=21504, tokens=8),
        # one token's attention in the 8B class, the reference's summation order
        dict(name="attn-8b-4096", kind="attn", mode="exact", heads=32, kv_heads=8, head_dim=128,
             past=4096, tokens=1),
        # a verify pass's attention in the 27B class
        dict(name="attn-27b-8192-8", kind="attn", mode="exact", heads=32, kv_heads=16,
             head_dim=128, past=8192, tokens=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eval", "eval", "eval", "gemv", "gemv", "gate_up", "qkv", "attn", "attn"])
    if kind == "eval":
        model = rng.choice(["4b", "8b", "27b", "tiny-512", "tiny-288"])
        layers = {"4b": rng.randint(1, 2), "8b": 1, "27b": 1}.get(model, 6)
        tokens = _log_int(rng, 1, 800 if model == "4b" else 250 if model in ("8b", "27b") else 400)
        return dict(kind="eval", model=model, layers=layers, vocab=rng.choice([8192, 9001, 16384]),
                    tokens=tokens, past=rng.choice([0, _log_int(rng, 1, 2000)]),
                    rows="all" if tokens <= 16 and rng.random() < 0.5 else "last")
    if kind == "gemv":
        t = rng.choice(sorted(TYPES))
        cols = 256 * _log_int(rng, 2, 84)
        if t == "F16":
            cols += 8 * rng.randint(0, 15)
        rows = _log_int(rng, 256, 24000)
        return dict(kind="gemv", type=t, cols=cols, rows=rows, tokens=rng.randint(1, 8))
    if kind == "gate_up":
        t = rng.choice(["TQ1_0", "TQ2_0", "Q4_K", "Q6_K"])
        return dict(kind="gate_up", type=t, cols=256 * _log_int(rng, 2, 21),
                    rows=16 * _log_int(rng, 24, 1344),
                    tokens=rng.randint(1, 8) if t.startswith("TQ") else 1)
    if kind == "qkv":
        t = rng.choice(["TQ1_0", "TQ2_0", "Q4_K", "Q4_K+Q6_K"])
        kv = rng.choice([4, 8, 16])
        return dict(kind="qkv", type=t, cols=256 * _log_int(rng, 4, 21),
                    heads=kv * rng.choice([1, 2, 4]), kv_heads=kv, head_dim=rng.choice([64, 128]),
                    past=_log_int(rng, 1, 4000),
                    tokens=rng.randint(1, 8) if t.startswith("TQ") else 1)
    kv = rng.choice([4, 6, 8, 16])
    return dict(kind="attn", mode=rng.choice(["exact", "exact", "split"]),
                heads=kv * rng.choice([1, 2, 4] if kv > 8 else [1, 2, 4, 5]), kv_heads=kv,
                head_dim=rng.choice([48, 64, 128, 128]), past=_log_int(rng, 16, 8000),
                tokens=rng.choice([1, 1, rng.randint(2, 8)]))


# ------------------------------------------------------------------ weights

_pools = {}


def _pool(t):
    """(POOL blocks as bytes, the same as float64 values) of a weight type."""
    if t not in _pools:
        rng = np.random.default_rng([11, t])
        if t == rf.F16:
            raw = (rng.standard_normal((POOL, 256), dtype=np.float32) * np.float32(0.02))
            raw = raw.astype(np.float16)
            val = raw.astype(np.float64)
            raw = raw.view(np.uint8)
        elif t in (rf.TQ1_0, rf.TQ2_0):
            trits = rng.integers(-1, 2, (POOL, 256))
            d = rng.uniform(0.01, 0.05, POOL).astype(np.float16)
            raw = (synth.tq1_encode if t == rf.TQ1_0 else synth.tq2_encode)(trits, d)
            val = trits * d.astype(np.float64)[:, None]
        else:
            w = rng.standard_normal((POOL, 256), dtype=np.float32) * np.float32(0.02)
            raw = (synth.q4k_quantize if t == rf.Q4_K else synth.q6k_quantize)(w).reshape(POOL, -1)
            val = (_q4k_values if t == rf.Q4_K else _q6k_values)(raw)
        _pools[t] = (np.ascontiguousarray(raw), val)
    return _pools[t]


def _q4k_values(raw):
    """Q4_K: value = d * scale * q - dmin * min per 32 elements (ggml's layout)."""
    d = raw[:, 0:2].copy().view(np.float16).astype(np.float64)
    dmin = raw[:, 2:4].copy().view(np.float16).astype(np.float64)
    s = raw[:, 4:16].astype(np.int64)
    sc = np.concatenate([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
    mn = np.concatenate([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    qs = raw[:, 16:144].astype(np.int64).reshape(-1, 4, 1, 32)
    q = np.concatenate([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    return ((d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]).reshape(-1, 256)


def _q6k_values(raw):
    """Q6_K: value = d * scale * (q - 32) per 16 elements (ggml's layout)."""
    ql = raw[:, :128].astype(np.int64).reshape(-1, 2, 2, 32)       # half, column half, l
    qh = raw[:, 128:192].astype(np.int64).reshape(-1, 2, 1, 32)
    sc = raw[:, 192:208].view(np.int8).astype(np.float64).reshape(-1, 2, 4, 2, 1)
    d = raw[:, 208:210].copy().view(np.float16).astype(np.float64)
    lo = np.concatenate([ql & 15, ql >> 4], 2)                     # half, group, l
    hi = np.concatenate([(qh >> (2 * g)) & 3 for g in range(4)], 2)
    q = ((lo | (hi << 4)) - 32).reshape(-1, 2, 4, 2, 16)
    return (d[:, :, None, None, None] * sc * q).reshape(-1, 256)


def _picks(t, rows, cols, key):
    """Which block of the pool each 256 values of a matrix are."""
    return np.random.default_rng(list(key)).integers(0, POOL, (rows, -(-cols // 256)),
                                                     dtype=np.int32)


def _bytes(t, rows, cols, key):
    raw = _pool(t)[0][_picks(t, rows, cols, key)].reshape(rows, -1)
    return np.ascontiguousarray(raw[:, :synth.row_bytes(t, cols)])


def _values(t, rows, cols, key):
    """The same matrix as float64 on the GPU."""
    pool = torch.from_numpy(_pool(t)[1]).cuda()
    pick = torch.from_numpy(_picks(t, rows, cols, key)).cuda()
    return pool[pick.long()].reshape(rows, -1)[:, :cols]


def _size(t, rows, cols):
    return rows * synth.row_bytes(t, cols)


# ------------------------------------------------------------------- states

_shared = {}


def _gpu():
    if "gpu" not in _shared:
        _shared["gpu"] = rf.Gpu(0)
    return _shared["gpu"]


def _spec(case):
    over = dict(n_layer=case["layers"], n_vocab=case["vocab"], n_ctx=8192)
    return synth.spec(case["model"], **over)


def _model(case):
    """The model a program keeps open: one per architecture, depth and vocabulary."""
    key = ("model", case["model"], case["layers"], case["vocab"])
    if key not in _shared:
        s = _spec(case)
        head, offsets = synth.gguf_header(s)
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "model.gguf")
            with open(path, "wb") as f:
                f.write(head)
                for i, ((name, k, n, t), off) in enumerate(zip(synth.tensor_list(s), offsets)):
                    f.seek(len(head) + off)
                    if name.endswith("norm.weight"):
                        f.write(np.ones(k, np.float32).tobytes())
                    else:
                        f.write(_bytes(t, n, k, (3, i)).data)
            _shared[key] = rf.Model(path)
    return _shared[key]


def _cache_rows(seed, layer, n, width):
    g = torch.Generator().manual_seed(seed * 64 + layer)
    return [torch.randn(n, width, generator=g) for _ in range(2)]


def _tokens(case, seed):
    return np.random.default_rng([seed, 5]).integers(0, case["vocab"], case["tokens"],
                                                     dtype=np.uint32)


def _randn(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


class _Dev:
    """A torch tensor on the GPU under the name the package's calls use."""

    def __init__(self, t):
        self.t = t.cuda().contiguous()
        self.ptr = self.t.data_ptr()


def _quads(v):
    """Rows of a value cache in the device's order: four positions of a column side by side."""
    n, w = v.shape
    pad = torch.zeros((-n) % 4, w, dtype=v.dtype, device=v.device)
    return torch.cat([v, pad]).reshape(-1, 4, w).transpose(1, 2).contiguous()


def _rope(n, hd):
    ex = 10000.0 ** (-2.0 * torch.arange(hd // 2, dtype=torch.float64) / hd)
    th = torch.arange(n, dtype=torch.float64)[:, None] * ex
    return th.cos().float(), th.sin().float()


def _copies(size):
    return max(1, min(24, ROTATE // max(size, 1)))


def _mats(case):
    """(type, rows) of the matrices of a stage."""
    if case["kind"] == "gemv":
        return [(TYPES[case["type"]], case["rows"])]
    if case["kind"] == "gate_up":
        return [(TYPES[case["type"]], case["rows"])] * 2
    a, b = (case["type"].split("+") * 2)[:2]
    q, kv = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    return [(TYPES[a], q), (TYPES[a], kv), (TYPES[b], kv)]


def prepare(case, seed):
    s = SimpleNamespace(case=case, turn=0)
    if case["kind"] == "eval":
        m = _model(case)
        s.ctx = m.context(case["past"] + case["tokens"] + 16)
        width = m.info.n_head_kv * m.info.head_dim
        if case["past"]:
            for l in range(case["layers"]):
                k, v = _cache_rows(seed, l, case["past"], width)
                s.ctx.set_kv(l, 0, k.numpy(), v.numpy())
        s.tokens = _tokens(case, seed)
        return s
    s.gpu = _gpu()
    M = case["tokens"]
    if case["kind"] == "attn":
        h, kvh, hd, past = case["heads"], case["kv_heads"], case["head_dim"], case["past"]
        s.n_ctx = past + M
        n = _copies(8 * s.n_ctx * kvh * hd)
        k, v = _cache_rows(seed, 0, s.n_ctx, kvh * hd)
        k, v = k.cuda(), _quads(v.cuda())
        s.caches = [(_Dev(k.clone()), _Dev(v.clone())) for _ in range(n)]
        s.q = _Dev(_randn(seed, M, h * hd))
        s.out = _Dev(torch.zeros(M, h * hd))
        s.pos = _Dev(torch.tensor([past], dtype=torch.int32))
        torch.cuda.synchronize()
        return s
    cols = case["cols"]
    mats = _mats(case)
    host = [_bytes(t, n, cols, (seed, i)) for i, (t, n) in enumerate(mats)]
    s.mats = [[s.gpu.tensor(t, cols, n, b) for (t, n), b in zip(mats, host)]
              for _ in range(_copies(sum(b.nbytes for b in host)))]
    s.x = _Dev(_randn(seed, M, cols))
    if case["kind"] != "gemv":
        s.norm = _Dev(1.0 + 0.1 * _randn(seed + 1, cols))
    s.out = _Dev(torch.zeros(M, mats[0][1]))
    if case["kind"] == "qkv":
        s.n_ctx = case["past"] + M
        width = case["kv_heads"] * case["head_dim"]
        s.cos, s.sin = (_Dev(t) for t in _rope(s.n_ctx, case["head_dim"]))
        k, v = _cache_rows(seed, 0, s.n_ctx, width)
        s.k, s.v = _Dev(k), _Dev(_quads(v.cuda()))
        s.pos = _Dev(torch.tensor([case["past"]], dtype=torch.int32))
    torch.cuda.synchronize()
    return s


def run(s):
    case, M = s.case, s.case["tokens"]
    if case["kind"] == "eval":
        s.ctx.set_position(case["past"])
        return s.ctx.eval_all(s.tokens) if case["rows"] == "all" else s.ctx.eval(s.tokens)
    s.turn += 1
    if case["kind"] == "attn":
        k, v = s.caches[s.turn % len(s.caches)]
        s.gpu.attention(s.out, s.q, k, v, case["heads"], case["kv_heads"], case["head_dim"], M,
                        s.pos, s.n_ctx, rf.ATTN_EXACT if case["mode"] == "exact" else rf.ATTN_SPLIT)
        return s.out.t
    w = s.mats[s.turn % len(s.mats)]
    if case["kind"] == "gemv":
        s.gpu.gemv(w[0], s.x, M, s.out)
        return s.out.t
    if case["kind"] == "gate_up":
        s.gpu.gate_up_silu(w[0], w[1], s.x, M, s.norm, EPS, s.out)
        return s.out.t
    s.gpu.qkv_rope(w[0], w[1], w[2], s.x, M, s.norm, EPS, s.out, s.cos, s.sin, s.pos, s.n_ctx,
                   s.k, s.v, case["head_dim"])
    return [s.out.t, s.k.t, s.v.t]


# ------------------------------------------------------------ what it takes

def _attn_work(M, past, heads, kv_heads, hd):
    pairs = M * past + M * (M + 1) // 2
    return (8 * (past + M) * kv_heads * hd + 8 * M * heads * hd, 4 * pairs * heads * hd)


def work(case):
    M = case["tokens"]
    if case["kind"] == "eval":
        s = _spec(case)
        byts = flops = 0
        for name, k, n, t in synth.tensor_list(s)[2:]:
            rows = M if name != "output.weight" or case["rows"] == "all" else 1
            byts += _size(t, max(n, 1), k)
            flops += 2 * rows * k * n
        b, f = _attn_work(M, case["past"], s.n_head, s.n_head_kv, s.head_dim)
        rows = M if case["rows"] == "all" else 1
        byts += s.n_layer * b + 2 * M * s.n_embd + 4 * rows * s.n_vocab
        return {"bytes": byts, "flops": flops + s.n_layer * f}
    if case["kind"] == "attn":
        b, f = _attn_work(M, case["past"], case["heads"], case["kv_heads"], case["head_dim"])
        return {"bytes": b, "flops": f}
    mats = _mats(case)
    rows = sum(n for _, n in mats)
    out = mats[0][1] if case["kind"] == "gate_up" else rows
    return {"bytes": sum(_size(t, n, case["cols"]) for t, n in mats) + 4 * M * (case["cols"] + out),
            "flops": 2 * M * case["cols"] * rows}


def tolerance(case):
    # the package computes every sum in the reference's order and promises its
    # bits; split attention merges float32 partial softmaxes in any order
    # (measured against 64 bits: about 2e-7)
    if case.get("mode") == "split":
        return {"rel": 1e-5}
    return "exact"


# ------------------------------------------------------------- in 64 bits

def _quantise(x, t):
    """The int8 activations of a weight type's products, as the values they stand for: one
    scale a token for the ternary types, one per 256 values for the K-quants, none for floats."""
    if t == rf.F16:
        return x
    shape = x.shape
    y = x.reshape(shape[0], -1, 256) if t in (rf.Q4_K, rf.Q6_K) else x.reshape(shape[0], 1, -1)
    amax = y.abs().amax(2, keepdim=True)
    v = y * (127.0 / amax)
    q = torch.sign(v) * torch.floor(v.abs() + 0.5)
    return (q.clamp(-127, 127) * (amax / 127.0)).reshape(shape)


def _product(x, t, rows, cols, key):
    return _quantise(x, t) @ _values(t, rows, cols, key).T


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w


def _rotate(x, cos, sin, hd):
    y = x.reshape(x.shape[0], -1, hd // 2, 2)
    c, s = cos[:, None, :].double(), sin[:, None, :].double()
    a, b = y[..., 0], y[..., 1]
    return torch.stack([a * c - b * s, a * s + b * c], 3).reshape(x.shape)


def _attend(q, k, v, past, heads, kv_heads, hd):
    M, n = q.shape[0], k.shape[0]
    seen = torch.arange(n, device=q.device)[None, :] <= past + torch.arange(M, device=q.device)[:, None]
    out = []
    for h in range(heads):
        j = h // (heads // kv_heads)
        s = (q[:, h * hd:(h + 1) * hd] @ k[:, j * hd:(j + 1) * hd].T) / math.sqrt(hd)
        p = torch.softmax(s.masked_fill(~seen, -math.inf), 1)
        out.append(p @ v[:, j * hd:(j + 1) * hd])
    return torch.cat(out, 1)


def _silu(g, u):
    return g / (1 + torch.exp(-g)) * u


def _exact_eval(case, seed):
    s = _spec(case)
    tl = synth.tensor_list(s)
    at = {name: (i, k, n, t) for i, (name, k, n, t) in enumerate(tl)}

    def project(x, name):
        i, k, n, t = at[name]
        return _product(x, t, n, k, (3, i))

    i, k, n, t = at["token_embd.weight"]
    pick = _picks(t, n, k, (3, i))[_tokens(case, seed)]
    x = torch.from_numpy(_pool(t)[1][pick].reshape(case["tokens"], -1)[:, :k]).cuda()
    past, M = case["past"], case["tokens"]
    th = torch.arange(past + M, dtype=torch.float64)[:, None] * s.rope_base ** (
        -2.0 * torch.arange(s.head_dim // 2, dtype=torch.float64) / s.head_dim)
    cos, sin = (f(th).float().double().cuda()[past:] for f in (torch.cos, torch.sin))
    kv = s.n_head_kv * s.head_dim
    for l in range(s.n_layer):
        p = "blk.%d." % l
        h = _rms(x, 1.0)
        q = _rotate(project(h, p + "attn_q.weight"), cos, sin, s.head_dim)
        kk = _rotate(project(h, p + "attn_k.weight"), cos, sin, s.head_dim)
        vv = project(h, p + "attn_v.weight")
        if past:
            ck, cv = _cache_rows(seed, l, past, kv)
            kk, vv = torch.cat([ck.double().cuda(), kk]), torch.cat([cv.double().cuda(), vv])
        a = _attend(q, kk, vv, past, s.n_head, s.n_head_kv, s.head_dim)
        x = x + project(a, p + "attn_output.weight")
        h = _rms(x, 1.0)
        h = _silu(project(h, p + "ffn_gate.weight"), project(h, p + "ffn_up.weight"))
        x = x + project(h, p + "ffn_down.weight")
    y = project(_rms(x if case["rows"] == "all" else x[-1:], 1.0), "output.weight")
    return y if case["rows"] == "all" else y[0]


def exact(case, seed):
    M = case["tokens"]
    if case["kind"] == "eval":
        return _exact_eval(case, seed).cpu()
    if case["kind"] == "attn":
        h, kvh, hd, past = case["heads"], case["kv_heads"], case["head_dim"], case["past"]
        k, v = (c.double().cuda() for c in _cache_rows(seed, 0, past + M, kvh * hd))
        return _attend(_randn(seed, M, h * hd).double().cuda(), k, v, past, h, kvh, hd)
    cols, mats = case["cols"], _mats(case)
    x = _randn(seed, M, cols).double().cuda()
    if case["kind"] != "gemv":
        x = _rms(x, (1.0 + 0.1 * _randn(seed + 1, cols)).double().cuda())
    y = [_product(x, t, n, cols, (seed, i)) for i, (t, n) in enumerate(mats)]
    if case["kind"] == "gemv":
        return y[0]
    if case["kind"] == "gate_up":
        return _silu(y[0], y[1])
    past, hd = case["past"], case["head_dim"]
    cos, sin = (t[past:].cuda() for t in _rope(past + M, hd))
    k, v = (c.double().cuda() for c in _cache_rows(seed, 0, past + M, case["kv_heads"] * hd))
    k[past:], v[past:] = _rotate(y[1], cos, sin, hd), y[2]
    return [_rotate(y[0], cos, sin, hd), k, _quads(v)]
