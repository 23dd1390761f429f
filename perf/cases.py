"""What the quantized matrix-product path is timed on: the calls that an engine makes of it while it serves a model.

Decode (one token): the output projection with the top-k of its logits, the fused gate + up projection, one small
projection. Small batches (a few sequences decoded together, a speculative draft being verified, a short prompt): 2 to
63 tokens. Prefill: 64 to 2048 tokens, one projection or the q, k and v of one activation from an x prepared once, and
the embedding rows with their norm. The weights are GGUF blocks of every type the library reads.

Weights are quantized here from normal values (0.02, as of a trained matrix), block by block, by plain torch code, and
`exact` decodes those bytes in 64 bits, with no code of the library. Activations are normal values whose channels have
magnitudes of their own, a few of them large, as behind a norm layer.
"""
import json
import math
import os
import weakref

import torch

import __graft_entry__

eff = __graft_entry__.package()

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"
BLOCK = {"Q8_0": (32, 34), "Q8_0R": (32, 34), "Q4_K": (256, 144), "Q6_K": (256, 210), "Q2_K": (256, 84),
         "IQ2_XXS": (256, 66)}
TOPK_PAIRS = 8 + 128            # words of the top-k record before its (id, bits) pairs
EPS = 1e-6
PAD = 64                        # readable bytes past a wrapped tensor
CHUNK = 1 << 23                 # weights quantized or decoded at a time
MOST_FLOPS = 2.0 * 8192 * 2048 * 2048
MOST_WEIGHTS = 65536 * 2048


def listed():
    return [
        # decode, one token: the smallest product (an attention projection in the smallest K type)
        {"name": "decode_q2k", "op": "matmul", "type": "Q2_K", "rows": 8192, "k": 2048, "tokens": 1},
        # decode, one token: gate and up with silu(gate) * up, one launch
        {"name": "decode_gate_up_q4k", "op": "gate_up", "type": "Q4_K", "rows": 8192, "k": 2048, "tokens": 1},
        # decode, one token: the output projection and the 40 candidates of the sampler
        {"name": "decode_head_q6k", "op": "head", "type": "Q6_K", "rows": 65536, "k": 2048, "tokens": 1},
        # 8 sequences decoded together: the FFN down projection, few rows and a long k
        {"name": "batch_down_q8", "op": "matmul", "type": "Q8_0", "rows": 2048, "k": 8192, "tokens": 8},
        # a short prompt: an FFN projection of a 7 B model, one token past two tiles of 16
        {"name": "batch_ffn_q4k", "op": "matmul", "type": "Q4_K", "rows": 14336, "k": 4096, "tokens": 33},
        # prompts, from 128 tokens to 2048, in the types' own ranges
        {"name": "prefill_iq2", "op": "matmul", "type": "IQ2_XXS", "rows": 8192, "k": 2048, "tokens": 128},
        {"name": "prefill_down_q6k", "op": "matmul", "type": "Q6_K", "rows": 2048, "k": 8192, "tokens": 300},
        {"name": "prefill_q4k", "op": "matmul", "type": "Q4_K", "rows": 8192, "k": 2048, "tokens": 512},
        # q, k and v of one activation (grouped-query attention), x prepared once
        {"name": "prefill_qkv_q4k", "op": "qkv", "type": "Q4_K", "rows": 4096, "k": 4096, "tokens": 1000},
        {"name": "prefill_q8", "op": "matmul", "type": "Q8_0", "rows": 8192, "k": 2048, "tokens": 512},
        # a long prompt over a repacked tensor
        {"name": "prefill_q8r_long", "op": "matmul", "type": "Q8_0R", "rows": 8192, "k": 2048, "tokens": 2048},
        # the prompt's embedding rows and their first norm
        {"name": "embed_norm_q6k", "op": "embed", "type": "Q6_K", "rows": 65536, "k": 2048, "tokens": 700},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["matmul"] * 6 + ["qkv", "gate_up", "head", "embed"])
    types = ["Q4_K", "Q6_K", "Q8_0", "Q8_0R", "Q2_K", "IQ2_XXS"]
    if op == "embed":
        return {"op": op, "type": rng.choice(types[:5]), "rows": _log(rng, 1000, 65536), "k": 256 * _log(rng, 2, 32),
                "tokens": _log(rng, 1, 1024)}
    t = rng.choice(types)
    if op == "head":
        return {"op": op, "type": rng.choice(["Q6_K", "Q8_0", "Q4_K"]), "rows": _log(rng, 32000, 65536),
                "k": 256 * _log(rng, 4, 8), "tokens": 1}
    rows, k = _log(rng, 512, 32768), 256 * _log(rng, 2, 56)
    if op == "gate_up":
        rows, k = min(rows, 16384), min(k, 8192)   # one launch holds x for all of k
    elif t in ("Q8_0", "Q8_0R") and rng.random() < 0.2:
        k += 32 * rng.randrange(1, 8)          # whole blocks of 32, not of 256
    if rng.random() < 0.7:
        rows = rows // 64 * 64                 # most matrices have a round number of rows
    mats = 2.0 if op == "gate_up" else 1.5 if op == "qkv" else 1.0
    while rows * k * mats > MOST_WEIGHTS:
        rows //= 2
    if op == "gate_up":
        return {"op": op, "type": t, "rows": rows, "k": k, "tokens": rng.randrange(1, 4)}
    lo = 64 if op == "qkv" else 1
    hi = max(lo, min(2048, int(MOST_FLOPS / (2.0 * rows * k * mats))))
    return {"op": op, "type": t, "rows": rows, "k": k, "tokens": _log(rng, lo, hi)}


# ---- weights: GGUF blocks from normal values, and back in 64 bits -----------

def _f16(v):
    """fp16 values as bytes, [..., 2]."""
    return v.to(torch.float16).contiguous().view(torch.uint8).view(*v.shape, 2)


def _q8_0(w):
    w = w.view(-1, 32)
    d = (w.abs().amax(1) / 127).to(torch.float16).float()
    q = (w / d[:, None]).round().clamp(-127, 127).to(torch.int8)
    return torch.cat([_f16(d), q.view(torch.uint8)], 1)


def _low(b):
    """The two nibbles' sources: [..., 2, 32] -> [..., 32] bytes."""
    return b[..., 0, :] | (b[..., 1, :] << 4)


def _scale_min(w, levels, steps):
    """Per group of the last axis: integer scale and minimum, and the block's d and dmin."""
    lo, hi = w.amin(-1).clamp(max=0), w.amax(-1)
    s, m = (hi - lo) / levels, -lo
    d = (s.amax(1) / steps).to(torch.float16).float()
    dm = (m.amax(1) / steps).to(torch.float16).float()
    sc = (s / d[:, None]).round().clamp(1, steps)
    mi = (m / dm[:, None]).round().clamp(0, steps)
    q = ((w + (dm[:, None] * mi)[..., None]) / (d[:, None] * sc)[..., None]).round().clamp(0, levels)
    return d, dm, sc.to(torch.uint8), mi.to(torch.uint8), q.to(torch.uint8)


def _q4_k(w):
    d, dm, sc, mi, q = _scale_min(w.view(-1, 8, 32), 15, 63)
    packed = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mi[:, :4] | ((mi[:, 4:] >> 4) << 6),
                        (sc[:, 4:] & 15) | ((mi[:, 4:] & 15) << 4)], 1)
    return torch.cat([_f16(d), _f16(dm), packed, _low(q.view(-1, 4, 2, 32)).reshape(-1, 128)], 1)


def _q2_k(w):
    d, dm, sc, mi, q = _scale_min(w.view(-1, 16, 16), 3, 15)
    q = q.view(-1, 2, 4, 32)                                   # half, shift, byte
    qs = q[:, :, 0] | (q[:, :, 1] << 2) | (q[:, :, 2] << 4) | (q[:, :, 3] << 6)
    return torch.cat([sc | (mi << 4), qs.reshape(-1, 64), _f16(d), _f16(dm)], 1)


def _q6_k(w):
    w = w.view(-1, 16, 16)
    s = w.abs().amax(2) / 32
    d = (s.amax(1) / 127).to(torch.float16).float()
    sc = (s / d[:, None]).round().clamp(1, 127)
    q = ((w / (d[:, None] * sc)[..., None]).round().clamp(-32, 31) + 32).to(torch.uint8).view(-1, 2, 4, 32)
    ql = torch.stack([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), _f16(d)], 1)


def _iq2_xxs(n, gen):
    """Blocks of random grid entries, signs and scales (the grid search of a quantizer is no part of this path)."""
    b = torch.randint(0, 256, (n, 8, 8), device=DEV, dtype=torch.uint8, generator=gen)
    b[:, :, 7] = (b[:, :, 7] & 15) | (torch.randint(6, 16, (n, 8), device=DEV, dtype=torch.uint8, generator=gen) << 4)
    d = 0.0003 * (0.6 + 0.8 * torch.rand(n, device=DEV, generator=gen))
    return torch.cat([_f16(d), b.view(n, 64)], 1)


QUANTIZE = {"Q8_0": _q8_0, "Q8_0R": _q8_0, "Q4_K": _q4_k, "Q6_K": _q6_k, "Q2_K": _q2_k}


def _half(b):
    return b.contiguous().view(torch.float16).double().squeeze(-1)


def _grid():
    with open(os.path.join(ROOT, "tests", "golden", "iq2xxs_grid.json")) as f:
        words = torch.tensor(json.load(f)["words"], dtype=torch.int64)
    return torch.stack([(words >> (8 * i)) & 255 for i in range(4)], 1).view(256, 8).double().to(DEV)


def _decode(t, b):
    """[blocks, bytes] -> [blocks, weights] in 64 bits."""
    if t in ("Q8_0", "Q8_0R"):
        return _half(b[:, :2])[:, None] * b[:, 2:].contiguous().view(torch.int8).double()
    if t == "Q4_K":
        d, dm, s = _half(b[:, :2]), _half(b[:, 2:4]), b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mi = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = b[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(-1, 8, 32)
        return ((d[:, None] * sc)[..., None] * q - (dm[:, None] * mi)[..., None]).view(-1, 256)
    if t == "Q2_K":
        s, q, d, dm = b[:, :16], b[:, 16:80].view(-1, 2, 1, 32), _half(b[:, 80:82]), _half(b[:, 82:])
        q = torch.cat([(q >> i) & 3 for i in (0, 2, 4, 6)], 2).view(-1, 16, 16)
        return ((d[:, None] * (s & 15))[..., None] * q - (dm[:, None] * (s >> 4))[..., None]).view(-1, 256)
    if t == "Q6_K":
        l, h = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 32)
        q = [(l[:, :, g & 1] >> (4 * (g >> 1))) & 15 | (((h >> (2 * g)) & 3) << 4) for g in range(4)]
        q = torch.stack(q, 2).view(-1, 16, 16).double() - 32
        return ((_half(b[:, 208:])[:, None] * b[:, 192:208].contiguous().view(torch.int8))[..., None] * q).view(-1, 256)
    g = b[:, 2:].view(-1, 8, 8).long()
    a1 = g[..., 4] | (g[..., 5] << 8) | (g[..., 6] << 16) | (g[..., 7] << 24)
    signs = torch.stack([(a1 >> (7 * i)) & 127 for i in range(4)], 2)
    bits = torch.stack([(signs >> i) & 1 for i in range(7)], 3)
    bits = torch.cat([bits, bits.sum(3, keepdim=True) & 1], 3)
    v = _grid()[g[..., :4]] * (1 - 2 * bits)
    return ((_half(b[:, :2])[:, None] * (2 * (a1 >> 28) + 1) / 8)[..., None, None] * v).view(-1, 256)


def _blocks(t, n, gen):
    """n blocks of type t, [n, bytes]."""
    if t == "IQ2_XXS":
        return _iq2_xxs(n, gen)
    e = BLOCK[t][0]
    parts = []
    for a in range(0, n, CHUNK // e):
        m = min(CHUNK // e, n - a)
        parts.append(QUANTIZE[t](0.02 * torch.randn(m * e, device=DEV, generator=gen)))
    return torch.cat(parts)


def _activations(tokens, k, gen):
    scale = torch.exp(0.5 * torch.randn(k, device=DEV, generator=gen))
    big = torch.rand(k, device=DEV, generator=gen) < 0.002
    return torch.randn(tokens, k, device=DEV, generator=gen) * torch.where(big, 10 * scale, scale)


def _shapes(case):
    """The (rows, k) of each matrix of the call."""
    r, k = case["rows"], case["k"]
    if case["op"] == "gate_up":
        return [(r, k)] * 2
    if case["op"] == "qkv":                       # four query heads to a key and value head
        return [(r, k), (max(r // 4, 1), k), (max(r // 4, 1), k)]
    return [(r, k)]


def _inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    e = BLOCK[case["type"]][0]
    w = [_blocks(case["type"], r * (k // e), gen) for r, k in _shapes(case)]
    if case["op"] == "embed":
        ids = torch.randint(0, case["rows"], (case["tokens"],), device=DEV, dtype=torch.int32, generator=gen)
        return w, ids, 1 + 0.1 * torch.randn(case["k"], device=DEV, generator=gen)
    return w, _activations(case["tokens"], case["k"], gen), None


# ---- the program's side ------------------------------------------------------

_program = {}


def _context():
    """The one context of the program, on a torch stream of its own."""
    if not _program:
        _program["stream"] = torch.cuda.Stream()
        _program["ctx"] = eff.Context(0)
        _program["ctx"].set_stream(_program["stream"].cuda_stream)
    return _program["ctx"]


class Tensor:
    """A torch tensor's memory as one of the library's buffers."""

    def __init__(self, ctx, n, dtype, shape):
        size = n * dtype.itemsize
        self.bytes = torch.empty(size + PAD, device=DEV, dtype=torch.uint8)
        self.view = self.bytes[:size].view(dtype).view(shape)
        h = eff.ctypes.c_void_p()
        ctx._check(eff.lib().eff_buf_wrap(ctx.h, self.bytes.data_ptr(), size, eff.ctypes.byref(h)))
        self.buf = eff.Buffer(ctx, h, size)
        weakref.finalize(self, eff.lib().eff_buf_free, ctx.h, h)   # gives the handle back; the memory is torch's

    @classmethod
    def of(cls, ctx, t):
        self = cls(ctx, t.numel(), t.dtype, t.shape)
        self.view.copy_(t)
        return self


def _weights(ctx, t, b):
    if t != "Q8_0R":
        return Tensor.of(ctx, b)
    n = b.shape[0]
    w = Tensor(ctx, eff.bytes_buffer_r(n), torch.uint8, (-1,))
    w.view.zero_()
    w.view[:32 * n] = b[:, 2:].reshape(-1)
    w.view[32 * n:34 * n] = b[:, :2].reshape(-1)
    w.buf.mark_r(n)
    return w


def prepare(case, seed):
    ctx = _context()
    op, t, tokens, k = case["op"], case["type"], case["tokens"], case["k"]
    w, x, norm = _inputs(case, seed)
    s = {"ctx": ctx, "op": op, "t": eff.type_code(t), "tokens": tokens, "k": k}
    s["w"] = [_weights(ctx, t, b) for b in w]
    s["x"] = Tensor.of(ctx, x)
    rows = [r for r, _ in _shapes(case)]
    s["rows"] = rows
    if op == "embed":
        s["norm"] = Tensor.of(ctx, norm)
        s["y"] = [Tensor(ctx, tokens * k, torch.float32, (tokens, k)) for _ in range(2)]
    else:
        outs = rows[:1] if op == "gate_up" else rows
        s["y"] = [Tensor(ctx, tokens * r, torch.float32, (tokens, r)) for r in outs]
    if op == "head":
        n = eff.lib().eff_topk_out_bytes() // 4
        s["top"] = Tensor(ctx, n, torch.int32, (n,))
    if op == "qkv":
        # x prepared once for each layout that the matrices' products read (none: the product reads x itself)
        s["layouts"], s["xp"] = [], {}
        for r in rows:
            try:
                n, lay = ctx.qmatmul_x_layout(s["t"], r, k, tokens)
            except eff.NotApplicable:
                n, lay = 0, 0
            s["layouts"].append(lay)
            if lay and lay not in s["xp"]:
                s["xp"][lay] = (r, Tensor(ctx, n, torch.uint8, (n,)))
    torch.cuda.synchronize()
    return s


def run(s):
    ctx, t, k, tokens, x = s["ctx"], s["t"], s["k"], s["tokens"], s["x"].buf
    if s["op"] == "matmul":
        ctx.qmatmul(t, s["w"][0].buf, x, s["y"][0].buf, s["rows"][0], k, tokens)
    elif s["op"] == "gate_up":
        ctx.qgemv_multi(t, eff.GEMV_SWIGLU, [w.buf for w in s["w"]], x, [y.buf for y in s["y"]], s["rows"], k, tokens)
    elif s["op"] == "head":
        ctx.qgemv_topk(t, s["w"][0].buf, x, s["y"][0].buf, s["rows"][0], k, 40, (), 1, s["top"].buf)
        top = s["top"].view
        pairs = top[TOPK_PAIRS:TOPK_PAIRS + 80].view(40, 2)
        return {"logits": s["y"][0].view, "head": top[:8], "ids": pairs[:, 0], "values": pairs[:, 1].view(torch.float32)}
    elif s["op"] == "embed":
        ctx.gather_norm(t, s["w"][0].buf, x, s["norm"].buf, EPS, s["y"][0].buf, s["y"][1].buf, k, tokens)
    else:
        for r, xp in s["xp"].values():
            ctx.qmatmul_prepare_x(t, x, xp.buf, r, k, tokens)
        for w, y, r, lay in zip(s["w"], s["y"], s["rows"], s["layouts"]):
            if lay:
                ctx.qmatmul_prepared(t, w.buf, s["xp"][lay][1].buf, y.buf, r, k, tokens)
            else:
                ctx.qmatmul(t, w.buf, x, y.buf, r, k, tokens)
    return [y.view for y in s["y"]]


def work(case):
    t, tokens, k = case["type"], case["tokens"], case["k"]
    e, b = BLOCK[t]
    if case["op"] == "embed":
        return {"bytes": tokens * (k // e * b + 4 + 8 * k) + 4 * k, "flops": 4.0 * tokens * k}
    weights = sum(r * k for r, k in _shapes(case))
    outs = case["rows"] if case["op"] == "gate_up" else sum(r for r, _ in _shapes(case))
    return {"bytes": weights // e * b + 4 * tokens * (k + outs), "flops": 2.0 * weights * tokens}


def tolerance(case):
    if case["op"] == "embed":
        return {"rel": 1e-6, "max": 1e-5}          # 32-bit decode and norm
    if case["type"] in ("Q8_0", "Q8_0R") and case["op"] in ("matmul", "qkv") and case["tokens"] >= 64:
        return {"rel": 1e-3, "max": 1e-2}          # operands rounded to fp16
    if case["op"] == "gate_up":
        return {"rel": 1e-5, "max": 4e-4}          # silu(g) u of two 32-bit sums, read against the rms of the product
    return {"rel": 1e-5, "max": 1e-4}              # 32-bit sums of x kept to 22 bits


def _product(t, b, rows, k, x):
    """x W' in 64 bits, W decoded a run of rows at a time."""
    y = torch.empty(x.shape[0], rows, device=DEV, dtype=torch.float64)
    b = b.view(rows, -1)
    step = max(1, CHUNK // k)
    for a in range(0, rows, step):
        n = min(step, rows - a)
        w = _decode(t, b[a:a + n].reshape(-1, BLOCK[t][1])).view(n, k)
        y[:, a:a + n] = x @ w.t()
    return y


def exact(case, seed):
    w, x, norm = _inputs(case, seed)
    t, k = case["type"], case["k"]
    if case["op"] == "embed":
        v = _decode(t, w[0].view(case["rows"], -1)[x.long()].reshape(-1, BLOCK[t][1])).view(-1, k)
        return [v, v / torch.sqrt(v.square().mean(1, keepdim=True) + EPS) * norm.double()]
    y = [_product(t, b, r, k, x.double()) for b, (r, k) in zip(w, _shapes(case))]
    if case["op"] == "gate_up":
        return [y[0] * torch.sigmoid(y[0]) * y[1]]
    if case["op"] == "head":
        return {"logits": y[0], "head": None, "ids": None, "values": y[0][0].topk(40).values}
    return y
