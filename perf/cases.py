"""The work a program has this library do, case by case, for timing it.

A serving program's day is layer calls: one token at a time for one user, one
token for each of a batch of users (few or many, contiguous caches or a paged
pool, contexts of unequal length), and prompts (whole, or a chunk after cached
positions).  Programs that schedule the stages themselves call the attention
and the FFN's stages through the same C ABI.  Weights are N(0, 0.02)
quantized to Q4_0, activations and cache rows N(0, 1), norm gains N(1, 0.1),
biases N(0, 0.02).  Everything is made from the seed, on the GPU.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "simple-inference_amd"))
import si_amd  # noqa: E402

DEV = "cuda"
QK = 32


def listed():
    return [
        # one user's next token: the smallest layer, latency and launches
        dict(name="decode_small", op="decode", model="0.5b", context=1024),
        # the attention sublayer alone, the contract of run_layer at the
        # reference's own shape, at a context that fills no tile
        dict(name="decode_sublayer", op="decode", model="1.5b_ref", context=333),
        # one user's next token on a large layer with a long context
        dict(name="decode_large", op="decode", model="7b", context=4096),
        # a quiet server: five users at different points of their chats
        dict(name="batch_few", op="batch", model="7b", rows=5, low=40, high=1500, page=0),
        # a busy server on a small model with a paged cache
        dict(name="batch_paged", op="batch", model="0.5b", rows=24, low=100, high=2048, page=16),
        # a busy server on a large model, every context long
        dict(name="batch_full", op="batch", model="7b", rows=64, low=4096, high=4096, page=0),
        # a whole prompt on a small layer
        dict(name="prefill_small", op="prefill", model="0.5b", rows=512, prefix=0),
        # the next piece of a prompt that is taken in pieces
        dict(name="prefill_chunk", op="prefill", model="7b", rows=333, prefix=1500),
        # a whole prompt on a large layer
        dict(name="prefill_large", op="prefill", model="7b", rows=2048, prefix=0),
        # the attention stage alone, one query for each of 48 users
        dict(name="attention_ragged", op="attention", model="7b", rows=48, low=200, high=4096),
        # the attention stage alone over a long prompt
        dict(name="attention_long", op="attention_prompt", model="1.5b_ref", rows=5000, prefix=0),
        # the FFN's stages, one call each
        dict(name="ffn_stages", op="ffn", model="0.5b", rows=777),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["decode", "batch", "batch", "prefill", "prefill", "attention",
                     "attention_prompt", "ffn"])
    model = rng.choice(["0.5b", "0.5b", "7b", "7b", "1.5b_ref"])
    if op == "decode":
        return dict(op=op, model=model, context=_log(rng, 16, 4096))
    if op in ("batch", "attention"):
        high = _log(rng, 64, 4096)
        c = dict(op=op, model=model, rows=_log(rng, 2, 64), low=rng.randint(1, high), high=high)
        if op == "batch":
            c["page"] = rng.choice([0, 0, 16, 64])
        return c
    if op == "prefill":
        rows = _log(rng, 2, 1600 if model == "7b" else 4000)
        return dict(op=op, model=model, rows=rows, prefix=rng.choice([0, 0, _log(rng, 16, 2000)]))
    if op == "attention_prompt":
        return dict(op=op, model=model, rows=_log(rng, 16, 2500 if model == "7b" else 5000),
                    prefix=rng.choice([0, 0, _log(rng, 16, 2000)]))
    model = "0.5b" if model == "1.5b_ref" else model
    return dict(op=op, model=model, rows=_log(rng, 2, 1600 if model == "7b" else 4000))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Inputs:
    """Seeded tensors on the GPU, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 17)

    def normal(self, *shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=self.g, device=DEV).mul_(std).add_(mean)

    def half(self, *shape):
        return torch.randn(shape, generator=self.g, device=DEV, dtype=torch.float16)

    def contexts(self, n, low, high):
        """n contexts in low..high, one of them the longest."""
        c = torch.randint(low, high + 1, (n,), generator=self.g, device=DEV, dtype=torch.int32)
        c[n // 2] = high
        return c

    def pages(self, n, each):
        return torch.randperm(n * each, generator=self.g, device=DEV).to(torch.int32).view(n, each)

    def q4(self, n, k):
        """Row-major Q4_0 blocks of N(0, 0.02) weights: uint8 [n][k/32][18], fp16 scale =
        (value of largest magnitude) / -8, then 16 bytes of nibbles j | j + 16 << 4."""
        w = self.normal(n, k // QK, QK, std=0.02)
        top = w.gather(2, w.abs().argmax(2, keepdim=True)) / -8
        q = (w / top + 8.5).floor_().clamp_(0, 15).to(torch.uint8)
        out = torch.empty(n, k // QK, 18, dtype=torch.uint8, device=DEV)
        out[..., :2] = top.to(torch.float16).view(torch.uint8)
        out[..., 2:] = q[..., :16] | q[..., 16:] << 4
        return out


def _dims(model):
    d = si_amd.SHAPES[model]
    return d["hidden"], d["qheads"], d["kvheads"], d["hdim"], d["ffn"]


def _weights(r, model):
    h, q, kv, d, f = _dims(model)
    t = dict(wq=r.q4(q * d, h), wk=r.q4(kv * d, h), wv=r.q4(kv * d, h), wo=r.q4(h, q * d),
             norm=r.normal(h, mean=1.0, std=0.1), bq=r.normal(q * d, std=0.02),
             bk=r.normal(kv * d, std=0.02), bv=r.normal(kv * d, std=0.02))
    if f:
        t.update(post_norm=r.normal(h, mean=1.0, std=0.1), wgate=r.q4(f, h), wup=r.q4(f, h),
                 wdown=r.q4(h, f))
    return t


def _flags(model):
    return si_amd.SI_LAYER_FULL if _dims(model)[4] else si_amd.SI_LAYER_ATTN_ONLY


def _inputs(case, seed):
    """(weights or None, the call's tensors) of a case, the same for every implementation."""
    r = _Inputs(seed)
    op, model = case["op"], case["model"]
    h, q, kv, d, f = _dims(model)
    if op == "ffn":
        t = dict(gate_up=r.q4(2 * f, h), down=r.q4(h, f), gain=r.normal(h, mean=1.0, std=0.1))
        return t, dict(x=r.normal(case["rows"], h), y=r.normal(case["rows"], h, std=0.5))
    w = None if op.startswith("attention") else _weights(r, model)
    if op == "decode":
        n = case["context"]
        return w, dict(x=r.normal(h), k=r.half(n, kv * d), v=r.half(n, kv * d))
    if op in ("prefill", "attention_prompt"):
        n = case["prefix"] + case["rows"]
        c = dict(k=r.half(n, kv * d), v=r.half(n, kv * d))
        c["x" if w else "q"] = r.normal(case["rows"], h if w else q * d)
        return w, c
    n, high, page = case["rows"], case["high"], case.get("page", 0)
    c = dict(ctx=r.contexts(n, case["low"], high))
    c["x" if w else "q"] = r.normal(n, h if w else q * d)
    if page:
        c["pages"] = r.pages(n, (high + page - 1) // page)
        c["k"], c["v"] = (r.half(c["pages"].numel() * page, kv * d) for _ in range(2))
    else:
        c["k"], c["v"] = (r.half(n, high, kv * d) for _ in range(2))
    return w, c


class _State:
    pass


def _device_q4(w):
    """A matrix in the device layout, as a program that calls the stages keeps it."""
    n, nb, _ = w.shape
    k, tile = nb * QK, si_amd.lib().si_q4_tile(n, nb * QK)
    m = _State()
    m.n, m.k, m.tile = n, k, tile
    m.qs = torch.empty(n * k // 2, dtype=torch.uint8, device=DEV)
    m.d = torch.zeros(si_amd.lib().si_q4_scale_count(n, k, tile), dtype=torch.int16, device=DEV)
    si_amd.call("si_q4_repack", si_amd.ptr(w), n, k, tile, si_amd.ptr(m.qs), si_amd.ptr(m.d),
                si_amd.stream_handle())
    return m


def _q8(rows, k):
    """Planar Q8_0 buffers (values, fp16 scales)."""
    return (torch.empty(rows, k, dtype=torch.int8, device=DEV),
            torch.empty(rows, k // QK, dtype=torch.float16, device=DEV))


def prepare(case, seed):
    w, c = _inputs(case, seed)
    s = _State()
    s.case, s.c = case, c
    s.shape = si_amd.make_shape(**si_amd.SHAPES[case["model"]])
    h, q, kv, d, f = _dims(case["model"])
    op, rows = case["op"], case.get("rows", 1)
    if op == "ffn":
        s.gu, s.down, s.gain = _device_q4(w["gate_up"]), _device_q4(w["down"]), w["gain"]
        s.h, s.out = (torch.empty(rows, h, device=DEV) for _ in range(2))
        s.xq, s.aq = _q8(rows, h), _q8(rows, f)
        lib = si_amd.lib()
        s.ws_bytes = max(lib.si_gemm_workspace(rows, 2 * f, h), lib.si_gemm_workspace(rows, h, f))
        s.ws = torch.empty(max(s.ws_bytes, 256), dtype=torch.uint8, device=DEV)
    elif op.startswith("attention"):
        s.max_ctx = case["high"] if op == "attention" else case["prefix"] + rows
        s.out = torch.empty(rows, q * d, device=DEV)
        s.oq = _q8(rows, q * d)
        s.ws_bytes = si_amd.lib().si_attention_workspace(ctypes.byref(s.shape), rows, s.max_ctx)
        s.ws = torch.empty(max(s.ws_bytes, 256), dtype=torch.uint8, device=DEV)
    else:
        host = {name: t.cpu().numpy() for name, t in w.items()}
        longest = case.get("context") or case.get("high") or case["prefix"] + rows
        s.layer = si_amd.Layer(s.shape, host, 1 << (rows - 1).bit_length(), longest)
        s.layer._keep = None  # the layer has its own copy on the device
        s.out = torch.empty(rows, h, device=DEV)
        s.flags = _flags(case["model"])
    torch.cuda.synchronize()
    return s


def run(s):
    case, c, op = s.case, s.c, s.case["op"]
    p = si_amd.ptr
    if op == "decode":
        s.layer.decode(c["x"], c["k"], c["v"], case["context"], s.out, flags=s.flags,
                       capture=False)
    elif op == "prefill":
        s.layer.prefill(c["x"], case["rows"], case["prefix"], c["k"], c["v"], s.out,
                        flags=s.flags, capture=False)
    elif op == "batch" and case["page"]:
        s.layer.decode_paged(c["x"], case["rows"], c["k"], c["v"], c["pages"].numel(),
                             case["page"], c["pages"], c["pages"].shape[1], c["ctx"],
                             case["high"], s.out, flags=s.flags, capture=False)
    elif op == "batch":
        s.layer.decode_batch(c["x"], case["rows"], c["k"], c["v"], c["k"].stride(0),
                             case["high"], case["high"], s.out, ctx_dev=c["ctx"], flags=s.flags,
                             capture=False)
    elif op == "attention":
        si_amd.call("si_attention", ctypes.byref(s.shape), p(c["q"]), case["rows"], p(c["k"]),
                    p(c["v"]), c["k"].stride(0), p(c["ctx"]), 0, 0, s.max_ctx, p(s.out),
                    p(s.oq[0]), p(s.oq[1]), None, p(s.ws), s.ws_bytes, si_amd.stream_handle())
    elif op == "attention_prompt":
        si_amd.call("si_attention", ctypes.byref(s.shape), p(c["q"]), case["rows"], p(c["k"]),
                    p(c["v"]), 0, None, case["prefix"] + 1, 1, s.max_ctx, p(s.out), p(s.oq[0]),
                    p(s.oq[1]), None, p(s.ws), s.ws_bytes, si_amd.stream_handle())
    else:
        st, m, gu, dn = si_amd.stream_handle(), case["rows"], s.gu, s.down
        si_amd.call("si_residual_rmsnorm_q8", p(c["x"]), p(c["y"]), p(s.gain), m, gu.k,
                    s.shape.rms_eps, p(s.h), None, p(s.xq[0]), p(s.xq[1]), None, st)
        si_amd.call("si_gemm_gateup_q8", p(gu.qs), p(gu.d), gu.tile, dn.k, gu.k, p(s.xq[0]),
                    p(s.xq[1]), m, None, None, p(s.aq[0]), p(s.aq[1]), None, 0, p(s.ws),
                    s.ws_bytes, st)
        si_amd.call("si_gemm_q4q8", p(dn.qs), p(dn.d), dn.tile, dn.n, dn.k, p(s.aq[0]),
                    p(s.aq[1]), m, None, p(s.h), p(s.out), dn.n, 0, p(s.ws), s.ws_bytes, st)
        return dict(h=s.h, xq=s.xq[0], xd=s.xq[1], aq=s.aq[0], ad=s.aq[1], out=s.out)
    if op.startswith("attention"):
        return dict(out=s.out, q8=s.oq[0], d=s.oq[1])
    return dict(out=s.out, k=c["k"], v=c["v"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Every weight, activation and live cache row read once, every output written once; 2 m n k
    per product, 4 hdim per (query head, visible position)."""
    h, q, kv, d, f = _dims(case["model"])
    op, m = case["op"], case.get("rows", 1)
    qd, kvd = q * d, kv * d
    full = f if op != "ffn" else 0
    weights = 0 if op.startswith("attention") else (qd + 2 * kvd) * h + h * qd + 3 * h * full
    if op == "ffn":
        weights = 3 * h * f
    if op in ("batch", "attention"):
        seen = m * (case["low"] + case["high"]) / 2  # positions, over the queries
        rows = seen  # cache rows read
    elif op == "ffn":
        seen = rows = 0
    else:
        first = case.get("context", 1) - 1 if op == "decode" else case["prefix"]
        seen = m * first + m * (m + 1) / 2
        rows = first + m
    cache = 4 * rows * kvd  # fp16 K and V
    if op == "ffn":
        acts = 4 * 4 * m * h + (h + f) * m * 34 / 32
    elif op.startswith("attention"):
        acts = m * qd * (4 + 4 + 34 / 32)
    else:
        acts = 2 * 4 * m * h + 4 * m * kvd
    return dict(bytes=weights * 18 / 32 + cache + acts, flops=2.0 * m * weights + 4.0 * seen * qd)


def tolerance(case):
    """About four times what the kernels, the exact-rounding kernels and 64 bits show between them.
    A stage alone differs by its sums and by the fp16 steps of its Q8_0 scales.  A layer rounds to
    Q8_0 three times inside, and each rounding turns a last bit into a step of 1/127 now and then:
    one step moves a small layer's output by 5e-4 (largest value 1.6e-2 over 2000 rows), and a
    large layer carries it on to 5e-3 (3.4e-2)."""
    if case["op"] == "ffn":
        return dict(rel=3e-4, max=1.5e-2, differ=2e-4)
    if case["op"].startswith("attention"):
        return dict(rel=5e-5, max=4e-3, differ=1e-4)
    return dict(rel=2e-2, max=0.14) if case["model"] == "7b" else dict(rel=3e-3, max=6e-2)


# ---------------------------------------------------------------------------
# the same in 64 bits, with the formats' own roundings (Q8_0 blocks, fp16
# scales and cache rows), which are part of what the path computes
# ---------------------------------------------------------------------------
def _w64(w):
    d = w[..., :2].contiguous().view(torch.float16).double()
    nib = torch.cat([w[..., 2:] & 15, w[..., 2:] >> 4], dim=2).double() - 8
    return (nib * d).view(w.shape[0], -1)


def _quantize64(x):
    """(scales before their rounding to fp16, the values that the blocks stand for) of Q8_0."""
    b = x.view(x.shape[0], -1, QK)
    d = b.abs().amax(2, keepdim=True) / 127
    v = torch.where(d > 0, b / d, torch.zeros_like(b)).round_()
    return d.squeeze(2), (v * d.to(torch.float16).double()).view_as(x)


def _project64(x, w, b=None):
    """Q8_0 rows times Q4_0 weights, the weights widened a few rows at a time."""
    xq = _quantize64(x)[1]
    y = torch.cat([xq @ _w64(p).T for p in w.split(8192)], dim=1)
    return y if b is None else y + b.double()


def _norm64(x, gain):
    return x / (x.square().mean(1, keepdim=True) + 1e-6).sqrt() * gain.double()


def _rope64(x, pos, heads, hdim):
    i = torch.arange(hdim // 2, device=DEV, dtype=torch.float64)
    # the angle is a binary32 number by the path's definition
    a = (pos.float()[:, None] / torch.pow(torch.tensor(1e6, device=DEV), (2 * i / hdim).float()))
    c, s = a.double().cos()[:, None], a.double().sin()[:, None]
    x = x.view(-1, heads, hdim)
    lo, hi = x[..., :hdim // 2], x[..., hdim // 2:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], 2).reshape(x.shape[0], -1)


def _attend64(q, k, v, heads, kvheads, first):
    """Rows of q at positions first, first + 1, ... over cache rows 0..position."""
    n, hdim = q.shape[0], q.shape[1] // heads
    k, v = (t[:first + n].double().view(first + n, kvheads, hdim) for t in (k, v))
    q, out = q.view(n, heads, hdim), torch.empty(n, heads, hdim, device=DEV, dtype=torch.float64)
    hidden = torch.ones(n, first + n, dtype=torch.bool, device=DEV).triu_(first + 1)
    for hq in range(heads):
        g = hq // (heads // kvheads)
        p = (q[:, hq] @ k[:, g].T.contiguous()) / math.sqrt(hdim)
        out[:, hq] = p.masked_fill_(hidden, -math.inf).softmax(1) @ v[:, g]
    return out.view(n, heads * hdim)


def _cache_rows(case, c, i):
    """Pool or cache rows of sequence i, in position order."""
    if not case.get("page"):
        return c["k"][i], c["v"][i], None
    at = (c["pages"][i].long()[:, None] * case["page"] +
          torch.arange(case["page"], device=DEV)).view(-1)
    return c["k"][at], c["v"][at], at


def _each_sequence(case, c, q, heads, kvheads):
    ctx = c["ctx"].tolist()
    rows = []
    for i, n in enumerate(ctx):
        k, v, _ = _cache_rows(case, c, i)
        rows.append(_attend64(q[i:i + 1], k, v, heads, kvheads, n - 1))
    return torch.cat(rows)


def _many(case):
    """Whether a result behind an inner Q8_0 rounding has a 64-bit value to be held against: a
    value next to a tie goes either way in any arithmetic, and moves the result by hundreds of
    times its own error, so over few rows the distance is the luck of a few ties (0 in one seed,
    5e-4 in the next); over many it is their steady share."""
    return case.get("rows", 1) >= (32 if case["model"] == "7b" else 512)


def exact(case, seed):
    w, c = _inputs(case, seed)
    op, rows = case["op"], case.get("rows", 1)
    h, q, kv, d, f = _dims(case["model"])
    if op == "ffn":
        hid = c["x"].double() + c["y"].double()
        n = _norm64(hid, w["gain"])
        act = _swiglu64(n, w["gate_up"][:f], w["gate_up"][f:])
        out = hid + _project64(act, w["down"]) if _many(case) else None
        return dict(h=hid, xq=None, xd=_quantize64(n)[0], aq=None, ad=_quantize64(act)[0], out=out)
    if op.startswith("attention"):
        qq = c["q"].double()
        a = (_each_sequence(case, c, qq, q, kv) if op == "attention"
             else _attend64(qq, c["k"], c["v"], q, kv, case["prefix"]))
        return dict(out=a, q8=None, d=_quantize64(a)[0])
    x = c["x"].double().view(rows, h)
    n1 = _norm64(x, w["norm"])
    qr, kr, vr = (_project64(n1, w["w" + t], w["b" + t]) for t in "qkv")
    if op == "batch":
        pos = c["ctx"].long() - 1
    else:
        first = case["context"] - 1 if op == "decode" else case["prefix"]
        pos = torch.arange(first, first + rows, device=DEV)
    qr, kr = _rope64(qr, pos, q, d), _rope64(kr, pos, kv, d)
    kc, vc = c["k"].double(), c["v"].double()  # the new rows before their rounding to fp16
    if op == "batch":
        page = case["page"]
        for i, p in enumerate(pos.tolist()):
            at = (c["pages"][i, p // page].long() * page + p % page,) if page else (i, p)
            kc[at], vc[at] = kr[i], vr[i]
        a = _each_sequence(case, dict(c, k=kc.half(), v=vc.half()), qr, q, kv)
    else:
        kc[first:first + rows], vc[first:first + rows] = kr, vr
        a = _attend64(qr, kc.half(), vc.half(), q, kv, first)
    o = _project64(a, w["wo"])
    if f:
        x = x + o
        o = x + _project64(_swiglu64(_norm64(x, w["post_norm"]), w["wgate"], w["wup"]), w["wdown"])
    return dict(out=o if _many(case) else None, k=kc, v=vc)


def _swiglu64(x, gate, up):
    g = _project64(x, gate)
    return g * torch.sigmoid(g) * _project64(x, up)
