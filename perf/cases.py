"""The work that users of u15h have it do, as cases that can be timed and
compared: the dense and quantized projections at text and image row counts,
the projection steps of a layer, SwiGLU, the int8 tier, attention over the
K/V cache, and whole decoder layers, each through `u15h.Ops`.

Widths are the model's: hidden 4096, 32 query heads over 8 K/V heads of 128,
MLP 12288 (q, o: 4096 x 4096; k, v: 1024 x 4096; gate, up: 12288 x 4096;
down: 4096 x 12288).  Weights are ~N(0, 0.02), activations ~N(0, 1).
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "vpipe-sensenova-u1.5_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import u15h  # noqa: E402

HIDDEN, HEADS, KV_HEADS, HEAD_DIM, INTER = 4096, 32, 8, 128, 12288
QDIM, KVDIM = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
D_T, D_H = 64, 32
EPS = 1e-6
BF16, F64 = torch.bfloat16, torch.float64

_OPS = None


def _ops():
    """The program's one context."""
    global _OPS
    if _OPS is None:
        _OPS = u15h.Ops(0)
    return _OPS


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one token through k_proj: the smallest call, launch and latency
        dict(name="linear_m1", kind="linear", M=1, K=4096, N=1024, bias=False),
        # a ragged batch of text rows through gate_proj, between the
        # weight-bound and the matrix-bound regimes
        dict(name="linear_m333_bias", kind="linear", M=333, K=4096, N=12288, bias=True),
        # a few tokens over a 4-bit checkpoint's up_proj
        dict(name="pack_w4_m4", kind="pack", M=4, K=4096, N=12288, bits=4, group=32, bias=False),
        # a prompt of ~300 tokens over an 8-bit checkpoint's q|k|v widths
        dict(name="pack_w8_m300", kind="pack", M=300, K=4096, N=6144, bits=8, group=64,
             bias=True),
        # the projections of one layer for a 1024x1024 image and its prompt
        # (the benchmark's step)
        dict(name="steps_128_4096", kind="steps", M_und=128, M_gen=4096),
        # gate|up with SwiGLU for a 512x512 image and its prompt
        dict(name="swiglu_128_1024", kind="swiglu", M_und=128, M_gen=1024),
        # the int8 tier's down projection, quantising its input
        dict(name="i8_down_128_4096", kind="i8", M_und=128, M_gen=4096, K=12288, N=4096),
        # the generation pass: an image's queries over prompt and image
        dict(name="attn_gen_4096", kind="attn", tq=4096, tk=4224, q_offset=128, mode=0,
             hq=32, hkv=8, d=128),
        # a line of text after two cached reference images
        dict(name="attn_text_41", kind="attn", tq=41, tk=2345, q_offset=2304, mode=1,
             hq=32, hkv=8, d=128),
        # one token through four whole layers, 1500 tokens in the cache
        dict(name="layers_decode", kind="layer", layers=4, M_und=1, M_gen=0, kv_off=1500,
             mode=1, i8=False),
        # an edit prompt's prefill: text around a 16x16 image block
        dict(name="layer_prefill_333", kind="layer", layers=1, M_und=333, M_gen=0, kv_off=0,
             mode=2, i8=False),
        # a text prompt's prefill in the int8 tier
        dict(name="layer_i8_77", kind="layer", layers=1, M_und=77, M_gen=0, kv_off=0,
             mode=1, i8=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _image_tokens(rng, most):
    """Tokens of an image of 16-pixel patches merged 2x2 or not: h x w."""
    h = rng.randint(12, 64)
    return h * max(12, min(rng.randint(12, 64), most // h))


def draw(rng):
    kind = rng.choice(["linear", "pack", "steps", "swiglu", "i8", "attn", "attn", "layer",
                       "layer"])
    widths = [(4096, 4096), (4096, 1024), (4096, 6144), (4096, 12288), (12288, 4096)]
    if kind == "linear":
        K, N = rng.choice(widths)
        if rng.random() < 0.3:                      # any width the entry point takes
            K, N = 8 * rng.randint(32, 1024), 8 * rng.randint(16, 1024)
        return dict(kind=kind, M=_log_int(rng, 1, 2048), K=K, N=N, bias=rng.random() < 0.5)
    if kind == "pack":
        K, N = rng.choice(widths)
        return dict(kind=kind, M=_log_int(rng, 1, 1024), K=K, N=N, bits=rng.choice([4, 8]),
                    group=rng.choice([32, 64]), bias=rng.random() < 0.5)
    if kind in ("steps", "swiglu", "i8"):
        what = rng.choice(["prompt", "image", "both"])
        mu = 0 if what == "image" else _log_int(rng, 1, 512)
        mg = 0 if what == "prompt" else _image_tokens(rng, 4096 - 512)
        c = dict(kind=kind, M_und=mu, M_gen=mg)
        if kind == "i8":
            c["K"], c["N"] = rng.choice(widths)
        return c
    if kind == "attn":
        d, hq, hkv = rng.choice([(128, 32, 8)] * 4 + [(64, 16, 4), (32, 8, 8)])
        mode = rng.choice([0, 1, 2])
        off = rng.choice([0, rng.randint(1, 256), rng.randint(256, 3000)])
        tq = _log_int(rng, 1, 4096)
        return dict(kind=kind, tq=tq, tk=off + tq, q_offset=off, mode=mode, hq=hq, hkv=hkv, d=d)
    i8 = rng.random() < 0.4
    what = rng.choice(["decode", "prompt", "image", "both"])
    layers = rng.randint(1, 3) if what == "decode" and not i8 else 1
    mu = {"decode": rng.randint(1, 8), "prompt": _log_int(rng, 9, 1024), "image": 0,
          "both": _log_int(rng, 4, 256)}[what]
    mg = _image_tokens(rng, 2048) if what in ("image", "both") else 0
    off = rng.randint(1, 3000) if what == "decode" else rng.choice([0, rng.randint(1, 600)])
    mode = {"decode": 1, "prompt": rng.choice([1, 2]), "image": 0, "both": 2}[what]
    return dict(kind="layer", layers=layers, M_und=mu, M_gen=mg, kv_off=off, mode=mode, i8=i8)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

class _Rand:
    """Seeded values on the GPU, the same for prepare() and exact()."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def bf16(self, *shape, std=1.0, mean=0.0):
        t = torch.empty(*shape, dtype=BF16, device="cuda").normal_(mean, std, generator=self.g)
        return t

    def weight(self, n, k):
        return self.bf16(n, k, std=0.02)

    def norm(self, n):
        return self.bf16(n, std=0.1, mean=1.0)


def _quant_rows(x):
    """Per-row symmetric int8: s = absmax / 127, q = round half away (x / s)."""
    s = x.float().abs().amax(1) / 127.0
    r = x.float() / torch.where(s > 0, s, torch.ones_like(s))[:, None]
    q = torch.sign(r) * torch.floor(r.abs() + 0.5)
    return q.clamp(-127, 127).to(torch.int8), s


def _pack(r, n, k, bits, group):
    """An affine pack as quantized checkpoints hold it: u32 codes (low bits
    first), bf16 scale and bias per group."""
    top = (1 << bits) - 1
    codes = torch.randint(0, top + 1, (n, k), generator=r.g, device="cuda", dtype=torch.int32)
    scale = (torch.rand(n, k // group, generator=r.g, device="cuda") + 0.5) * (0.08 / top)
    bias = -scale * (top / 2)
    per = 32 // bits
    words = torch.zeros(n, k // per, dtype=torch.int64, device="cuda")
    for i in range(per):
        words |= codes[:, i::per].long() << (bits * i)
    words = torch.where(words >= 1 << 31, words - (1 << 32), words).to(torch.int32)
    return codes, words.contiguous(), scale.to(BF16), bias.to(BF16)


def _positions(case):
    """(t, h, w) positions and the t index over the whole cache of a pass:
    text counts up in t; an image's tokens share one t and count rows and
    columns.  A prompt in block-causal mode holds one image block."""
    M, off = case["M_und"] + case["M_gen"], case["kv_off"]
    pos = torch.zeros(3, M, dtype=torch.int64)
    t_all = torch.arange(off + M)
    image = case["M_gen"]
    start = M - image
    if image == 0 and case["mode"] == 2 and M >= 24:
        image = min(256, M // 2)
        start = (M - image) // 2
    pos[0] = t_all[off:]
    if image:
        side = max(1, math.isqrt(image))
        i = torch.arange(image)
        pos[0, start:start + image] = off + start
        pos[1, start:start + image] = i // side
        pos[2, start:start + image] = i % side
        t_all[off + start:off + start + image] = off + start
        if start + image < M:                       # the text after the image
            n = M - start - image
            pos[0, start + image:] = off + start + 1 + torch.arange(n)
            t_all[off + start + image:] = pos[0, start + image:]
    return pos.int(), t_all.int()


_PROJ = ((QDIM, HIDDEN), (KVDIM, HIDDEN), (KVDIM, HIDDEN), (HIDDEN, QDIM), (INTER, HIDDEN),
         (INTER, HIDDEN), (HIDDEN, INTER))
_NORM = (HIDDEN, HIDDEN, HEAD_DIM // 2, HEAD_DIM // 2, HEAD_DIM // 2, HEAD_DIM // 2)


def _experts(case):
    return [e for e, n in ((u15h.UND, case["M_und"]), (u15h.GEN, case["M_gen"])) if n]


def _layer_tensors(case, r):
    """Weights, norms, caches and hidden states of a whole-layer case."""
    W, G = {}, {}
    for l in range(case["layers"]):
        for e in _experts(case):
            for p, (n, k) in enumerate(_PROJ):
                W[l, e, p] = r.weight(n, k)
            for i, n in enumerate(_NORM):
                G[l, e, i] = r.norm(n)
    M = case["M_und"] + case["M_gen"]
    cap = (case["kv_off"] + M + 63) // 64 * 64
    kc, vc = [], []
    for _ in range(case["layers"]):
        for c in (kc, vc):
            t = torch.zeros(KV_HEADS, cap, HEAD_DIM, dtype=BF16, device="cuda")
            t[:, :case["kv_off"]] = r.bf16(KV_HEADS, case["kv_off"], HEAD_DIM)
            c.append(t)
    return W, G, kc, vc, r.bf16(M, HIDDEN)


def _rows(case):
    return case["M_und"], case["M_gen"], case["M_und"] + case["M_gen"]


def prepare(case, seed):
    r, kind = _Rand(seed), case["kind"]
    s = dict(case=case, ops=_ops())
    if kind == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        s.update(x=r.bf16(M, K), w=r.weight(N, K), b=r.bf16(N) if case["bias"] else None,
                 y=torch.empty(M, N, dtype=BF16, device="cuda"))
    elif kind == "pack":
        M, K, N = case["M"], case["K"], case["N"]
        _, words, sc, bi = _pack(r, N, K, case["bits"], case["group"])
        s.update(qw=(words, sc, bi, case["bits"], case["group"]), x=r.bf16(M, K),
                 b=r.bf16(N) if case["bias"] else None,
                 y=torch.empty(M, N, dtype=BF16, device="cuda"))
    elif kind == "steps":
        mu, mg, M = _rows(case)
        stack = u15h.Stack(1)
        for e in _experts(case):
            for p, (n, k) in enumerate(_PROJ):
                stack.bind(u15h.slot_name(0, e, p), r.weight(n, k))
        io = dict(x=r.bf16(M, HIDDEN), attn=r.bf16(M, QDIM), x2=r.bf16(M, HIDDEN),
                  h=r.bf16(M, INTER))
        for name, n in (("q", QDIM), ("k", KVDIM), ("v", KVDIM), ("o", HIDDEN),
                        ("gate", INTER), ("up", INTER), ("down", HIDDEN)):
            io[name] = torch.empty(M, n, dtype=BF16, device="cuda")
        s.update(stack=stack, bufs=io, io=u15h.layer_io(**io))
    elif kind == "swiglu":
        mu, mg, M = _rows(case)
        w = {}
        for e in _experts(case):
            w[e] = (r.weight(INTER, HIDDEN), r.weight(INTER, HIDDEN))
        s.update(x=r.bf16(M, HIDDEN), w=w, h=torch.empty(M, INTER, dtype=BF16, device="cuda"))
    elif kind == "i8":
        mu, mg, M = _rows(case)
        K, N = case["K"], case["N"]
        proj = dict(y=torch.empty(M, N, dtype=BF16, device="cuda"))
        for e in _experts(case):
            tag = "gen" if e == u15h.GEN else "und"
            proj["wq_" + tag], proj["sw_" + tag] = _quant_rows(r.weight(N, K))
        s.update(x=r.bf16(M, K), xq=torch.empty(M, K, dtype=torch.int8, device="cuda"),
                 sx=torch.empty(M, dtype=torch.float32, device="cuda"), proj=proj)
    elif kind == "attn":
        cap = (case["tk"] + 63) // 64 * 64
        s.update(q=r.bf16(case["tq"], case["hq"] * case["d"]),
                 k=r.bf16(case["hkv"], cap, case["d"]), v=r.bf16(case["hkv"], cap, case["d"]))
        s["out"] = torch.empty_like(s["q"])
        s["t"] = _attn_t(case).cuda() if case["mode"] == 2 else None
    else:
        W, G, kc, vc, x = _layer_tensors(case, r)
        stack = u15h.Stack(case["layers"])
        tier = u15h.TIER_I8 if case["i8"] else u15h.TIER_BF16
        for (l, e, p), w in W.items():
            if case["i8"]:
                stack.bind_i8(u15h.slot_name(l, e, p), *_quant_rows(w))
            else:
                stack.bind(u15h.slot_name(l, e, p), w)
        for (l, e, i), g in G.items():
            stack.bind_norm(u15h.norm_slot_name(l, e, i), g)
        pos, t_all = _positions(case)
        cos, sin = u15h.build_rope_tables(*pos.numpy(), HEAD_DIM, D_T, D_H)
        s.update(stack=stack, x=x, kc=kc, vc=vc, tier=tier, cos=torch.from_numpy(cos).cuda(),
                 sin=torch.from_numpy(sin).cuda(), t=t_all.cuda(),
                 scratch=u15h.layer_scratch(stack, x.shape[0], tier))
    return s


def _attn_t(case):
    """The t index of a block-causal attention: text, then one image block
    over the last three quarters of the queries."""
    t = torch.arange(case["tk"])
    at = case["q_offset"] + case["tq"] // 4
    t[at:] = at
    return t.int()


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(s):
    c, ops = s["case"], s["ops"]
    kind = c["kind"]
    if kind == "linear":
        ops.linear(s["x"], s["w"], s["b"], s["y"], c["M"], c["K"], c["N"])
        return s["y"]
    if kind == "pack":
        ops.linear_q(s["x"], s["qw"], s["b"], s["y"], c["M"], c["K"], c["N"])
        return s["y"]
    if kind == "steps":
        ops.stack_layer(s["stack"], 0, s["io"], c["M_und"], c["M_gen"])
        return {n: s["bufs"][n] for n in ("q", "k", "v", "o", "gate", "up", "down")}
    if kind == "swiglu":
        und, gen = s["w"].get(u15h.UND, (None, None)), s["w"].get(u15h.GEN, (None, None))
        ops.mot_gate_up_swiglu(s["x"], c["M_und"], c["M_gen"], HIDDEN, *und, *gen, s["h"])
        return s["h"]
    if kind == "i8":
        ops.quant_rows_i8(s["x"], s["xq"], s["sx"])
        ops.mot_gemm_i8(s["xq"], s["sx"], c["M_und"], c["M_gen"], c["K"], [s["proj"]])
        return [s["proj"]["y"], s["xq"], s["sx"]]
    if kind == "attn":
        ops.attention_token_major(s["q"], s["k"], s["v"], s["out"], c["hq"], c["hkv"], c["tk"],
                                  c["mode"], s["t"], c["q_offset"])
        return s["out"]
    ops.stack_forward_full(s["stack"], 0, c["layers"], c["M_und"], c["M_gen"], s["x"], s["kc"],
                           s["vc"], s["cos"], s["sin"], kv_off=c["kv_off"], mode=c["mode"],
                           t_index=s["t"], eps=EPS, tier=s["tier"], scratch=s["scratch"])
    return [s["x"], s["kc"], s["vc"]]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far off it may be
# ---------------------------------------------------------------------------

def _visible(c):
    """(query, key) pairs a pass of attention sees."""
    tq, tk, off = c["tq"], c["tk"], c["q_offset"]
    if c["mode"] == 0:
        return tq * tk
    seen = sum(min(tk, off + i + 1) for i in range(tq))
    if c["mode"] == 2:                             # the image block sees all of itself
        n = c["tq"] - c["tq"] // 4
        seen += n * (n - 1) // 2
    return seen


def work(c):
    kind = c["kind"]
    if kind in ("linear", "pack"):
        M, K, N = c["M"], c["K"], c["N"]
        w = N * K * 2 if kind == "linear" else N * K * c["bits"] // 8 + N * K // c["group"] * 4
        return dict(bytes=w + 2 * M * (K + N) + (2 * N if c["bias"] else 0), flops=2 * M * K * N)
    if kind == "attn":
        q = 2 * c["tq"] * c["hq"] * c["d"]
        return dict(bytes=2 * q + 4 * c["hkv"] * c["tk"] * c["d"],
                    flops=4 * c["hq"] * c["d"] * _visible(c))
    M, sets = c["M_und"] + c["M_gen"], len(_experts(c))
    params = sum(n * k for n, k in _PROJ)
    if kind == "steps":
        acts = M * sum(n for n, _ in _PROJ) + M * (2 * HIDDEN + QDIM + INTER)
        return dict(bytes=2 * (params * sets + acts), flops=2 * M * params)
    if kind == "swiglu":
        return dict(bytes=2 * (2 * INTER * HIDDEN * sets + M * (HIDDEN + INTER)),
                    flops=4 * M * INTER * HIDDEN)
    if kind == "i8":
        return dict(bytes=c["N"] * c["K"] * sets + M * (3 * c["K"] + 2 * c["N"] + 4),
                    flops=2 * M * c["K"] * c["N"])
    tk = c["kv_off"] + M
    a = dict(tq=M, tk=tk, q_offset=c["kv_off"], mode=c["mode"])
    kv = 4 * KVDIM * tk
    one = params * sets * (1 if c["i8"] else 2) + kv
    return dict(bytes=c["layers"] * one + 4 * M * HIDDEN,
                flops=c["layers"] * (2 * M * params + 4 * QDIM * _visible(a)))


def tolerance(c):
    """Relative 2-norm errors between correct programs of this precision.
    Sums in another order (no split K, the tiled kernels at every row count,
    the 32-wide matrix instructions) change a GEMM's bf16 outputs by up to
    6e-5 (one rounding step, 7.8e-3, in a few of 10^4 outputs) and a whole
    layer's by 3e-3, four layers' by 8e-3.  Attention also rounds its
    probabilities, by their distance to a running maximum that depends on
    the order of the keys: 2.3e-3 off the exact result.  The int8 tier turns
    a rounding step of its inputs into a code's."""
    if c["kind"] == "layer":
        many = c["i8"] or c["layers"] > 1
        return {"rel": 3e-2, "max": 0.3} if many else {"rel": 1.3e-2, "max": 0.12}
    if c["kind"] == "i8":
        return {"rel": 2.5e-4, "max": 3e-2, "differ": 0.0}
    if c["kind"] == "attn":
        return {"rel": 6e-3, "max": 5e-2}
    return {"rel": 2e-3, "max": 3e-2}      # one step in a call of 128 outputs: 1.4e-3


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _mm(x, w):
    """x . w^T in 64 bits, the weight converted in pieces."""
    step = max(1, (1 << 27) // w.shape[1])
    return torch.cat([x @ w[i:i + step].to(F64).t() for i in range(0, w.shape[0], step)], 1)


def _attend(q, k, v, q_offset, mode, t):
    """q [tq][hq][d], k and v [hkv][tk][d], all 64-bit; [tq][hq][d]."""
    tq, hq, d = q.shape
    hkv, tk, _ = k.shape
    out = torch.empty_like(q)
    keys = torch.arange(tk, device="cuda")
    pos = q_offset + torch.arange(tq, device="cuda")
    ok = None
    if mode:
        ok = keys[None] <= pos[:, None]
        if mode == 2:
            ok |= t[keys][None] == t[pos][:, None]
    for h in range(hq):
        kv = h // (hq // hkv)
        sc = q[:, h] @ k[kv].t().contiguous() / math.sqrt(d)
        if ok is not None:
            sc.masked_fill_(~ok, -math.inf)
        out[:, h] = torch.softmax(sc, 1) @ v[kv]
    return out


def _rms(x, g):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * g.to(F64)


def _rope(x, pos):
    """x [T][heads][128]: rotate_half on the ranges t, h, w."""
    out, at = x.clone(), 0
    for p, width, theta in zip(pos, (D_T, D_H, D_H), (5e6, 1e4, 1e4)):
        half = width // 2
        inv = theta ** (-torch.arange(half, dtype=F64, device="cuda") * 2 / width)
        a = p.to("cuda", F64)[:, None] * inv
        c, sn = a.cos()[:, None], a.sin()[:, None]
        lo, hi = x[..., at:at + half], x[..., at + half:at + width]
        out[..., at:at + half] = lo * c - hi * sn
        out[..., at + half:at + width] = hi * c + lo * sn
        at += width
    return out


def _exact_layers(case, r):
    W, G, kc, vc, x = _layer_tensors(case, r)
    x = x.to(F64)
    pos, t_all = _positions(case)
    t_all = t_all.cuda()
    M, off = x.shape[0], case["kv_off"]
    groups = [(e, sl) for e, sl in ((u15h.UND, slice(0, case["M_und"])),
                                    (u15h.GEN, slice(case["M_und"], M))) if sl.stop > sl.start]

    def proj(inp, l, p):
        y = torch.empty(M, _PROJ[p][0], dtype=F64, device="cuda")
        for e, sl in groups:
            a, w = inp[sl], W[l, e, p]
            if case["i8"]:
                s = a.abs().amax(1, keepdim=True) / 127
                ra = a / s
                qa = torch.sign(ra) * torch.floor(ra.abs() + 0.5)
                wq, sw = _quant_rows(w)
                y[sl] = _mm(qa, wq) * s * sw.to(F64)
            else:
                y[sl] = _mm(a, w)
        return y

    def norm(inp, l, i):
        return torch.cat([_rms(inp[sl], G[l, e, i]) for e, sl in groups])

    def head_norm(y, l, heads, i):
        y = y.view(M, heads, 2, HEAD_DIM // 2)
        return torch.cat([torch.stack([_rms(y[sl, :, 0], G[l, e, i]),
                                       _rms(y[sl, :, 1], G[l, e, i + 2])], 2)
                          for e, sl in groups]).view(M, heads, HEAD_DIM)

    kx, vx = [], []
    for l in range(case["layers"]):
        n = norm(x, l, 0)
        q = _rope(head_norm(proj(n, l, 0), l, HEADS, 2), pos)
        k = _rope(head_norm(proj(n, l, 1), l, KV_HEADS, 3), pos)
        v = proj(n, l, 2).view(M, KV_HEADS, HEAD_DIM)
        ke, ve = kc[l].to(F64), vc[l].to(F64)
        ke[:, off:off + M], ve[:, off:off + M] = k.transpose(0, 1), v.transpose(0, 1)
        kx.append(ke)
        vx.append(ve)
        a = _attend(q, ke[:, :off + M], ve[:, :off + M], off, case["mode"], t_all)
        x = x + proj(a.reshape(M, QDIM), l, 3)
        n = norm(x, l, 1)
        g = proj(n, l, 4)
        x = x + proj(g * torch.sigmoid(g) * proj(n, l, 5), l, 6)
    return [x, kx, vx]


def exact(case, seed):
    r, kind = _Rand(seed), case["kind"]
    if kind == "linear":
        x, w = r.bf16(case["M"], case["K"]), r.weight(case["N"], case["K"])
        y = _mm(x.to(F64), w)
        return y + r.bf16(case["N"]).to(F64) if case["bias"] else y
    if kind == "pack":
        codes, _, sc, bi = _pack(r, case["N"], case["K"], case["bits"], case["group"])
        rep = lambda t: t.float().repeat_interleave(case["group"], 1)  # noqa: E731
        w = (rep(sc) * codes.float() + rep(bi)).to(BF16)   # the weights the format defines
        y = _mm(r.bf16(case["M"], case["K"]).to(F64), w)
        return y + r.bf16(case["N"]).to(F64) if case["bias"] else y
    if kind == "attn":
        cap = (case["tk"] + 63) // 64 * 64
        hq, hkv, d, tk = case["hq"], case["hkv"], case["d"], case["tk"]
        q = r.bf16(case["tq"], hq * d).to(F64).view(-1, hq, d)
        k, v = r.bf16(hkv, cap, d)[:, :tk].to(F64), r.bf16(hkv, cap, d)[:, :tk].to(F64)
        t = _attn_t(case).cuda() if case["mode"] == 2 else None
        return _attend(q, k, v, case["q_offset"], case["mode"], t).reshape(-1, hq * d)
    if kind == "layer":
        return _exact_layers(case, r)
    mu, mg, M = _rows(case)
    sl = {u15h.UND: slice(0, mu), u15h.GEN: slice(mu, M)}
    if kind == "steps":
        W = {(e, p): r.weight(n, k) for e in _experts(case) for p, (n, k) in enumerate(_PROJ)}
        x, attn, x2, h = (r.bf16(M, n) for n in (HIDDEN, QDIM, HIDDEN, INTER))
        src = (x, x, x, attn, x2, x2, h)
        return {n: torch.cat([_mm(src[p][sl[e]].to(F64), W[e, p]) for e in _experts(case)])
                for p, n in enumerate(("q", "k", "v", "o", "gate", "up", "down"))}
    if kind == "swiglu":
        W = {e: (r.weight(INTER, HIDDEN), r.weight(INTER, HIDDEN)) for e in _experts(case)}
        x, out = r.bf16(M, HIDDEN).to(F64), []
        for e in _experts(case):
            g = _mm(x[sl[e]], W[e][0])
            out.append(g * torch.sigmoid(g) * _mm(x[sl[e]], W[e][1]))
        return torch.cat(out)
    W = {e: _quant_rows(r.weight(case["N"], case["K"])) for e in _experts(case)}
    xq, sx = _quant_rows(r.bf16(M, case["K"]))
    y = torch.cat([_mm(xq[sl[e]].to(F64), W[e][0]) * sx[sl[e], None].to(F64) * W[e][1].to(F64)
                   for e in _experts(case)])
    return [y, None, sx.to(F64)]
