"""Performance cases: what a program that uses ssa_amd has it do.

Six kinds of call, each through public entry points:

  layer    SSAAttention forward (projections, RoPE, routing, attention, o_proj)
  train    SSAAttention forward and backward: the output, the gradients of the
           input and of the four projections
  attend   ssa_attention_bnhd on q, k, v that a model's own projections made
           (the Qwen2 adapter's call); with "grad" also its backward (dq, dk, dv)
  dropin   the reference's two calls in its order: CodebookRouter(q, k, mask)
           (int64 indices by score), then sparse_exact_attention over them
  decode   SSADecodeCache.step for a few new tokens against a filled cache; a
           step of many tokens is a chunk of a long prompt
  blocks   convert_indices_to_blocks on a selection, then ssa_triton_attention
           over the most referenced key blocks

q and k are drawn from a mixture of Gaussian clusters and rotated by position,
as trained heads group their keys; a layer's hidden states are N(0, 1), its
weights the default initialisation's distribution.
"""

import math

import torch

import ssa_amd
from ssa_amd.blocks import convert_indices_to_blocks, ssa_triton_attention
from ssa_amd.decode import SSADecodeCache
from ssa_amd.hf import ssa_attention_bnhd

DEV = "cuda"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


def _case(name, kind, dtype, B, n, h_q, h_kv, d, n_c, a, b, k, d_s=32, **more):
    c = {"kind": kind, "dtype": dtype, "B": B, "n": n, "h_q": h_q, "h_kv": h_kv, "d": d,
         "d_s": d_s, "n_c": n_c, "a": a, "b": b, "k": k, **more}
    return {"name": name, **c} if name else c


def listed():
    return [
        # The smallest call: SSAAttention as constructed without arguments, one short prompt
        # of a ragged length. Latency, launches and host work.
        _case("layer-default", "layer", "fp32", 1, 203, 8, 2, 64, 512, 8, 4, 64, d_s=16, hidden=512),
        # The README's quick-start layer, inference in fp32.
        _case("layer-readme", "layer", "fp32", 2, 1024, 8, 2, 64, 2048, 16, 4, 256, hidden=512),
        # The same layer trained: one forward and backward, as a training step runs them.
        _case("train-readme", "train", "fp32", 2, 1024, 8, 2, 64, 2048, 16, 4, 256, hidden=512),
        # A decoder layer of a large model over a batch of prompts, bf16 inference.
        _case("layer-4x8k", "layer", "bf16", 4, 8192, 32, 8, 128, 4096, 16, 4, 512, hidden=4096),
        # One long prompt through an attention layer.
        _case("attend-32k", "attend", "bf16", 1, 32768, 32, 8, 128, 4096, 16, 4, 512, clusters=64),
        # The longest context: 8:1 GQA, a larger codebook, more keys per query.
        _case("attend-128k", "attend", "bf16", 1, 131072, 16, 2, 128, 8192, 32, 4, 1024, clusters=256),
        # Attention of a fine-tuning step on a long sequence: forward and backward.
        _case("attend-grad-16k", "attend", "bf16", 1, 16384, 32, 8, 128, 4096, 16, 4, 512, clusters=64,
              grad=True),
        # The reference's own two calls in bf16, a program that only changed its import; a ragged length.
        _case("dropin-12k", "dropin", "bf16", 1, 12001, 32, 8, 128, 2048, 16, 4, 512, clusters=64),
        # ... and in fp32 with every key selected, the check against dense attention.
        _case("dropin-all-keys", "dropin", "fp32", 1, 2048, 8, 2, 64, 1024, 16, 4, 2048, clusters=16),
        # One generated token against a long cache with a part-filled tail.
        _case("decode-32k", "decode", "bf16", 1, 32700, 32, 8, 128, 4096, 16, 4, 512, clusters=64, m=1),
        # A chunk of a long prompt against what is cached of it.
        _case("chunk-2k-of-32k", "decode", "bf16", 1, 30720, 32, 8, 128, 4096, 16, 4, 512, clusters=64,
              m=2048),
        # The block-granular path: 64-position blocks, 16 key blocks to a query block.
        _case("blocks-32k", "blocks", "bf16", 1, 32768, 32, 8, 128, 0, 0, 0, 512, block=64, blocks=16),
    ]


def _spread(rng, lo, hi):
    """A size between lo and hi, spread over its logarithm; every second one odd."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n | 1 if rng.random() < 0.5 else n


def _codes(rng, n, k, few=False):
    """Codebook settings in use: enough codes that a query's buckets hold about 2.5 k keys at most."""
    a, b = (rng.choice((8, 16)) if few else rng.choice((16, 16, 32))), 4
    sizes = [s for s in (512, 1024, 2048, 4096, 8192, 16384) if a * b * n <= 2.5 * k * s] or [16384]
    return rng.choice(sizes[:3]), a, b


def draw(rng):
    kind = rng.choice(("layer", "train", "attend", "attend", "grad", "dropin", "decode", "decode", "blocks"))
    if kind in ("layer", "train"):
        if rng.random() < 0.5 or kind == "train":  # the reference's fp32 layers
            hidden, h_q, h_kv, d = rng.choice(((256, 4, 2, 64), (512, 8, 2, 64), (512, 8, 8, 64), (768, 12, 4, 64)))
            n, B, k = _spread(rng, 128, 2000), rng.choice((1, 2)), rng.choice((64, 128, 256))
            dtype = "fp32"
        else:
            hidden, h_q, h_kv, d = rng.choice(((1024, 16, 4, 64), (2048, 16, 4, 128), (4096, 32, 8, 128)))
            n, B, k = _spread(rng, 1000, 8192), rng.choice((1, 2)), rng.choice((256, 512))
            dtype = "bf16"
        k = min(k, n)
        n_c, a, b = _codes(rng, n, k, few=True)
        return _case("", kind, dtype, B, n, h_q, h_kv, d, n_c, a, b, k, d_s=rng.choice((16, 32)), hidden=hidden)
    if kind == "blocks":
        h_q, h_kv, d = rng.choice(((32, 8, 128), (16, 2, 128), (16, 4, 64), (28, 4, 128)))
        n, block = _spread(rng, 2048, 32768), rng.choice((32, 64, 64, 128))
        return _case("", kind, "bf16", 1, n, h_q, h_kv, d, 0, 0, 0, rng.choice((256, 512)), block=block,
                     blocks=rng.randrange(4, 1 + min(16, 1024 // block)))
    h_q, h_kv, d = rng.choice(((32, 8, 128), (16, 2, 128), (28, 4, 128), (16, 4, 64), (12, 4, 128)))
    k = rng.choice((256, 512, 512, 1024))
    n = _spread(rng, *{"attend": (2048, 65536), "grad": (2048, 16384), "dropin": (2048, 20000),
                       "decode": (2048, 65536)}[kind])
    k = min(k, n)
    n_c, a, b = _codes(rng, n, k)
    more = {"clusters": rng.choice((16, 64, 256))}
    if kind == "grad":
        kind, more["grad"] = "attend", True
    if kind == "decode":
        if rng.random() < 0.6:
            more["m"], B = rng.choice((1, 1, 2, 4)), rng.choice((1, 1, 4, 8))
        else:
            more["m"], B = _spread(rng, 300, 4096), 1
        if B * n > 131072:
            n = 131072 // B
        return _case("", kind, "bf16", B, n, h_q, h_kv, d, n_c, a, b, k, **more)
    dtype = "bf16"
    if kind == "dropin" and rng.random() < 0.3:
        dtype, n, h_q, h_kv, d, k = "fp32", _spread(rng, 512, 4096), 8, 2, 64, 256
        n_c, a, b = _codes(rng, n, k)
    return _case("", kind, dtype, 1, n, h_q, h_kv, d, n_c, a, b, k, **more)


# ---- inputs -------------------------------------------------------------------


def _gen(seed, part):
    return torch.Generator(device=DEV).manual_seed(1000003 * (seed + 1) + part)


def _router_weights(c, seed, dtype):
    g = _gen(seed, 1)
    s = 1.0 / math.sqrt(c["d"])
    return {"W_qr.weight": (torch.rand(c["d_s"], c["d"], generator=g, device=DEV) * 2 - 1).mul_(s).to(dtype),
            "W_kr.weight": (torch.rand(c["d_s"], c["d"], generator=g, device=DEV) * 2 - 1).mul_(s).to(dtype),
            "codebook": (torch.randn(c["h_kv"], c["n_c"], c["d_s"], generator=g, device=DEV)
                         / c["d_s"] ** 0.5).to(dtype)}


def _rotate(x, theta=1e6):
    """Rotary embedding by position of x [B, n, h, d]."""
    n, d = x.shape[1], x.shape[3]
    inv = theta ** (-torch.arange(0, d, 2, device=DEV, dtype=torch.float64) / d)
    ang = (torch.arange(n, device=DEV, dtype=torch.float64)[:, None] * inv).to(torch.float32)
    cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]
    lo, hi = x[..., : d // 2], x[..., d // 2:]
    return torch.cat((lo * cos - hi * sin, hi * cos + lo * sin), dim=-1)


def _qkv(c, seed, total):
    """Clustered q and k, rotated by position, and v ~ N(0, 1): [B, total, heads, d]."""
    B, h_q, h_kv, d, dt = c["B"], c["h_q"], c["h_kv"], c["d"], DTYPES[c["dtype"]]
    gen = _gen(seed, 2)
    m = c.get("clusters", 64)
    centres = torch.randn(B, h_kv, m, d, generator=gen, device=DEV)
    z = torch.randint(0, m, (B, total, h_kv), generator=gen, device=DEV)
    kc = centres[torch.arange(B, device=DEV)[:, None, None], torch.arange(h_kv, device=DEV), z]
    k = _rotate(kc + 0.3 * torch.randn(B, total, h_kv, d, generator=gen, device=DEV)).to(dt)
    q = kc.repeat_interleave(h_q // h_kv, dim=2)
    q = _rotate(q.add_(0.3 * torch.randn(B, total, h_q, d, generator=gen, device=DEV))).to(dt)
    v = torch.randn(B, total, h_kv, d, generator=gen, device=DEV).to(dt)
    return q, k, v


def _layer_inputs(c, seed):
    dt, hid = DTYPES[c["dtype"]], c["hidden"]
    gen = _gen(seed, 3)
    x = torch.randn(c["B"], c["n"], hid, generator=gen, device=DEV).to(dt)
    dy = torch.randn(c["B"], c["n"], hid, generator=gen, device=DEV).to(dt)
    w = {}
    for name, rows, cols in (("q_proj", c["h_q"] * c["d"], hid), ("k_proj", c["h_kv"] * c["d"], hid),
                             ("v_proj", c["h_kv"] * c["d"], hid), ("o_proj", hid, c["h_q"] * c["d"])):
        w[name + ".weight"] = (torch.rand(rows, cols, generator=gen, device=DEV) * 2 - 1).mul_(cols ** -0.5).to(dt)
    w.update({"router." + name: t for name, t in _router_weights(c, seed, dt).items()})
    half = c["d"] // 2                           # the reference layer rotates half the features
    inv = 10000.0 ** (-torch.arange(0, half, 2, device=DEV, dtype=torch.float32) / half)
    ang = torch.arange(max(c["n"], c["h_q"]), device=DEV, dtype=torch.float32)[:, None] * inv
    return x, dy, w, torch.cat((ang, ang), dim=-1)


def _selection(c, seed):
    """Token selections as a router leaves them for the block path: every row its neighbourhood, the
    sequence's first keys and keys around a few places that neighbouring rows share."""
    n, h, k, bs = c["n"], c["h_kv"], c["k"], c["block"]
    gen = _gen(seed, 4)
    i = torch.arange(n, device=DEV)[:, None, None]
    near = i - torch.randint(0, 3 * bs, (n, h, k // 4), generator=gen, device=DEV)
    first = torch.randint(0, 2 * bs, (n, h, k // 8), generator=gen, device=DEV)
    nb = -(-n // bs)
    places = (torch.rand(nb, h, 12, generator=gen, device=DEV) * torch.arange(1, nb + 1, device=DEV)[:, None, None] * bs)
    mine = places.long()[torch.arange(n, device=DEV) // bs]                        # [n, h, 12]
    rest = k - near.shape[2] - first.shape[2]
    which = torch.randint(0, 12, (n, h, rest), generator=gen, device=DEV)
    far = mine.gather(2, which) + torch.randint(0, 2 * bs, (n, h, rest), generator=gen, device=DEV)
    return torch.cat((near, first, far), dim=-1).clamp_(0, n - 1)


def _router(c, seed, dtype):
    with torch.device(DEV):
        r = ssa_amd.CodebookRouter(head_dim=c["d"], route_dim=c["d_s"], num_kv_heads=c["h_kv"],
                                   num_codebook=c["n_c"], codes_per_key=c["b"], codes_per_query=c["a"],
                                   top_k=c["k"])
    r = r.to(dtype)
    r.load_state_dict(_router_weights(c, seed, dtype))
    return r


def prepare(case, seed):
    c = case
    kind, dt = c["kind"], DTYPES[c["dtype"]]
    if kind in ("layer", "train"):
        x, dy, w, freqs = _layer_inputs(c, seed)
        with torch.device(DEV):
            layer = ssa_amd.SSAAttention(hidden_size=c["hidden"], num_q_heads=c["h_q"], num_kv_heads=c["h_kv"],
                                         head_dim=c["d"], route_dim=c["d_s"], num_codebook=c["n_c"],
                                         codes_per_key=c["b"], codes_per_query=c["a"], top_k=c["k"])
        layer = layer.to(dt)
        layer.load_state_dict(w)
        state = {"kind": kind, "layer": layer, "x": x, "freqs": freqs}
        if kind == "train":
            x.requires_grad_(True)
            state["dy"] = dy
            state["wrt"] = [x] + [getattr(layer, p).weight for p in ("q_proj", "k_proj", "v_proj", "o_proj")]
        return state
    if kind == "blocks":
        q, k, v = _qkv(c, seed, c["n"])
        return {"kind": kind, "q": q[0], "k": k[0], "v": v[0], "indices": _selection(c, seed),
                "block": c["block"], "blocks": c["blocks"]}
    if kind == "decode":
        m, n0, B = c["m"], c["n"], c["B"]
        q, k, v = _qkv(c, seed, n0 + m)
        cache = SSADecodeCache(_router(c, seed, dt), B, n0 + m, c["d"], dt)
        tail = 200 if m < 256 else 0   # tokens generated since the prompt
        for lo, hi in ((0, n0 - tail), (n0 - tail, n0)):
            if hi > lo:
                cache.step(q[:, lo:hi], k[:, lo:hi], v[:, lo:hi])
        new = [t[:, n0:].contiguous() for t in (q, k, v)]
        return {"kind": kind, "cache": cache, "n0": n0, "new": new}
    q, k, v = _qkv(c, seed, c["n"])
    state = {"kind": kind, "q": q, "k": k, "v": v}
    if kind == "attend":
        state["router"] = _router(c, seed, torch.float32)
        if c.get("grad"):
            for t in (q, k, v):
                t.requires_grad_(True)
            state["dout"] = torch.randn(q.shape, generator=_gen(seed, 5), device=DEV).to(dt)
    else:
        state["router"] = _router(c, seed, dt)
        state.update(q=q[0], k=k[0], v=v[0])
    return state


def run(state):
    s = state
    kind = s["kind"]
    if kind == "layer":
        with torch.no_grad():
            return s["layer"](s["x"], freqs=s["freqs"])
    if kind == "train":
        y = s["layer"](s["x"], freqs=s["freqs"])
        return [y.detach(), *torch.autograd.grad(y, s["wrt"], s["dy"])]
    if kind == "attend":
        if "dout" in s:
            out = ssa_attention_bnhd(s["q"], s["k"], s["v"], s["router"])
            return [out.detach(), *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"])]
        with torch.no_grad():
            return ssa_attention_bnhd(s["q"], s["k"], s["v"], s["router"])
    if kind == "dropin":
        with torch.no_grad():
            idx = s["router"](s["q"], s["k"], causal_mask=True)
            return [idx, ssa_amd.sparse_exact_attention(s["q"], s["k"], s["v"], idx)]
    if kind == "decode":
        cache = s["cache"]
        cache.len = s["n0"]          # the tokens of the last pass were not accepted
        out, idx = cache.step(*s["new"], return_indices=True)
        return [out, idx]
    blocks = convert_indices_to_blocks(s["indices"], s["block"])[..., : s["blocks"]]
    return [blocks, ssa_triton_attention(s["q"], s["k"], s["v"], blocks, s["block"])]


# ---- what is compared and what cannot be done without -----------------------------


def work(case):
    c = case
    s = 4 if c["dtype"] == "fp32" else 2
    m = c.get("m", c["n"])                       # query rows
    n = c["n"] + c["m"] if c["kind"] == "decode" else c["n"]
    B, h_q, h_kv, d, k = c["B"], c["h_q"], c["h_kv"], c["d"], c["k"]
    qo, kv = B * m * h_q * d, B * n * h_kv * d
    if c["kind"] == "blocks":
        # listed keys, causally: about what a row's list holds of its own past
        return {"bytes": 2 * qo * s + 2 * kv * s + n * h_kv * k * 8,
                "flops": 4.0 * n * h_q * d * min(c["blocks"] * c["block"], n / 2)}
    cb = h_kv * c["n_c"] * c["d_s"]
    new = B * m                                  # rows routed
    route = 2.0 * new * (h_q + h_kv) * d * c["d_s"] + 4.0 * new * h_kv * c["n_c"] * c["d_s"]
    attend = 4.0 * B * m * h_q * min(k, n) * d
    if c["kind"] == "decode":
        # a step reads no more of the cache than the keys its rows select
        kv = min(kv, B * m * h_kv * k * d) + B * m * h_kv * d
        return {"bytes": 2 * qo * s + 2 * kv * s + B * m * h_kv * k * 4 + cb * 4, "flops": route + attend}
    if c["kind"] in ("layer", "train"):
        w = (2 * h_q + 2 * h_kv) * d * c["hidden"]
        t = 3 if c["kind"] == "train" else 1
        x = B * n * c["hidden"]
        return {"bytes": (2 * x + w) * s * (2 if t == 3 else 1) + cb * s,
                "flops": t * 2.0 * B * n * w + route + (3.5 if t == 3 else 1) * attend}
    idx = n * h_kv * k * 8 if c["kind"] == "dropin" else 0
    grad = bool(c.get("grad"))
    return {"bytes": (2 * qo + 2 * kv) * s * (2 if grad else 1) + cb * 4 + idx,
            "flops": route + (3.5 if grad else 1) * attend}


def tolerance(case):
    # Selections and block lists are whole numbers and the same for every correct implementation.
    # bf16 results are rounded once from 32-bit sums (2^-9 a value, about 1.7e-3 over a tensor, seen
    # against exact); fp32 results carry the order of their 32-bit sums and the exponential's last bits.
    return {"rel": 7e-3 if case["dtype"] == "bf16" else 1e-5, "differ": 0.0}


# ---- the same in 64 bits -------------------------------------------------------------


def _unit(x):
    return x / x.norm(dim=-1, keepdim=True).clamp_min(1e-12)


def _attend64(c, q, k, v, w, pos0=0, dout=None):
    """Routing, selection and attention of q [B, m, h_q, d] at positions pos0.. against k, v
    [B, n, h_kv, d], all float64; with dout also the gradients."""
    B, m, h_q, d = q.shape
    n, h = k.shape[1], c["h_kv"]
    g = h_q // h
    sel = min(c["k"], n)
    wq, wk, cb = (w[x].double() for x in ("W_qr.weight", "W_kr.weight", "codebook"))
    out = torch.empty_like(q)
    dq, dk, dv = (torch.zeros_like(t) for t in (q, k, v)) if dout is not None else (None, None, None)
    ids = torch.arange(n, device=DEV)
    rows = max(1, min(m, (1 << 28) // (n * g)))
    for bb in range(B):
        for hh in range(h):
            K, V = k[bb, :, hh], v[bb, :, hh].contiguous()
            Kt = K.t().contiguous()
            C = _unit(cb[hh]).t().contiguous()
            has = torch.zeros(c["n_c"], n, dtype=torch.bool, device=DEV)
            for lo in range(0, n, 65536):
                code = (_unit(K[lo:lo + 65536] @ wk.t()) @ C).topk(c["b"], dim=-1).indices
                has[code, ids[lo:lo + 65536, None]] = True
            for lo in range(0, m, rows):
                hi = min(m, lo + rows)
                r = hi - lo
                Q = q[bb, lo:hi, hh * g:(hh + 1) * g].reshape(r * g, d)
                qr = _unit((Q @ wq.t()).view(r, g, -1).mean(1))
                code = (qr @ C).topk(c["a"], dim=-1).indices
                cand = has[code[:, 0]]
                for t in range(1, c["a"]):
                    cand |= has[code[:, t]]
                cand &= ids[None] <= (torch.arange(lo, hi, device=DEV) + pos0)[:, None]
                S = (Q @ Kt).div_(math.sqrt(d)).view(r, g, n)
                rank = torch.where(cand, S.mean(1), (-1e6 - ids.double())[None])
                top = rank.topk(sel, dim=-1, sorted=False).indices
                keep = torch.zeros(r, n, dtype=torch.bool, device=DEV).scatter_(1, top, True)
                P = S.masked_fill_(~keep[:, None], -math.inf).softmax(-1).view(r * g, n)
                O = P @ V
                out[bb, lo:hi, hh * g:(hh + 1) * g] = O.view(r, g, d)
                if dout is None:
                    continue
                dO = dout[bb, lo:hi, hh * g:(hh + 1) * g].reshape(r * g, d)
                dv[bb, :, hh] += P.t() @ dO
                dS = (dO @ V.t()).sub_((dO * O).sum(-1, keepdim=True)).mul_(P).div_(math.sqrt(d))
                dq[bb, lo:hi, hh * g:(hh + 1) * g] = (dS @ K).view(r, g, d)
                dk[bb, :, hh] += dS.t() @ Q
    return (out, dq, dk, dv) if dout is not None else out


def _layer64(c, seed, train):
    x, dy, w, freqs = _layer_inputs(c, seed)
    dt, B, n, d, half = DTYPES[c["dtype"]], c["B"], c["n"], c["d"], c["d"] // 2
    x64 = x.double()
    W = {p: w[p + ".weight"].double() for p in ("q_proj", "k_proj", "v_proj", "o_proj")}

    def rounded(t):                              # the layer's tensors between its steps have its type
        return t.to(dt).double()

    q, k, v = (rounded(x64 @ W[p].t()).view(B, n, -1, d) for p in ("q_proj", "k_proj", "v_proj"))

    def rope(t, sign=1.0):                       # one angle for each head; sign -1 is the transpose
        ang = freqs[: t.shape[2], : half // 2]
        cos, sin = ang.cos().double(), ang.sin().double() * sign
        lo, hi = t[..., : half // 2], t[..., half // 2: half]
        return rounded(torch.cat((lo * cos - hi * sin, hi * cos + lo * sin, t[..., half:]), dim=-1))

    q, k = rope(q), rope(k)
    rw = {p: w["router." + p] for p in ("W_qr.weight", "W_kr.weight", "codebook")}
    if not train:
        o = rounded(_attend64(c, q, k, v, rw)).reshape(B, n, -1)
        return o @ W["o_proj"].t()
    dy64 = dy.double()
    do = (dy64 @ W["o_proj"]).view(B, n, -1, d)
    o, dq, dk, dv = _attend64(c, q, k, v, rw, 0, do)
    o = o.reshape(B * n, -1)
    dq, dk = rope(dq, -1.0), rope(dk, -1.0)
    flat = [t.reshape(B * n, -1) for t in (dq, dk, dv)]
    xf = x64.view(B * n, -1)
    dx = sum(t @ W[p] for t, p in zip(flat, ("q_proj", "k_proj", "v_proj")))
    return [(o @ W["o_proj"].t()).view(B, n, -1), dx.view_as(x64), *(t.t() @ xf for t in flat),
            dy64.view(B * n, -1).t() @ o]


def _blocks64(c, seed):
    q, k, v = (t[0].double() for t in _qkv(c, seed, c["n"]))
    n, bs, h, d = c["n"], c["block"], c["h_kv"], c["d"]
    g, nb = c["h_q"] // h, -(-c["n"] // c["block"])
    idx = _selection(c, seed) // bs
    count = torch.zeros(nb, h, nb, dtype=torch.int64, device=DEV)
    for r in range(bs):
        part = idx[r::bs]
        count[: part.shape[0]].scatter_add_(2, part, torch.ones_like(part))
    count[-1, :, 0] += (nb * bs - n) * c["k"]    # rows past the end refer to block 0
    rank = count * nb + torch.arange(nb - 1, -1, -1, device=DEV)
    picked = rank.sort(-1, descending=True).indices[..., : min(c["blocks"], c["k"], nb)]
    listed_ = torch.zeros(nb, h, nb, dtype=torch.bool, device=DEV).scatter_(2, picked, True)
    ids = torch.arange(n, device=DEV)
    out = torch.empty_like(q)
    rows = max(bs, (1 << 28) // (n * g) // bs * bs)
    for hh in range(h):
        Kt, V = k[:, hh].t().contiguous(), v[:, hh].contiguous()
        for lo in range(0, n, rows):
            i = ids[lo:lo + rows]
            keep = listed_[i // bs, hh][:, ids // bs] & (ids[None] <= i[:, None])
            Q = q[lo:lo + rows, hh * g:(hh + 1) * g].reshape(-1, d)
            S = (Q @ Kt).div_(math.sqrt(d)).view(len(i), g, n).masked_fill_(~keep[:, None], -math.inf)
            P = S.softmax(-1).nan_to_num_(0.0)   # a row with no key of its past among the blocks
            out[lo:lo + rows, hh * g:(hh + 1) * g] = (P.view(-1, n) @ V).view(len(i), g, d)
    return [None, out]


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind in ("layer", "train"):
        return _layer64(c, seed, kind == "train")
    if kind == "blocks":
        return _blocks64(c, seed)
    if kind == "decode":
        q, k, v = (t.double() for t in _qkv(c, seed, c["n"] + c["m"]))
        w = _router_weights(c, seed, DTYPES[c["dtype"]])
        return [_attend64(c, q[:, c["n"]:].contiguous(), k, v, w, c["n"]), None]
    if c["n"] > 65536:                           # takes longer than the comparison is worth
        return None
    q, k, v = (t.double() for t in _qkv(c, seed, c["n"]))
    if kind == "attend":
        w = _router_weights(c, seed, torch.float32)
        if not c.get("grad"):
            return _attend64(c, q, k, v, w)
        dout = torch.randn(q.shape, generator=_gen(seed, 5), device=DEV).to(DTYPES[c["dtype"]]).double()
        return list(_attend64(c, q, k, v, w, 0, dout))
    w = _router_weights(c, seed, DTYPES[c["dtype"]])
    return [None, _attend64(c, q, k, v, w)[0]]
