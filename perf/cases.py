"""The work that programs built on this package have it do, as cases that can be timed and compared.

Each case goes through a public entry point of the package: the drop-in BitLinear modules (inference, and
training through their straight-through estimator), the fused single-token MLP op, causal prompt attention and
ragged decode attention over a KV cache, the dense LM head of a greedy decoder, the offline weight pack, and a
decode step of a whole decoder replayed from a HIP graph.  Shapes are the package's own configurations
(SmolLM2-135M, BitNet-2B and Llama-3-8B widths); ``draw`` spreads over the ranges between them, odd sizes among
them.
"""

from __future__ import annotations

import dataclasses
import math

import torch

from __graft_entry__ import load_package

pkg = load_package()

DEV = "cuda:0"
_DT = {"bf16": torch.bfloat16, "fp32": torch.float32, "fp16": torch.float16}
_SIZE = {"bf16": 2, "fp32": 4, "fp16": 2}


def listed():
    return [
        # one projection of a small model for one token: launch latency and the host path
        {"name": "linear_smollm2_1", "kind": "linear", "m": 1, "k": 576, "n": 576, "dtype": "fp32", "subln": False},
        # the fused MLP op of one token at BitNet-2B size (the serving op of the reference's torch extension)
        {"name": "mlp_2b_1", "kind": "mlp", "hidden": 2560, "inter": 6912},
        # a batch of decoding sequences, or a short prompt, through one projection; an odd number of rows
        {"name": "linear_2b_37", "kind": "linear", "m": 37, "k": 2560, "n": 6912, "dtype": "bf16", "subln": False},
        # gate|up of a 2048-token prompt
        {"name": "linear_2b_2048", "kind": "linear", "m": 2048, "k": 2560, "n": 13824, "dtype": "bf16", "subln": False},
        # SubLN + down projection of a long prompt, as stage 1 lays o_proj and down_proj out
        {"name": "subln_2b_8192", "kind": "linear", "m": 8192, "k": 6912, "n": 2560, "dtype": "bf16", "subln": True},
        # a training step's forward and backward through one projection, bf16 working weights refreshed from
        # the optimizer's fp32 master copy
        {"name": "train_2b_2048", "kind": "train", "m": 2048, "k": 2560, "n": 6912, "dtype": "bf16", "subln": False,
         "bias": False},
        # the same through SubLN + BitLinear of a small fp32 model with an odd number of tokens
        {"name": "train_subln_smollm2_501", "kind": "train", "m": 501, "k": 1536, "n": 576, "dtype": "fp32",
         "subln": True, "bias": True},
        # causal attention of a whole prompt at Llama-3-8B heads
        {"name": "prompt_attention_4096", "kind": "prompt_attention", "batch": 1, "tokens": 4096, "start": 0,
         "heads": 32, "kv_heads": 8, "dim": 128},
        # one decode token of eight sequences of different lengths
        {"name": "decode_attention_2304", "kind": "decode_attention", "batch": 8, "max_len": 2304, "heads": 32,
         "kv_heads": 8, "dim": 128, "dtype": "bf16"},
        # greedy pick and logits of a batch over the tied embedding of BitNet-2B
        {"name": "lm_head_2b_4", "kind": "lm_head", "m": 4, "hidden": 2560, "vocab": 128256, "dtype": "bf16"},
        # packing one projection while a checkpoint is loaded
        {"name": "pack_llama3_gate", "kind": "pack", "n": 14336, "k": 4096, "dtype": "fp32"},
        # a whole decode step of a Llama-3-8B-wide decoder (ternary head) in a HIP graph, logits out; 32-bit glue,
        # as the native engine runs a float32 checkpoint (16-bit glue turns a last-bit change of one layer into
        # percents of the logits, whoever computes it)
        {"name": "decode_llama3_8", "kind": "decode", "layers": 2, "batch": 8, "context": 256},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "train", "train", "prompt_attention", "prompt_attention",
                       "decode_attention", "lm_head", "pack", "decode"])
    if kind in ("linear", "train"):
        most = 8192 * 6912 * 2560 if kind == "linear" else 2048 * 2560 * 6912
        while True:
            m = _log(rng, 1, 8192 if kind == "linear" else 4096)
            # widths are multiples of 64 in every configuration; one draw in four is odd
            k, n = (_log(rng, 128, 14336) for _ in range(2))
            if rng.random() < 0.75:
                k, n = k // 64 * 64, n // 64 * 64
            if m * k * n <= most:
                break
        c = {"kind": kind, "m": m, "k": k, "n": n, "dtype": rng.choice(["bf16", "bf16", "fp32"]),
             "subln": rng.random() < 0.5}
        if c["subln"]:  # the fused norm takes rows of a multiple of 8
            c["k"] = k // 8 * 8
        if kind == "train":
            c["bias"] = rng.random() < 0.25
        return c
    if kind == "mlp":
        return {"kind": kind, "hidden": 128 * _log(rng, 2, 32), "inter": 128 * _log(rng, 4, 112)}
    if kind == "prompt_attention":
        while True:
            c = {"kind": kind, "batch": _log(rng, 1, 8), "tokens": _log(rng, 16, 4096),
                 "start": rng.choice([0, 0, _log(rng, 16, 1024)]), "kv_heads": rng.choice([1, 2, 3, 5, 8]),
                 "dim": rng.choice([64, 128])}
            c["heads"] = c["kv_heads"] * rng.choice([1, 2, 3, 4, 5, 8])
            if _attention_pairs(c) * c["heads"] * c["dim"] <= 4096 * 4097 // 2 * 32 * 128:
                return c
    if kind == "decode_attention":
        kv = rng.choice([1, 2, 3, 5, 8])
        return {"kind": kind, "batch": _log(rng, 1, 16), "max_len": _log(rng, 64, 4096), "kv_heads": kv,
                "heads": kv * rng.choice([1, 2, 3, 4, 5, 8]), "dim": rng.choice([64, 128]),
                "dtype": rng.choice(["bf16", "bf16", "fp32"])}
    if kind == "lm_head":
        while True:
            c = {"kind": kind, "m": _log(rng, 1, 16), "hidden": 64 * _log(rng, 8, 64), "vocab": _log(rng, 4096, 128256),
                 "dtype": rng.choice(["bf16", "bf16", "fp32"])}
            if c["m"] * c["hidden"] <= 16384 and c["hidden"] * c["vocab"] * _SIZE[c["dtype"]] <= 128256 * 2560 * 2:
                return c
    if kind == "pack":
        return {"kind": kind, "n": _log(rng, 64, 14336), "k": 8 * _log(rng, 16, 512),
                "dtype": rng.choice(["fp32", "bf16", "fp16"])}
    return {"kind": "decode", "layers": rng.choice([1, 2]), "batch": _log(rng, 1, 8), "context": _log(rng, 8, 256)}


# ---- inputs ----------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _hidden(g, m, h, dtype):
    """Hidden states N(0, 1) with 1% outliers at +-20."""
    x = torch.randn((m, h), generator=g, device=DEV)
    r = torch.rand((m, h), generator=g, device=DEV)
    return torch.where(r < 0.01, torch.where(r < 0.005, -20.0, 20.0), x).to(dtype)


def _weight(g, n, k, dtype=torch.float32):
    return (torch.randn((n, k), generator=g, device=DEV) * 0.02).to(dtype)


def _gamma(g, h, dtype):
    return (1.0 + 0.1 * torch.randn(h, generator=g, device=DEV)).to(dtype)


def _module(c, g, bias=False):
    dt = _DT[c["dtype"]]
    if c["subln"]:
        mod = pkg.SubLNBitLinear(c["k"], c["n"], bias=bias, device=DEV, dtype=dt)
        lin = mod.linear
    else:
        mod = lin = pkg.BitLinear(c["k"], c["n"], bias=bias, device=DEV, dtype=dt)
    master = _weight(g, c["n"], c["k"])
    with torch.no_grad():
        lin.weight.copy_(master)
        if bias:
            lin.bias.copy_(0.1 * torch.randn(c["n"], generator=g, device=DEV))
        if c["subln"]:
            mod.norm_weight.copy_(_gamma(g, c["k"], torch.float32))
    return mod, lin, master


def _llama_layers(layers):
    return dataclasses.replace(pkg.model.LLAMA3_8B, num_layers=layers)


def prepare(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    if kind == "linear":
        mod, lin, _ = _module(c, g)
        lin.pack()
        return {"kind": kind, "mod": mod.requires_grad_(False), "x": _hidden(g, c["m"], c["k"], _DT[c["dtype"]])}
    if kind == "train":
        mod, lin, master = _module(c, g, c["bias"])
        dt = _DT[c["dtype"]]
        x = _hidden(g, c["m"], c["k"], dt).requires_grad_(True)
        gy = (torch.randn((c["m"], c["n"]), generator=g, device=DEV) / math.sqrt(c["n"])).to(dt)
        wrt = [x, lin.weight] + ([lin.bias] if c["bias"] else []) + ([mod.norm_weight] if c["subln"] else [])
        return {"kind": kind, "mod": mod, "lin": lin, "master": master, "x": x, "gy": gy, "wrt": wrt}
    if kind == "mlp":
        h, f = c["hidden"], c["inter"]
        packs = [pkg.pack_ternary_i2s(_weight(g, *s)) for s in ((f, h), (f, h), (h, f))]
        return {"kind": kind, "x": _hidden(g, 1, h, torch.float32).reshape(h), "qw": [p[0] for p in packs],
                "scales": [float(p[1].item()) for p in packs], "norm": _gamma(g, f, torch.float32), "eps": 1e-6}
    if kind == "prompt_attention":
        b, t, hq, hkv, d = c["batch"], c["tokens"], c["heads"], c["kv_heads"], c["dim"]
        total = c["start"] + t
        qkv = torch.randn((b * t, (hq + 2 * hkv) * d), generator=g, device=DEV).to(torch.bfloat16)
        cache = [torch.randn((b, hkv, total, d), generator=g, device=DEV).to(torch.bfloat16) for _ in range(2)]
        cos, sin = pkg.rope_tables(500000.0, d, total)
        q, k, v = torch.split(qkv, [hq * d, hkv * d, hkv * d], dim=1)  # column slices of one projection output
        return {"kind": kind, "q": q, "k": k, "v": v, "kc": cache[0], "vc": cache[1], "start": c["start"], "t": t,
                "cos": cos.to(DEV), "sin": sin.to(DEV)}
    if kind == "decode_attention":
        b, hq, hkv, d, dt = c["batch"], c["heads"], c["kv_heads"], c["dim"], _DT[c["dtype"]]
        qkv = torch.randn((b, (hq + 2 * hkv) * d), generator=g, device=DEV).to(dt)
        cache = [torch.randn((b, hkv, c["max_len"], d), generator=g, device=DEV).to(dt) for _ in range(2)]
        pos = torch.randint(c["max_len"] // 2, c["max_len"], (b,), generator=g, device=DEV)
        cos, sin = pkg.rope_tables(500000.0, d, c["max_len"])
        q, k, v = torch.split(qkv, [hq * d, hkv * d, hkv * d], dim=1)
        return {"kind": kind, "q": q, "k": k, "v": v, "kc": cache[0], "vc": cache[1], "pos": pos, "cos": cos.to(DEV),
                "sin": sin.to(DEV)}
    if kind == "lm_head":
        dt = _DT[c["dtype"]]
        return {"kind": kind, "x": _hidden(g, c["m"], c["hidden"], dt), "w": _weight(g, c["vocab"], c["hidden"], dt),
                "norm": _gamma(g, c["hidden"], dt)}
    if kind == "pack":
        return {"kind": kind, "w": _weight(g, c["n"], c["k"], _DT[c["dtype"]]), "k_pad": (c["k"] + 127) // 128 * 128}
    # decode: a prompt run through the decoder, then one decode step captured in a HIP graph
    m = pkg.model.BitNetDecoder(_llama_layers(c["layers"]), seed=int(seed), device=DEV, dtype=torch.float32,
                                backend=pkg.model.HipBackend(out_dtype=torch.float32, fused=True), init_on_device=True)
    m.reset(c["batch"], c["context"] + 64)
    with torch.no_grad():
        m.forward(torch.randint(0, m.cfg.vocab_size, (c["batch"], c["context"]), generator=g, device=DEV), 0)
        ids = torch.randint(0, m.cfg.vocab_size, (c["batch"], 1), generator=g, device=DEV)
        pos = torch.full((c["batch"],), c["context"], dtype=torch.long, device=DEV)
        m.decode_step(ids, pos)
        graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
            logits = m.decode_step(ids, pos)
        torch.cuda.current_stream().wait_stream(stream)
    return {"kind": kind, "model": m, "ids": ids, "pos": pos, "graph": graph, "logits": logits}


# ---- one pass --------------------------------------------------------------------------------------


def run(state):
    s, kind = state, state["kind"]
    if kind == "linear":
        with torch.no_grad():
            return s["mod"](s["x"])
    if kind == "train":
        with torch.no_grad():
            s["lin"].weight.copy_(s["master"])  # the optimizer's update reaches the working weight
        y = s["mod"](s["x"])
        return [y.detach(), *torch.autograd.grad(y, s["wrt"], s["gy"])]
    if kind == "mlp":
        return torch.ops.wfbitnet.bitnet_mlp_forward(s["x"], *s["qw"], *s["scales"], s["norm"], s["eps"])
    if kind == "prompt_attention":
        return [pkg.gqa_prefill_attention(s["q"], s["k"], s["v"], s["kc"], s["vc"], s["start"], s["t"], s["cos"],
                                          s["sin"]), s["kc"], s["vc"]]
    if kind == "decode_attention":
        return [pkg.gqa_decode_attention(s["q"], s["k"], s["v"], s["kc"], s["vc"], s["pos"], s["cos"], s["sin"]),
                s["kc"], s["vc"]]
    if kind == "lm_head":
        return list(pkg.lm_head_argmax(s["x"], s["w"], s["norm"], return_logits=True))
    if kind == "pack":
        return list(pkg.pack_ternary_i2s(s["w"], k_pad=s["k_pad"]))
    s["graph"].replay()
    return s["logits"]


# ---- what a pass cannot do without -----------------------------------------------------------------


def _attention_pairs(c):
    """Query-key pairs of a causal prompt chunk, all sequences."""
    t = c["tokens"]
    return c["batch"] * (t * c["start"] + t * (t + 1) // 2)


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        m, k, n, e = c["m"], c["k"], c["n"], _SIZE[c["dtype"]]
        return {"bytes": n * k / 4 + m * (k + n) * e, "flops": 2 * m * n * k}
    if kind == "train":  # x, dy, the master weight in; y, dx, the working weight and dw out
        m, k, n, e = c["m"], c["k"], c["n"], _SIZE[c["dtype"]]
        return {"bytes": 2 * m * (k + n) * e + n * k * (4 + 2 * e), "flops": 6 * m * n * k}
    if kind == "mlp":
        h, f = c["hidden"], c["inter"]
        return {"bytes": 3 * h * f / 4 + 4 * (2 * h + f), "flops": 6 * h * f}
    if kind == "prompt_attention":
        rows, d = c["batch"] * c["tokens"], c["dim"]
        seen = c["batch"] * c["kv_heads"] * d * (c["start"] + 2 * c["tokens"])  # old keys read, new ones read and written
        return {"bytes": 2 * (2 * rows * c["heads"] * d + 2 * seen), "flops": 4 * _attention_pairs(c) * c["heads"] * d}
    if kind == "decode_attention":
        keys = c["batch"] * 0.75 * c["max_len"]
        return {"bytes": 2 * keys * c["kv_heads"] * c["dim"] * _SIZE[c["dtype"]],
                "flops": 4 * keys * c["heads"] * c["dim"]}
    if kind == "lm_head":
        m, h, n = c["m"], c["hidden"], c["vocab"]
        return {"bytes": n * h * _SIZE[c["dtype"]] + 4 * m * n, "flops": 2 * m * n * h}
    if kind == "pack":
        return {"bytes": c["n"] * c["k"] * (_SIZE[c["dtype"]] + 0.25), "flops": 3 * c["n"] * c["k"]}
    cfg, b = _llama_layers(c["layers"]), c["batch"]
    qd, kvd = cfg.num_heads * cfg.head_dim, cfg.num_kv_heads * cfg.head_dim
    per = cfg.hidden_size * (2 * qd + 2 * kvd) + 3 * cfg.hidden_size * cfg.intermediate_size
    weights = c["layers"] * per + cfg.vocab_size * cfg.hidden_size
    return {"bytes": weights / 4 + c["layers"] * b * c["context"] * 2 * kvd * 4 + 4 * b * cfg.vocab_size,
            "flops": 2 * b * weights + c["layers"] * 4 * b * c["context"] * qd}


def tolerance(case):
    kind, dt = case["kind"], case.get("dtype")
    if kind == "pack":
        return "exact"
    if kind == "linear":
        # the product of int8 codes and ternary weights is exact; bf16 outputs round once, and a norm summed
        # in another order moves single int8 codes by one
        return {"rel": 1e-2} if dt == "bf16" else {"rel": 1e-3 if case["subln"] else 1e-5, "max": 5e-2}
    if kind == "train":
        return {"rel": 1e-2} if dt == "bf16" else {"rel": 1e-3 if case["subln"] else 1e-5, "max": 5e-2}
    if kind == "mlp":
        return {"rel": 1e-3, "max": 5e-2}
    if kind == "decode":  # a few int8 codes that sit on a rounding boundary, carried through the later layers
        return {"rel": 2e-2, "max": 0.2}
    if kind == "lm_head":  # fp32 logits of a hidden state rounded to the weights' type
        return {"rel": 2e-4 if dt == "bf16" else 1e-5, "max": 1e-2, "differ": 0.0}
    return {"rel": 1e-2 if dt == "bf16" or kind == "prompt_attention" else 1e-5, "max": 5e-2}


# ---- the same in 64 bits ---------------------------------------------------------------------------


def _absmean(w):
    s = w.double().abs().mean().float()
    return torch.where(s.double() < 1e-8, torch.ones_like(s), s)


def _ternary(w, s):
    return torch.clamp(torch.round(w.float() / s), -1, 1)


def _codes(x):
    """Per-token absmax int8 codes of fp32 rows, and their scales: the definition's own 32-bit operations."""
    mx = x.abs().amax(-1, keepdim=True)
    mx = torch.where(mx < 1e-6, torch.ones_like(mx), mx)
    return torch.clamp(torch.round(x * (127.0 / mx)), -128, 127).double(), (mx / 127.0).double()


def _norm64(x, w, eps):
    x = x.double()
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()


def _qlinear(x, w_codes, s, norm=None, eps=1e-6):
    """(y, codes * scales) of [norm ->] quantise -> ternary product, 64-bit but for the quantiser."""
    xs = x.float() if norm is None else _norm64(x, norm, eps).float()
    q, a = _codes(xs)
    return (q @ w_codes.double().t()) * (a * s.double()), q * a


def _unpack(qw):
    """int8 codes {-1, 0, 1} of I2_S bytes [n, k/4]: byte j of a 128-weight block holds weights j, j+32, j+64, j+96
    from the high bits down."""
    n = qw.shape[0]
    b = qw.view(n, -1, 1, 32)
    f = torch.cat([(b >> sh) & 3 for sh in (6, 4, 2, 0)], dim=2)
    return f.reshape(n, -1).to(torch.int8) - 1


def _rope64(x, pos, cos, sin):
    """Rotate-half rotary embedding of x [..., heads, d] at positions pos [...], rounded to x's type."""
    c, s = (t[pos].double().unsqueeze(-2) for t in (cos, sin))
    h = x.shape[-1] // 2
    x1, x2 = x[..., :h].double(), x[..., h:].double()
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], -1).to(x.dtype)


def _attend64(q, k, v, first):
    """Softmax attention of one head: q [t, d] at positions first.., k and v [first + t, d]."""
    t, keys = q.shape[0], k.shape[0]
    sc = (q.double() @ k.double().t().contiguous()) / math.sqrt(q.shape[1])
    mask = torch.arange(keys, device=q.device)[None, :] > torch.arange(first, first + t, device=q.device)[:, None]
    return torch.softmax(sc.masked_fill(mask, float("-inf")), -1) @ v.double()


def _attention64(q, k, v, kc, vc, pos, cos, sin, t):
    """(out [rows, heads*d] in 64 bits, caches with the new keys and values) of t tokens per sequence at pos.."""
    b, hkv, total, d = kc.shape
    hq = q.shape[1] // d
    kc, vc = kc.clone(), vc.clone()
    out = torch.empty((b, t, hq, d), dtype=torch.float64, device=q.device)
    for i in range(b):
        p = torch.arange(t, device=q.device) + int(pos[i])
        qi, ki = (_rope64(x[i * t:(i + 1) * t].reshape(t, -1, d), p, cos, sin) for x in (q, k))
        kc[i, :, p], vc[i, :, p] = ki.transpose(0, 1), v[i * t:(i + 1) * t].reshape(t, hkv, d).transpose(0, 1)
        n = int(pos[i]) + t
        for h in range(hq):
            out[i, :, h] = _attend64(qi[:, h].contiguous(), kc[i, h * hkv // hq, :n], vc[i, h * hkv // hq, :n], n - t)
    return out.reshape(b * t, hq * d), kc, vc


def _decode64(c, s):
    """The decode step of BitNetDecoder in 64 bits, activations rounded to 32 where the quantisers take them."""
    m, cfg = s["model"], s["model"].cfg
    cos, sin = (t.to(DEV) for t in pkg.rope_tables(cfg.rope_theta, cfg.head_dim, c["context"] + 64))
    lin = lambda x, l, norm, eps: _qlinear(x, _unpack(l.qweight), l.scale, norm, eps)[0]  # noqa: E731
    x = m.embed[s["ids"][:, 0]].double()
    for li, L in enumerate(m.layers):
        q, k, v = (lin(x, l, L.input_norm, cfg.rms_eps) for l in (L.q, L.k, L.v))
        kc, vc = (t.double() for t in m.kv[li])
        a, _, _ = _attention64(q, k, v, kc, vc, s["pos"], cos, sin, 1)
        x = x + lin(a, L.o, L.attn_sub_norm, cfg.subln_eps)
        gate, up = (lin(x, l, L.post_attn_norm, cfg.rms_eps) for l in (L.gate, L.up))
        x = x + lin(gate * torch.sigmoid(gate) * up, L.down, L.ffn_sub_norm, cfg.subln_eps)
    y = lin(x, m.lm_head, m.final_norm, cfg.rms_eps)
    return y


def exact(case, seed):
    c, kind, s = case, case["kind"], prepare(case, seed)
    if kind in ("linear", "train"):
        lin = s["mod"].linear if c["subln"] else s["mod"]
        norm = s["mod"].norm_weight.detach() if c["subln"] else None
        w = lin.weight.detach()
        sw = _absmean(w)
        t, x = _ternary(w, sw), s["x"].detach()
        y, xq = _qlinear(x, t, sw, norm)
        if kind == "linear":
            return y
        if c["bias"]:
            y = y + lin.bias.detach().double()
        gy = s["gy"].double()
        gx = (gy @ t.double()) * sw.double()
        grads = [gx, gy.t().contiguous() @ xq] + ([gy.sum(0)] if c["bias"] else [])
        if c["subln"]:
            x64, g64 = x.double().requires_grad_(True), norm.double().requires_grad_(True)
            gx, gg = torch.autograd.grad(_norm64(x64, g64, 1e-6), [x64, g64], gx)
            grads = [gx, *grads[1:], gg]
        return [y, *grads]
    if kind == "mlp":
        codes, sc = [_unpack(q) for q in s["qw"]], [torch.tensor(v, device=DEV) for v in s["scales"]]
        x = s["x"][None]
        gate, up = (_qlinear(x, codes[i], sc[i])[0] for i in (0, 1))
        mid = (torch.relu(gate) ** 2 * up).float()
        return _qlinear(mid, codes[2], sc[2], s["norm"], s["eps"])[0].reshape(-1)
    if kind in ("prompt_attention", "decode_attention"):
        b = c["batch"]
        pos = s["pos"] if kind == "decode_attention" else torch.full((b,), c["start"])
        t = 1 if kind == "decode_attention" else c["tokens"]
        return list(_attention64(s["q"], s["k"], s["v"], s["kc"], s["vc"], pos, s["cos"], s["sin"], t))
    if kind == "lm_head":
        y = _norm64(s["x"], s["norm"], 1e-5).to(s["x"].dtype).double()
        return [None, torch.cat([y @ w.double().t() for w in torch.split(s["w"], 16384)], dim=1)]
    if kind == "pack":
        return [None, _absmean(s["w"]).reshape(1)] if c["k"] == s["k_pad"] else None
    return _decode64(c, s)
