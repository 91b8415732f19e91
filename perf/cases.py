"""Performance cases of the SmolLM3-3B engine on one GPU.

What a program that uses this library has it do, through its public entry
points: whole model calls (a prompt, then greedy decode steps) and the blocks
of a layer through the kernel-level calls on device pointers (the single-token
MLP and projections, the lm_head, decode and prompt attention, the prompt
GEMM, sampling). Shapes are SmolLM3-3B's; draw() spreads them over the sizes,
formats and options that the entry points take.

Weights are random in the library's Q4 layout (q in 1..15, f16 scales
|N(0, 0.02)| / 7) or binary16 N(0, 0.02); activations N(0, 1).
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

pkg = importlib.import_module("qora-llm_amd")

DEV = "cuda:0"
HIDDEN, INTER, VOCAB = 2048, 11008, 128256


def listed():
    model = dict(op="model", hidden=HIDDEN, inter=INTER, heads=16, kv_heads=4, head_dim=128, vocab=VOCAB)
    return [
        # A chat turn on the whole model: a 64-token prompt, then 16 greedy
        # tokens, each step a call of the host (prefill and decode).
        dict(model, name="chat_q4", fmt="q4", layers=36, prompt=64, steps=16, kv="f32"),
        # The first token after a long prompt on the whole model (prefill).
        dict(model, name="prompt_q4", fmt="q4", layers=36, prompt=512, steps=0, kv="f32"),
        # The binary16 weight format on a stack of eight layers: a ragged
        # prompt that crosses one attention tile, then 16 decode steps, with
        # the f16 cache.
        dict(model, name="chat_f16", fmt="f16", layers=8, prompt=100, steps=16, kv="f16"),
        # The smallest call: one token's k (or v) projection, where launches
        # and latency are everything.
        dict(name="kv_proj_q4", op="gemv", fmt="q4", k=HIDDEN, n=512),
        # One token's MLP as a host drives it call by call: RMSNorm, fused
        # gate|up with SiLU, down.
        dict(name="mlp_q4", op="mlp", fmt="q4", k=HIDDEN, n=INTER),
        dict(name="mlp_f16", op="mlp", fmt="f16", k=HIDDEN, n=INTER),
        # One token's logits from the tied embedding, in the layout it was
        # uploaded in.
        dict(name="lm_head_q4", op="lm_head", fmt="q4", rows=VOCAB, cols=HIDDEN),
        # Decode attention of one layer over a long f16 cache.
        dict(name="attn_long_f16", op="attn_decode", kv="f16", positions=32700, heads=16, kv_heads=4, head_dim=128),
        # Causal attention of one layer over a 512-token prompt chunk.
        dict(name="attn_prompt", op="attn_prefill", kv="f32", tokens=512, pos0=0, heads=16, kv_heads=4, head_dim=128),
        # One prompt projection: a full chunk through the gate projection,
        # and a short ragged prompt through down.
        dict(name="gemm_q4_512", op="gemm", fmt="q4", tokens=512, k=HIDDEN, n=INTER),
        dict(name="gemm_q4_24", op="gemm", fmt="q4", tokens=24, k=INTER, n=HIDDEN),
        # The sampler with the default settings over the whole vocabulary,
        # with a history of generated tokens to penalise.
        dict(name="sample_top20", op="sample", vocab=VOCAB, top_k=20, history=200),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["model", "gemv", "gemv", "mlp", "mlp", "lm_head", "attn_decode", "attn_decode", "attn_prefill",
                     "attn_prefill", "gemm", "gemm", "gemm", "sample"])
    heads, kv_heads, head_dim = rng.choice([(16, 4, 128), (16, 4, 128), (4, 2, 64), (8, 8, 64), (12, 4, 128)])
    kv = rng.choice(["f32", "f16"])
    fmt = rng.choice(["q4", "q4", "f16"])
    if op == "model":
        return dict(op=op, fmt=fmt, layers=rng.randint(2, 8), hidden=rng.choice([256, 512, 1024, 2048, 2048]),
                    inter=32 * _log_int(rng, 16, 344), heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                    vocab=_log_int(rng, 1000, 32000), prompt=_log_int(rng, 2, 600), steps=rng.randint(0, 16), kv=kv)
    if op == "gemv":
        return dict(op=op, fmt=fmt, k=_log_int(rng, 500, INTER), n=32 * _log_int(rng, 8, 344))
    if op == "mlp":
        return dict(op=op, fmt=fmt, k=32 * _log_int(rng, 8, 64), n=32 * _log_int(rng, 16, 344))
    if op == "lm_head":
        return dict(op=op, fmt=fmt, rows=_log_int(rng, 4000, VOCAB), cols=rng.choice([512, 1024, 2048]))
    if op == "attn_decode":
        return dict(op=op, kv=kv, positions=_log_int(rng, 20, 32768), heads=heads, kv_heads=kv_heads,
                    head_dim=head_dim)
    if op == "attn_prefill":
        return dict(op=op, kv=kv, tokens=_log_int(rng, 16, 512), pos0=rng.choice([0, rng.randint(1, 1536)]),
                    heads=heads, kv_heads=kv_heads, head_dim=head_dim)
    if op == "gemm":
        return dict(op=op, fmt=fmt, tokens=_log_int(rng, 4, 512), k=32 * _log_int(rng, 8, 344),
                    n=32 * _log_int(rng, 8, 344))
    return dict(op=op, vocab=_log_int(rng, 4000, VOCAB), top_k=rng.choice([1, 20, 20, 40, 64, 0]),
                history=rng.randint(0, 1000))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + stream) & 0x7FFFFFFFFFFFFFFF)
    return g


def _normal(seed, stream, *shape, std=1.0):
    return torch.randn(*shape, generator=_gen(seed, stream), device=DEV, dtype=torch.float32) * std


def _weight_dev(fmt, seed, stream, k, n):
    """A weight's stored values on the GPU: (bytes [k][n/2], f16 scales [k][n/32]) or f16 [k][n]."""
    if fmt == "f16":
        return (_normal(seed, stream, k, n, std=0.02).half(),)
    g = _gen(seed, stream)
    # both nibbles uniform in 1..15, as one draw of 0..224 per byte
    b = torch.randint(0, 225, (k, n // 2), generator=g, device=DEV, dtype=torch.uint8)
    packed = (b % 15 + 1) | ((torch.div(b, 15, rounding_mode="floor") + 1) << 4)
    scales = (torch.randn(k, n // 32, generator=g, device=DEV).abs() * (0.02 / 7)).half()
    return packed, scales


def _weight(fmt, seed, stream, k, n):
    t = [x.cpu().numpy() for x in _weight_dev(fmt, seed, stream, k, n)]
    if fmt == "f16":
        return pkg.Weight(k, n, data=t[0].view(np.uint16).reshape(-1))
    return pkg.Weight(k, n, packed=t[0].reshape(-1), scales=t[1].view(np.uint16).reshape(-1))


def _weight64(fmt, seed, stream, k, n):
    t = _weight_dev(fmt, seed, stream, k, n)
    if fmt == "f16":
        return t[0].double()
    q = torch.stack((t[0] & 15, t[0] >> 4), dim=-1).reshape(k, n).double() - 8.0
    return (q.reshape(k, n // 32, 32) * t[1].double().unsqueeze(-1)).reshape(k, n)


def _norm_gamma(seed, stream, n):
    return (1.0 + _normal(seed, stream, n, std=0.1)).half()


def _config(c):
    return pkg.ModelConfig(num_layers=c["layers"], vocab=c["vocab"], hidden=c["hidden"], intermediate=c["inter"],
                           num_heads=c["heads"], num_kv_heads=c["kv_heads"], head_dim=c["head_dim"],
                           rope_half_dim=c["head_dim"] // 2)


def _capacity(c):
    return max(2048, c["prompt"] + c["steps"])


def _prompt(c, seed):
    return torch.randint(0, c["vocab"], (c["prompt"],), generator=_gen(seed, 7), device=DEV).cpu().numpy()


def prepare(case, seed):
    op = case["op"]
    ctx = pkg.HipContext(0)
    s = dict(case, ctx=ctx, lib=ctx.lib, h=ctx.h)
    if op == "model":
        cfg = _config(case)
        layers = [[_weight(case["fmt"], seed, 100 + 16 * l + j, k, n) for j, (k, n) in enumerate(cfg.weight_shapes())]
                  for l in range(cfg.num_layers)]
        embed = _weight(case["fmt"], seed, 90, cfg.vocab, cfg.hidden)
        gam = [_norm_gamma(seed, 10000 + i, cfg.hidden).cpu().numpy().view(np.uint16)
               for i in range(2 * cfg.num_layers + 1)]
        cos_t, sin_t = pkg.rope_tables(_capacity(case), cfg.rope_half_dim, cfg.rope_theta)
        flags = np.array([1 if i % 4 == 3 else 0 for i in range(cfg.num_layers)], dtype=np.uint8)
        w = pkg.DecodeWeights(cfg, pkg.FORMAT_Q4 if case["fmt"] == "q4" else pkg.FORMAT_F16, layers, gam[0:-1:2],
                              gam[1:-1:2], embed, gam[-1], cos_t, sin_t, flags)
        s["model"] = pkg.HipBackend(ctx, w, kv_capacity=_capacity(case),
                                    kv_dtype=pkg.KV_F16 if case["kv"] == "f16" else pkg.KV_F32)
        s["ids"] = _prompt(case, seed)
        s["model"].raw_prefill([0, 1], want_logits=False)   # a loaded server has run its buffers' set-up
    elif op == "gemv":
        wid = ctx.upload(_weight(case["fmt"], seed, 1, case["k"], case["n"]))
        s.update(w=ctx.weight_ptrs(wid), x=_normal(seed, 2, case["k"]), y=torch.zeros(case["n"], device=DEV))
    elif op == "mlp":
        k, n, fmt = case["k"], case["n"], case["fmt"]
        s.update(wg=ctx.weight_ptrs(ctx.upload(_weight(fmt, seed, 1, k, n))),
                 wu=ctx.weight_ptrs(ctx.upload(_weight(fmt, seed, 2, k, n))),
                 wd=ctx.weight_ptrs(ctx.upload(_weight(fmt, seed, 3, n, k))),
                 gamma=_norm_gamma(seed, 4, k), x=_normal(seed, 5, k), xn=torch.zeros(k, device=DEV),
                 a=torch.zeros(n, device=DEV), y=torch.zeros(k, device=DEV))
    elif op == "lm_head":
        wid = ctx.upload(_weight(case["fmt"], seed, 1, case["rows"], case["cols"]))
        s.update(w=ctx.weight_ptrs(wid), x=_normal(seed, 2, case["cols"]), y=torch.zeros(case["rows"], device=DEV))
    elif op in ("attn_decode", "attn_prefill"):
        rows = case["positions"] if op == "attn_decode" else case["pos0"] + case["tokens"]
        t = 1 if op == "attn_decode" else case["tokens"]
        kv = torch.float16 if case["kv"] == "f16" else torch.float32
        q = _normal(seed, 1, t, case["heads"] * case["head_dim"])
        k, v = (_normal(seed, i, rows, case["kv_heads"] * case["head_dim"]).to(kv) for i in (2, 3))
        s.update(q=q, k=k, v=v, y=torch.zeros_like(q))
    elif op == "gemm":
        s["wid"] = ctx.upload(_weight(case["fmt"], seed, 1, case["k"], case["n"]))
        s.update(x=_normal(seed, 2, case["tokens"], case["k"]),
                 y=torch.zeros(case["tokens"], case["n"], device=DEV))
    elif op == "sample":
        # a language model's logits: a broad bulk and a few likely tokens
        logits = _normal(seed, 1, case["vocab"], std=2.0)
        top = torch.randperm(case["vocab"], generator=_gen(seed, 2), device=DEV)[:32]
        logits[top] += 8.0 + 3.0 * _normal(seed, 3, 32)
        hist = torch.randint(0, case["vocab"], (case["history"],), generator=_gen(seed, 4), device=DEV)
        hist[: case["history"] // 4] = top[: 8].repeat(case["history"])[: case["history"] // 4]
        s.update(logits=logits, hist=hist.cpu().numpy().astype(np.uint32),
                 params=pkg.SampleParams(0.7, 0.95, case["top_k"], 1.1, 1.5),
                 rng=(int(seed) * 2654435761 + 88172645463325252) & 0xFFFFFFFFFFFFFFFF)
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _gemv(s, w, x, y, k, n):
    if s["fmt"] == "q4":
        s["ctx"].check(s["lib"].qora_hip_gemv_q4(s["h"], w[0], w[1], x.data_ptr(), y.data_ptr(), k, n, None))
    else:
        s["ctx"].check(s["lib"].qora_hip_gemv_f16(s["h"], w[0], x.data_ptr(), y.data_ptr(), k, n, None))


def run(state):
    s = state
    op, ctx, lib, h = s["op"], s["ctx"], s["lib"], s["h"]
    if op == "model":
        m = s["model"]
        first, tok = m.raw_prefill(s["ids"])
        out, last = [tok], first
        for i in range(s["steps"]):
            # the host reads the token of every step, the logits of the last
            last, tok = m.forward_decode_raw(tok, want_logits=i + 1 == s["steps"])
            out.append(tok)
        return dict(first=first, last=last, tokens=np.array(out, dtype=np.int64))
    if op == "gemv":
        _gemv(s, s["w"], s["x"], s["y"], s["k"], s["n"])
        return s["y"]
    if op == "mlp":
        k, n = s["k"], s["n"]
        ctx.check(lib.qora_hip_rmsnorm(h, s["x"].data_ptr(), s["gamma"].data_ptr(), k, s["xn"].data_ptr(), None))
        wg, wu, xn, a = s["wg"], s["wu"], s["xn"].data_ptr(), s["a"].data_ptr()
        if s["fmt"] == "q4":
            ctx.check(lib.qora_hip_gate_up_q4(h, wg[0], wg[1], wu[0], wu[1], xn, a, k, n, None))
        else:
            ctx.check(lib.qora_hip_gate_up_f16(h, wg[0], wu[0], xn, a, k, n, None))
        _gemv(s, s["wd"], s["a"], s["y"], n, k)
        return s["a"], s["y"]
    if op == "lm_head":
        x, y = s["x"].data_ptr(), s["y"].data_ptr()
        if s["fmt"] == "q4":
            ctx.check(lib.qora_hip_gemv_q4_rowdot(h, s["w"][0], s["w"][1], x, y, s["rows"], s["cols"], None))
        else:
            ctx.check(lib.qora_hip_gemv_f16_rowdot(h, s["w"][0], x, y, s["rows"], s["cols"], None))
        return s["y"]
    if op == "attn_decode":
        ctx.check(lib.qora_hip_attn_decode(h, s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                                           int(s["kv"] == "f16"), s["positions"], s["heads"], s["kv_heads"],
                                           s["head_dim"], s["y"].data_ptr(), None))
        return s["y"]
    if op == "attn_prefill":
        ctx.check(lib.qora_hip_attn_prefill(h, s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                                            int(s["kv"] == "f16"), s["pos0"], s["tokens"], s["heads"], s["kv_heads"],
                                            s["head_dim"], s["y"].data_ptr(), None))
        return s["y"]
    if op == "gemm":
        ctx.check(lib.qora_hip_gemm(h, s["wid"], s["x"].data_ptr(), s["y"].data_ptr(), s["tokens"], None))
        return s["y"]
    tok, rng = ctx.sample(s["logits"].data_ptr(), s["vocab"], s["hist"], s["params"], s["rng"])
    return np.array([tok, rng & 0xFFFFFFFF, rng >> 32], dtype=np.int64)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------

def _wbytes(fmt, k, n):
    return k * n * 2 if fmt == "f16" else k * n // 2 + k * n // 16


def work(case):
    op, c = case["op"], case
    if op == "model":
        cfg = _config(c)
        layer = sum(_wbytes(c["fmt"], k, n) for k, n in cfg.weight_shapes())
        params = cfg.num_layers * sum(k * n for k, n in cfg.weight_shapes())
        head, eb = _wbytes(c["fmt"], cfg.vocab, cfg.hidden), 2 if c["kv"] == "f16" else 4
        row = 2 * cfg.num_layers * cfg.num_kv_heads * cfg.head_dim * eb      # one position's K and V
        chunks = -(-c["prompt"] // 512)                                      # the weights stream once a chunk
        ctxs = [c["prompt"] + i + 1 for i in range(c["steps"])]
        pairs = c["prompt"] * (c["prompt"] + 1) // 2 + sum(ctxs)
        return {"bytes": (chunks + c["steps"]) * cfg.num_layers * layer + (1 + c["steps"]) * head
                + row * (2 * c["prompt"] + sum(ctxs)),
                "flops": 2 * params * (c["prompt"] + c["steps"]) + 2 * cfg.vocab * cfg.hidden * (1 + c["steps"])
                + 4 * cfg.num_layers * cfg.num_heads * cfg.head_dim * pairs}
    if op == "gemv":
        return {"bytes": _wbytes(c["fmt"], c["k"], c["n"]) + 4 * (c["k"] + c["n"]), "flops": 2 * c["k"] * c["n"]}
    if op == "mlp":
        return {"bytes": 3 * _wbytes(c["fmt"], c["k"], c["n"]) + 2 * c["k"] + 4 * (2 * c["k"] + c["n"]),
                "flops": 6 * c["k"] * c["n"]}
    if op == "lm_head":
        return {"bytes": _wbytes(c["fmt"], c["rows"], c["cols"]) + 4 * (c["rows"] + c["cols"]),
                "flops": 2 * c["rows"] * c["cols"]}
    if op in ("attn_decode", "attn_prefill"):
        t, pos0 = (1, c["positions"] - 1) if op == "attn_decode" else (c["tokens"], c["pos0"])
        pairs = t * pos0 + t * (t + 1) // 2
        return {"bytes": 2 * (pos0 + t) * c["kv_heads"] * c["head_dim"] * (2 if c["kv"] == "f16" else 4)
                + 8 * t * c["heads"] * c["head_dim"], "flops": 4 * pairs * c["heads"] * c["head_dim"]}
    if op == "gemm":
        return {"bytes": _wbytes(c["fmt"], c["k"], c["n"]) + 4 * c["tokens"] * (c["k"] + c["n"]),
                "flops": 2 * c["tokens"] * c["k"] * c["n"]}
    return {"bytes": 4 * c["vocab"], "flops": 2 * c["vocab"]}


def tolerance(case):
    op = case["op"]
    if op == "sample":
        return "exact"
    # About four times the distance from exact(): up to 5e-7 for one block
    # (32-bit sums), 2.4e-6 for a whole model, and 4.6e-5 for a model with an
    # f16 cache, where a last-bit difference of a layer's input moves some of
    # the rounded K and V to the neighbouring binary16 value.
    if op == "model":
        return {"rel": 2e-4 if case["kv"] == "f16" else 1e-5}
    return {"rel": 2e-6}


def _model64(c, seed):
    cfg, fmt = _config(c), c["fmt"]
    mats = [[_weight64(fmt, seed, 100 + 16 * l + j, k, n) for j, (k, n) in enumerate(cfg.weight_shapes())]
            for l in range(cfg.num_layers)]
    embed = _weight64(fmt, seed, 90, cfg.vocab, cfg.hidden)
    gam = [_norm_gamma(seed, 10000 + i, cfg.hidden).double() for i in range(2 * cfg.num_layers + 1)]
    half, H, KVH, hd = cfg.rope_half_dim, cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    cos_t, sin_t = (torch.from_numpy(t).to(DEV).double().reshape(-1, half)
                    for t in pkg.rope_tables(_capacity(c), half, cfg.rope_theta))
    cache = [None] * cfg.num_layers

    def norm(x, g):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * g

    def rope(x, pos):
        a, b = x[..., :half], x[..., half:]
        cs, sn = (t[pos:pos + x.shape[0]].unsqueeze(1) for t in (cos_t, sin_t))
        return torch.cat((a * cs - b * sn, b * cs + a * sn), -1)

    def forward(ids, pos):
        """Logits of the last of the tokens `ids` at positions pos, pos + 1, ..."""
        x = embed[torch.as_tensor(ids, device=DEV)]
        t = x.shape[0]
        for l, (wq, wk, wv, wo, wg, wu, wd) in enumerate(mats):
            xn = norm(x, gam[2 * l])
            q, k, v = (xn @ wq).view(t, H, hd), (xn @ wk).view(t, KVH, hd), (xn @ wv).view(t, KVH, hd)
            if l % 4 == 3:
                q, k = rope(q, pos), rope(k, pos)
            if c["kv"] == "f16":             # what the cache holds is rounded
                k, v = k.half().double(), v.half().double()
            if cache[l] is not None:
                k, v = torch.cat((cache[l][0], k)), torch.cat((cache[l][1], v))
            cache[l] = (k, v)
            mask = torch.arange(pos + t, device=DEV)[None, :] > pos + torch.arange(t, device=DEV)[:, None]
            att = torch.empty_like(q)
            for i in range(H):
                sc = (q[:, i] @ k[:, i // (H // KVH)].t() / math.sqrt(hd)).masked_fill(mask, -math.inf)
                att[:, i] = torch.softmax(sc, -1) @ v[:, i // (H // KVH)]
            x = x + att.reshape(t, H * hd) @ wo
            xn = norm(x, gam[2 * l + 1])
            x = x + (torch.nn.functional.silu(xn @ wg) * (xn @ wu)) @ wd
        return embed @ norm(x[-1], gam[-1])

    return forward


def exact(case, seed):
    op, c = case["op"], case
    if op == "model":
        forward = _model64(c, seed)
        first = last = forward(_prompt(c, seed), 0)
        for i in range(c["steps"]):
            last = forward([int(last.argmax())], c["prompt"] + i)
        return dict(first=first, last=last, tokens=None)
    if op == "gemv":
        return _normal(seed, 2, c["k"]).double() @ _weight64(c["fmt"], seed, 1, c["k"], c["n"])
    if op == "mlp":
        k, n, x = c["k"], c["n"], _normal(seed, 5, c["k"]).double()
        xn = x / torch.sqrt((x * x).mean() + 1e-6) * _norm_gamma(seed, 4, k).double()
        a = torch.nn.functional.silu(xn @ _weight64(c["fmt"], seed, 1, k, n)) * (xn @ _weight64(c["fmt"], seed, 2, k, n))
        return a, a @ _weight64(c["fmt"], seed, 3, n, k)
    if op == "lm_head":
        return _weight64(c["fmt"], seed, 1, c["rows"], c["cols"]) @ _normal(seed, 2, c["cols"]).double()
    if op in ("attn_decode", "attn_prefill"):
        t, pos0 = (1, c["positions"] - 1) if op == "attn_decode" else (c["tokens"], c["pos0"])
        H, KVH, hd = c["heads"], c["kv_heads"], c["head_dim"]
        kv = torch.float16 if c["kv"] == "f16" else torch.float32
        q = _normal(seed, 1, t, H * hd).double().view(t, H, hd)
        k, v = (_normal(seed, i, pos0 + t, KVH * hd).to(kv).double().view(-1, KVH, hd) for i in (2, 3))
        mask = torch.arange(pos0 + t, device=DEV)[None, :] > pos0 + torch.arange(t, device=DEV)[:, None]
        out = torch.empty_like(q)
        for i in range(H):
            sc = (q[:, i] @ k[:, i // (H // KVH)].t() / math.sqrt(hd)).masked_fill(mask, -math.inf)
            out[:, i] = torch.softmax(sc, -1) @ v[:, i // (H // KVH)]
        return out.reshape(t, H * hd)
    if op == "gemm":
        return _normal(seed, 2, c["tokens"], c["k"]).double() @ _weight64(c["fmt"], seed, 1, c["k"], c["n"])
    return None
