"""The calls that a program on this framework makes, as timed cases.

A decoder served from Q8_0 weights spends its time in: the linears of one
decode token, of a batch of sequences and of a prompt; the attention of a
decode step and of a prompt; the blocks that chain them; the sampler; and the
other numerics a linear can be asked for (W8A8, the exact sums, per-row int8
and int4).  Each case is one such call (or one block or step) through
ferrum_hip's public functions on device buffers that a program would keep.

Shapes are the ones the repository's configurations, tests and bench use
(GPT-2 124M and medium, Qwen2-0.5B, the tiny GPT-2) and ragged neighbours of
them; values are theirs too: weights N(0, 0.02), activations N(0, 1).

exact() restates each call in float64 torch, the Q8_0 and per-row codecs
included, without the framework's code.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ferrum-cpu_amd"))
import ferrum_hip as fh  # noqa: E402

NUMERICS = {"w8a32": fh.W8A32, "w8a8": fh.W8A8, "w8a8_fast": fh.W8A8_FAST, "exact": fh.W8A32_EXACT}
# (outputs, inputs) of the linears of the three model families
LAYERS = [(2304, 768), (768, 768), (3072, 768), (768, 3072),          # GPT-2 124M
          (3072, 1024), (1024, 1024), (4096, 1024), (1024, 4096),     # GPT-2 medium
          (1152, 896), (896, 896), (9728, 896), (896, 4864),          # Qwen2-0.5B
          (384, 128), (128, 128), (512, 128), (128, 512)]             # tiny GPT-2
HEADS = [(50257, 768), (50257, 1024), (151936, 896), (4096, 128)]
GPT2 = {"tiny": dict(d=128, heads=4, layers=4, vocab=4096, context=256),
        "124m": dict(d=768, heads=12, layers=12, vocab=50257, context=1024),
        "medium": dict(d=1024, heads=16, layers=24, vocab=50257, context=1024)}
QWEN2 = dict(d=896, heads=14, kv=2, hd=64, ffn=4864)
LN_EPS, RMS_EPS = 1e-5, 1e-6


def listed():
    return [
        # one token's Q|K|V projection, the smallest call of a decode step
        {"name": "linear_token", "kind": "linear", "m": 1, "n": 2304, "k": 768, "numerics": "w8a32", "bias": True,
         "gelu": False},
        # the up projection with its GELU over one 128-id prompt (its last id is the first step's)
        {"name": "linear_prompt", "kind": "linear", "m": 127, "n": 3072, "k": 768, "numerics": "w8a32", "bias": True,
         "gelu": True},
        # the same over 32 prompts of 512 ids at GPT-2 medium: the largest call
        {"name": "linear_prefill", "kind": "linear", "m": 16352, "n": 4096, "k": 1024, "numerics": "w8a32",
         "bias": True, "gelu": False},
        # llama.cpp's numerics over one 512-id prompt
        {"name": "linear_w8a8", "kind": "linear", "m": 511, "n": 3072, "k": 1024, "numerics": "w8a8", "bias": True,
         "gelu": False},
        # the reference's own sums, bit for bit, over a prompt (the down projection: its longest sums)
        {"name": "linear_exact", "kind": "linear", "m": 127, "n": 768, "k": 3072, "numerics": "exact", "bias": True,
         "gelu": False},
        # a per-row int8 model: one decode token, and a per-row int4 model's prompt
        {"name": "qlinear_token", "kind": "qlinear", "m": 1, "n": 3072, "k": 768, "bits": 8, "bias": True},
        {"name": "qlinear_prompt", "kind": "qlinear", "m": 127, "n": 2304, "k": 768, "bits": 4, "bias": True},
        # one block of a batched decode step: 32 GPT-2 124M sequences, 64 Qwen2 ones
        {"name": "block_gpt2", "kind": "block", "family": "124m", "rows": 32, "pos": 255},
        {"name": "block_qwen2", "kind": "block", "family": "qwen2", "rows": 64, "pos": 511},
        # the attention of eight 300-id prompts
        {"name": "attention_prompt", "kind": "attention", "d": 768, "heads": 12, "seqs": 8, "rows": 300, "pos0": 0},
        # one token for each of 32 sequences, the run parameters of the GPT-2 configuration
        {"name": "sampler", "kind": "sampler", "rows": 32, "vocab": 50257, "gpt2": True, "temperature": 0.8,
         "top_k": 40, "top_p": 0.95, "penalty": 1.1, "recent": 256},
        # a whole single-sequence decode step: embedding, 12 blocks, head, sampler
        {"name": "step_gpt2", "kind": "step", "family": "124m", "pos": 255},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["qlinear"] * 2 + ["block"] * 2 + ["attention", "sampler", "step"])
    if kind == "linear":
        numerics = rng.choice(["w8a32", "w8a32", "w8a32", "w8a8", "w8a8_fast", "exact", "exact_f32"])
        exact = numerics.startswith("exact")
        m = _log(rng, 1, 256 if exact else 16352)
        n, k = rng.choice(LAYERS + (HEADS if m <= 64 else []))
        if rng.random() < 0.4:
            n -= rng.randint(1, 31)  # a ragged output width
        if rng.random() < 0.25:
            k -= 32 * rng.randint(1, 3)
        if numerics == "exact_f32" and rng.random() < 0.5:
            k -= rng.randint(1, 15)  # the rows that a file stores as F32 because they are no multiple of 32
        return {"kind": kind, "m": m, "n": n, "k": k, "numerics": numerics, "bias": rng.random() < 0.75,
                "gelu": numerics == "w8a32" and rng.random() < 0.3}
    if kind == "qlinear":
        m = 1 if rng.random() < 0.4 else _log(rng, 2, 512)
        n, k = rng.choice(LAYERS + (HEADS[:2] if m == 1 else []))
        return {"kind": kind, "m": m, "n": n - (rng.randint(1, 31) if rng.random() < 0.4 else 0),
                "k": k - (rng.randint(1, 60) if rng.random() < 0.25 else 0), "bits": rng.choice([4, 8]),
                "bias": rng.random() < 0.75}
    if kind == "block":
        return {"kind": kind, "family": rng.choice(["124m", "medium", "qwen2"]), "rows": _log(rng, 3, 64),
                "pos": _log(rng, 16, 1000)}
    if kind == "attention":
        d, heads = rng.choice([(768, 12), (1024, 16), (128, 4)])
        rows = _log(rng, 16, 128 if d == 128 else 900)
        seqs = _log(rng, 1, max(1, min(32, 16352 // rows)))
        return {"kind": kind, "d": d, "heads": heads, "seqs": seqs, "rows": rows,
                "pos0": rng.randint(1, 100) if rng.random() < 0.3 else 0}
    if kind == "sampler":
        return {"kind": kind, "rows": _log(rng, 1, 64), "vocab": rng.choice([4096, 32000, 50257, 151936]),
                "gpt2": rng.random() < 0.5, "temperature": rng.choice([0.0, 0.7, 0.8, 1.0]),
                "top_k": rng.choice([40, 50, 64]), "top_p": rng.choice([0.9, 0.95, 1.0]),
                "penalty": rng.choice([1.0, 1.05, 1.1]), "recent": _log(rng, 16, 1024)}
    family = rng.choice(["tiny", "124m", "medium"])
    return {"kind": kind, "family": family, "pos": _log(rng, 8, GPT2[family]["context"] - 1)}


# ---- weights and inputs ----------------------------------------------------

_context = []


def _ctx():
    """The program's one context."""
    if not _context:
        _context.append(fh.Context(0))
    return _context[0]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device="cuda") * std + mean


def _encode(x):
    """Rows of floats as Q8_0: f16 scales [rows, k / 32] and quants [rows, k / 32, 32]."""
    b = x.reshape(x.shape[0], -1, 32)
    top = b.abs().amax(dim=2)
    d = top / torch.full_like(top, 127.0)  # (a number as the divisor would be a product with its reciprocal)
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    t = (b * inv[:, :, None]).double()
    q = (torch.sign(t) * torch.floor(t.abs() + 0.5)).clamp(-128, 127)
    return d.to(torch.float16), q.to(torch.int8)


def _bytes(d, q):
    """The GGUF bytes of _encode's blocks."""
    return torch.cat([d.view(torch.uint8).reshape(*d.shape, 2), q.view(torch.uint8)], dim=2).contiguous()


def _wide(d, q):
    """The weights that Q8_0 blocks stand for, in float64."""
    return (d.double()[:, :, None] * q.double()).reshape(d.shape[0], -1)


def _q8(g, n, k):
    return _encode(_normal(g, n, k, std=0.02))


def _upload(blocks):
    raw, (n, kb) = _bytes(*blocks), blocks[0].shape
    torch.cuda.synchronize()  # the context works on its own stream
    w = fh.Q8_0Weight.upload_device(_ctx(), raw, n, kb * 32)
    _ctx().sync()
    return w


def _linear_inputs(case, seed):
    g = _generator(seed)
    m, n, k = case["m"], case["n"], case["k"]
    w = _normal(g, n, k, std=0.02) if case["numerics"] == "exact_f32" else _q8(g, n, k)
    return w, _normal(g, m, k), _normal(g, n, std=0.1) if case["bias"] else None


def _qlinear_inputs(case, seed):
    """Per-row symmetric levels of a [k, n] weight (int8: amax / 127, int4: amax / 7)."""
    g = _generator(seed)
    w = _normal(g, case["k"], case["n"], std=0.02)
    top = 127.0 if case["bits"] == 8 else 7.0
    scale = w.abs().amax(dim=1) / top
    level = torch.round(w / scale[:, None]).clamp(-top, top).to(torch.int8)
    return scale, level, _normal(g, case["m"], case["k"]), _normal(g, case["n"], std=0.1) if case["bias"] else None


def _packed(level, bits):
    """int8 levels as bytes; int4 as nibbles, the first half of the columns in the low ones."""
    if bits == 8:
        return level.view(torch.uint8).cpu().numpy()
    half = (level.shape[1] + 1) // 2
    u = (level & 15).to(torch.uint8)
    b = u[:, :half].clone()
    b[:, :level.shape[1] - half] |= u[:, half:] << 4
    return b.cpu().numpy()


def _block_inputs(case, seed):
    """One block's weights, the residual stream of its rows, their positions and caches."""
    g = _generator(seed)
    rows, pos = case["rows"], case["pos"]
    if case["family"] == "qwen2":
        c = QWEN2
        d, hd, heads, kv, ffn = c["d"], c["hd"], c["heads"], c["kv"], c["ffn"]
    else:
        d, heads = GPT2[case["family"]]["d"], GPT2[case["family"]]["heads"]
        hd, kv, ffn = 64, heads, 4 * d
    qkv = (heads + 2 * kv) * hd
    qwen = case["family"] == "qwen2"
    s = dict(d=d, hd=hd, heads=heads, kv=kv, ffn=ffn, width=qkv, qwen=qwen, rows=rows, capacity=pos + 1)
    s["qkv"], s["out"] = _q8(g, qkv, d), _q8(g, d, heads * hd)
    s["up"], s["down"] = _q8(g, 2 * ffn if qwen else ffn, d), _q8(g, d, ffn)
    s["qkv_b"] = _normal(g, qkv, std=0.02)
    if not qwen:
        s["out_b"], s["up_b"], s["down_b"] = (_normal(g, w, std=0.02) for w in (d, ffn, d))
        s["beta1"], s["beta2"] = _normal(g, d, std=0.02), _normal(g, d, std=0.02)
    s["gamma1"], s["gamma2"] = _normal(g, d, std=0.02, mean=1.0), _normal(g, d, std=0.02, mean=1.0)
    s["x"] = _normal(g, rows, d)
    # sequences of one batch are about as long as each other
    s["pos"] = torch.randint(pos - pos // 4, pos + 1, (rows,), generator=g, device="cuda", dtype=torch.int32)
    s["pos"][0] = pos
    s["k"] = _normal(g, rows, s["capacity"], kv * hd, std=0.5)
    s["v"] = _normal(g, rows, s["capacity"], kv * hd, std=0.5)
    return s


def _group_stats(x):
    """(mean, sum of squared deviations) of each 32 columns of each row, as a projection leaves them."""
    b = x.double().reshape(x.shape[0], -1, 32)
    mean = b.mean(dim=2)
    return torch.stack([mean, ((b - mean[:, :, None]) ** 2).sum(dim=2)], dim=2).float().contiguous()


def _attention_inputs(case, seed):
    g = _generator(seed)
    d, seqs, capacity = case["d"], case["seqs"], case["pos0"] + case["rows"]
    qkv = _normal(g, seqs * case["rows"], 3 * d, std=0.55)
    return qkv, _normal(g, seqs, capacity, d, std=0.5), _normal(g, seqs, capacity, d, std=0.5)


def _sampler_inputs(case, seed):
    g = _generator(seed)
    rows, vocab = case["rows"], case["vocab"]
    logits = _normal(g, rows, vocab, std=3.0)
    peaks = torch.randint(0, vocab, (5,), generator=g, device="cuda")
    if not case["gpt2"]:
        logits[:, peaks] += 12.0
    recent = torch.randint(0, vocab, (rows, case["recent"]), generator=g, device="cuda", dtype=torch.int32)
    recent[:, :3] = peaks[:3].to(torch.int32)
    offsets = torch.arange(0, (rows + 1) * case["recent"], case["recent"], device="cuda", dtype=torch.int32)
    draws = torch.randint(0, 2 ** 63 - 1, (rows,), generator=g, device="cuda", dtype=torch.int64)
    return logits, recent.contiguous(), offsets, draws


def _step_inputs(case, seed):
    """A GPT-2's blocks, its caches up to `pos` and the token at `pos`."""
    g, c = _generator(seed), GPT2[case["family"]]
    d, vocab = c["d"], c["vocab"]
    w = {"token": _q8(g, vocab, d), "position": _normal(g, c["context"], d, std=0.02),
         "lnf": (_normal(g, d, std=0.02, mean=1.0), _normal(g, d, std=0.02)), "blocks": []}
    for _ in range(c["layers"]):
        b = {"ln1": (_normal(g, d, std=0.02, mean=1.0), _normal(g, d, std=0.02)),
             "ln2": (_normal(g, d, std=0.02, mean=1.0), _normal(g, d, std=0.02))}
        for name, n, k in (("qkv", 3 * d, d), ("out", d, d), ("up", 4 * d, d), ("down", d, 4 * d)):
            b[name], b[name + "_b"] = _q8(g, n, k), _normal(g, n, std=0.02)
        b["k"], b["v"] = (_normal(g, c["context"], d, std=0.5) for _ in range(2))
        w["blocks"].append(b)
    w["id"] = torch.randint(0, vocab, (1,), generator=g, device="cuda", dtype=torch.int32)
    w["recent"] = torch.randint(0, vocab, (case["pos"] + 1,), generator=g, device="cuda", dtype=torch.int32)
    w["draw"] = torch.randint(0, 2 ** 63 - 1, (1,), generator=g, device="cuda", dtype=torch.int64)
    return w


def prepare(case, seed):
    s = dict(case)
    ctx = s["ctx"] = _ctx()
    kind = case["kind"]
    if kind == "linear":
        w, s["x"], s["b"] = _linear_inputs(case, seed)
        s["w"] = fh.Q8_0Weight.upload_f32(ctx, w.cpu().numpy()) if case["numerics"] == "exact_f32" else _upload(w)
        s["mode"] = NUMERICS[case["numerics"].replace("_f32", "")]
        s["y"] = torch.empty((case["m"], case["n"]), device="cuda")
    elif kind == "qlinear":
        scale, level, s["x"], s["b"] = _qlinear_inputs(case, seed)
        s["w"] = _QWeight(ctx, scale.cpu().numpy(), _packed(level, case["bits"]), case["k"], case["n"],
                          fh.QINT8 if case["bits"] == 8 else fh.QINT4)
        s["y"] = torch.empty((case["m"], case["n"]), device="cuda")
    elif kind == "block":
        s.update(_block_inputs(case, seed))
        if s["qwen"]:  # gate and up rows interleaved in groups of 32, as the model loader stores them for SwiGLU
            s["up"] = tuple(t.reshape(2, s["ffn"] // 32, 32, *t.shape[1:]).transpose(0, 1).reshape(t.shape)
                            .contiguous() for t in s["up"])
        for name in ("qkv", "out", "up", "down"):
            s[name] = _upload(s[name])
        s["stats"] = _group_stats(s["x"])
        rows, d = s["rows"], s["d"]
        s["qkv_y"], s["att"] = (torch.empty((rows, w), device="cuda") for w in (s["width"], s["heads"] * s["hd"]))
        s["x1"], s["x2"] = (torch.empty((rows, d), device="cuda") for _ in range(2))
        s["stats1"], s["stats2"] = (torch.empty((rows, d // 32, 2), device="cuda") for _ in range(2))
        s["mid"] = torch.empty((rows, s["ffn"]), device="cuda")
    elif kind == "attention":
        s["qkv"], s["k"], s["v"] = _attention_inputs(case, seed)
        s["out"] = torch.empty((case["seqs"] * case["rows"], case["d"]), device="cuda")
    elif kind == "sampler":
        s["logits"], s["ids"], s["offsets"], s["draws"] = _sampler_inputs(case, seed)
        s["params"] = fh.SamplingParams(case["temperature"], case["top_k"], case["top_p"], case["penalty"])
        s["out"] = torch.zeros(case["rows"], dtype=torch.int32, device="cuda")
    else:
        w, c = _step_inputs(case, seed), GPT2[case["family"]]
        host = {"token_embd_q8": _bytes(*w["token"]).cpu().numpy().ravel(), "position_embd": w["position"].cpu().numpy(),
                "lnf_g": w["lnf"][0].cpu().numpy(), "lnf_b": w["lnf"][1].cpu().numpy()}
        for i, b in enumerate(w["blocks"]):
            for name in ("ln1", "ln2"):
                host[f"blk{i}.{name}_g"], host[f"blk{i}.{name}_b"] = (t.cpu().numpy() for t in b[name])
            for name in ("qkv", "out", "up", "down"):
                host[f"blk{i}.{name}_q8"] = _bytes(*b[name]).cpu().numpy().ravel()
                host[f"blk{i}.{name}_b"] = b[name + "_b"].cpu().numpy()
        s["model"] = _Model(ctx, host, c)
        for b, mine in zip(w["blocks"], s["model"].m.blocks):
            mine["k"].copy_(b["k"])
            mine["v"].copy_(b["v"])
        s.update({name: w[name] for name in ("id", "recent", "draw")})
        s["offsets"] = torch.tensor([0, case["pos"] + 1], dtype=torch.int32, device="cuda")
        s["params"] = fh.SamplingParams(0.8, 40, 0.95, 1.1)
        s["next"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    ctx.sync()
    return s


class _QWeight(fh.QWeight):
    """Gives its device memory back with the state that holds it."""

    def __del__(self):
        self.free()


class _Model:
    """A GPT2Device that is freed with the state that holds it."""

    def __init__(self, ctx, weights, c):
        self.m = fh.GPT2Device.from_weights(ctx, weights, c["vocab"], c["d"], c["heads"], c["layers"], 4 * c["d"],
                                            c["context"])

    def __del__(self):
        self.m.free()


# ---- one pass --------------------------------------------------------------

def run(s):
    ctx, kind = s["ctx"], s["kind"]
    if kind == "linear":
        n = s["n"] if s["b"] is not None else 0
        if s["gelu"]:
            fh.linear_act_async(ctx, s["w"], s["x"], s["m"], s["k"], s["b"], n, s["y"], fh.ACT_GELU, s["mode"])
        else:
            fh.linear_forward_async(ctx, s["w"], s["x"], s["m"], s["k"], s["b"], n, s["y"], s["mode"])
        return s["y"]
    if kind == "qlinear":
        fh.qlinear_async(ctx, s["w"], s["x"], s["m"], s["k"], s["b"], s["n"] if s["b"] is not None else 0, s["y"])
        return s["y"]
    if kind == "block":
        return _run_block(s)
    if kind == "attention":
        fh.attention_prefill_seqs_async(ctx, s["qkv"], s["k"], s["v"], (s["pos0"] + s["rows"]) * s["d"],
                                        s["pos0"] + s["rows"], s["d"], s["heads"], s["pos0"], s["rows"], s["seqs"],
                                        s["out"])
        return {"out": s["out"], "k": s["k"], "v": s["v"]}
    if kind == "sampler":
        fh.sample_rows_async(ctx, s["logits"], s["rows"], s["vocab"], s["params"], s["ids"], s["offsets"], s["draws"],
                             s["out"], fh.LOGITS_GPT2_SOFTMAX if s["gpt2"] else fh.LOGITS_RAW)
        return s["out"]
    m = s["model"].m
    m.feed_async(s["id"], s["pos"])
    fh.sample_rows_async(ctx, m.z, 1, m.vocab, s["params"], s["recent"], s["offsets"], s["draw"], s["next"],
                         fh.LOGITS_GPT2_SOFTMAX)
    return {"scores": m.z, "id": s["next"], "k": [b["k"] for b in m.blocks], "v": [b["v"] for b in m.blocks]}


def _run_block(s):
    """GPT2Batch's and LlamaDevice's batched block: five launches from residual stream to residual stream."""
    ctx, rows, d, h, kv, hd, ffn = s["ctx"], s["rows"], s["d"], s["heads"], s["kv"], s["hd"], s["ffn"]
    top, q = s["capacity"] - 1, h * hd
    if s["qwen"]:
        fh.linear_normed_async(ctx, s["qkv"], s["x"], rows, d, s["stats"], s["gamma1"], None, RMS_EPS, True, s["qkv_b"],
                               s["width"], s["qkv_y"])
        fh.gqa_attention_rope_decode_async(ctx, s["qkv_y"], s["width"], rows, h, kv, hd, s["k"], s["v"], s["capacity"],
                                           s["pos"], top, hd, 1e6, fh.ROPE_NEOX, None, 1.0, s["att"])
        fh.linear_residual_async(ctx, s["out"], s["att"], rows, q, None, 0, s["x"], s["x1"], s["stats1"])
        fh.linear_normed_async(ctx, s["up"], s["x1"], rows, d, s["stats1"], s["gamma2"], None, RMS_EPS, True, None, 0,
                               s["mid"], fh.ACT_SWIGLU32)
        fh.linear_residual_async(ctx, s["down"], s["mid"], rows, ffn, None, 0, s["x1"], s["x2"], s["stats2"])
    else:
        fh.linear_normed_async(ctx, s["qkv"], s["x"], rows, d, s["stats"], s["gamma1"], s["beta1"], LN_EPS, False,
                               s["qkv_b"], s["width"], s["qkv_y"])
        fh.gqa_attention_decode_async(ctx, s["qkv_y"], s["width"], rows, h, kv, hd, s["k"], s["v"], s["capacity"],
                                      s["pos"], top, s["att"])
        fh.linear_residual_async(ctx, s["out"], s["att"], rows, q, s["out_b"], d, s["x"], s["x1"], s["stats1"])
        fh.linear_normed_async(ctx, s["up"], s["x1"], rows, d, s["stats1"], s["gamma2"], s["beta2"], LN_EPS, False,
                               s["up_b"], ffn, s["mid"], fh.ACT_GELU)
        fh.linear_residual_async(ctx, s["down"], s["mid"], rows, ffn, s["down_b"], d, s["x1"], s["x2"], s["stats2"])
    return {"x": s["x2"], "stats": s["stats2"], "k": s["k"], "v": s["v"]}


# ---- what a pass cannot do without -----------------------------------------

def _q8_bytes(n, k):
    return n * k * 34 // 32


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        w = 4 * n * k if case["numerics"] == "exact_f32" else _q8_bytes(n, k)
        return {"bytes": w + 4 * m * (n + k) + (4 * n if case["bias"] else 0), "flops": 2 * m * n * k}
    if kind == "qlinear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k * case["bits"] // 8 + 4 * k + 4 * m * (n + k) + (4 * n if case["bias"] else 0),
                "flops": 2 * m * n * k}
    if kind == "block":
        rows, seen = case["rows"], case["rows"] * (case["pos"] - case["pos"] // 8 + 1)
        if case["family"] == "qwen2":
            d, q, kv, ffn = QWEN2["d"], QWEN2["heads"] * QWEN2["hd"], QWEN2["kv"] * QWEN2["hd"], QWEN2["ffn"]
            shapes = [(q + 2 * kv, d), (d, q), (2 * ffn, d), (d, ffn)]
        else:
            d = GPT2[case["family"]]["d"]
            q = kv = d
            shapes = [(3 * d, d), (d, d), (4 * d, d), (d, 4 * d)]
        return {"bytes": sum(_q8_bytes(n, k) for n, k in shapes) + 8 * seen * kv + 8 * rows * (d + kv),
                "flops": 2 * rows * sum(n * k for n, k in shapes) + 4 * seen * q}
    if kind == "attention":
        d, seqs, rows, pos0 = case["d"], case["seqs"], case["rows"], case["pos0"]
        pairs = seqs * (rows * pos0 + rows * (rows + 1) // 2)
        return {"bytes": 4 * seqs * (3 * rows * d + 2 * pos0 * d + 2 * rows * d + rows * d), "flops": 4 * pairs * d}
    if kind == "sampler":
        return {"bytes": 4 * case["rows"] * (case["vocab"] + case["recent"] + 3), "flops": 4 * case["rows"] * case["vocab"]}
    c = GPT2[case["family"]]
    d, seen = c["d"], case["pos"] + 1
    weights = c["layers"] * _q8_bytes(12 * d, d) + _q8_bytes(c["vocab"], d)
    return {"bytes": weights + 8 * c["layers"] * seen * d + 4 * c["vocab"],
            "flops": 2 * (12 * c["layers"] * d * d + c["vocab"] * d) + 4 * c["layers"] * seen * d}


def tolerance(case):
    # Whole numbers, and the sums whose every bit the reference fixes.
    if case["kind"] in ("sampler", "qlinear") or case.get("numerics", "").startswith("exact"):
        return "exact"
    # float32 sums.  Against float64, over the ranges of draw(): linears 2.4e-7
    # (largest value 2.7e-6), attention 2.0e-7 (3.2e-6), blocks 1.0e-7 (8e-7;
    # their group statistics are sums of such values), steps 5.6e-7 (2.9e-6).
    # Two orders of the same sums are up to twice that apart.
    return {"linear": {"rel": 1e-6, "max": 1e-5}, "block": {"rel": 1e-6, "max": 1e-5},
            "attention": {"rel": 1e-6, "max": 1e-5}, "step": {"rel": 2e-6, "max": 1e-5}}[case["kind"]]


# ---- the same in float64 ---------------------------------------------------

def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(0.7978846 * (x + 0.044715 * x ** 3)))


def _norm(x, gamma, beta):
    """LayerNorm, or RmsNorm where there is no beta."""
    if beta is None:
        return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + RMS_EPS) * gamma.double()
    c = x - x.mean(dim=-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(dim=-1, keepdim=True) + LN_EPS) * gamma.double() + beta.double()


def _attend(q, k, v):
    """q [heads, r, hd], k and v [heads, n, hd]; query i sees the first n - r + i + 1 positions."""
    r, n = q.shape[1], k.shape[1]
    score = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[2])
    hidden = torch.ones((r, n), dtype=torch.bool, device=q.device).triu(n - r + 1)
    return torch.matmul(torch.softmax(score.masked_fill(hidden, -math.inf), dim=2), v)


def _split(x, heads):
    return x.reshape(x.shape[0], heads, -1).transpose(0, 1).contiguous()


def _rope(x, pos, heads, hd):
    """Pairs (i, i + hd / 2) of each head turned by pos / base^(2 i / hd); frequency and angle are float32 values."""
    freq = (1e6 ** (-2.0 * torch.arange(hd // 2, device=x.device, dtype=torch.float64) / hd)).float()
    theta = (pos.float()[:, None] * freq).double()[:, None, :]
    h = x.reshape(x.shape[0], heads, 2, hd // 2)
    a, b = h[:, :, 0], h[:, :, 1]
    c, t = torch.cos(theta), torch.sin(theta)
    return torch.stack([a * c - b * t, a * t + b * c], dim=2).reshape(x.shape)


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, x, b = _linear_inputs(case, seed)
        if case["numerics"].startswith("w8a8"):
            x = _wide(*_encode(x))
        y = x.double() @ (w.double() if case["numerics"] == "exact_f32" else _wide(*w)).T
        y = y if b is None else y + b.double()
        return _gelu(y) if case["gelu"] else y
    if kind == "qlinear":
        scale, level, x, b = _qlinear_inputs(case, seed)
        y = (x.double() * scale.double()) @ level.double()
        return y if b is None else y + b.double()
    if kind == "block":
        return _exact_block(_block_inputs(case, seed))
    if kind == "attention":
        qkv, k, v = (t.double() for t in _attention_inputs(case, seed))
        d, h, pos0 = case["d"], case["heads"], case["pos0"]
        qkv, out = qkv.reshape(case["seqs"], case["rows"], 3 * d), []
        k[:, pos0:], v[:, pos0:] = qkv[:, :, d:2 * d], qkv[:, :, 2 * d:]
        for i in range(case["seqs"]):
            a = _attend(_split(qkv[i, :, :d], h), _split(k[i], h), _split(v[i], h))
            out.append(a.transpose(0, 1).reshape(case["rows"], d))
        return {"out": torch.cat(out), "k": k, "v": v}
    if kind == "sampler":
        return None
    w, c, p = _step_inputs(case, seed), GPT2[case["family"]], case["pos"]
    d, h, table = c["d"], c["heads"], _wide(*w["token"])
    x = table[w["id"].long()].float().double() + w["position"].double()[p:p + 1]
    keys, values = [], []
    for b in w["blocks"]:
        qkv = _norm(x, *b["ln1"]) @ _wide(*b["qkv"]).T + b["qkv_b"].double()
        k, v = b["k"].double(), b["v"].double()
        k[p], v[p] = qkv[0, d:2 * d], qkv[0, 2 * d:]
        a = _attend(_split(qkv[:, :d], h), _split(k[:p + 1], h), _split(v[:p + 1], h)).reshape(1, d)
        x = x + a @ _wide(*b["out"]).T + b["out_b"].double()
        u = _gelu(_norm(x, *b["ln2"]) @ _wide(*b["up"]).T + b["up_b"].double())
        x = x + u @ _wide(*b["down"]).T + b["down_b"].double()
        keys.append(k)
        values.append(v)
    return {"scores": (_norm(x, *w["lnf"]) @ table.T)[0], "id": None, "k": keys, "v": values}


def _exact_block(s):
    h, kv, hd, q = s["heads"], s["kv"], s["hd"], s["heads"] * s["hd"]
    beta1, beta2 = s.get("beta1"), s.get("beta2")
    x = s["x"].double()
    qkv = _norm(x, s["gamma1"], beta1) @ _wide(*s["qkv"]).T + s["qkv_b"].double()
    qs, ks, vs = qkv[:, :q], qkv[:, q:q + kv * hd], qkv[:, q + kv * hd:]
    if s["qwen"]:
        qs, ks = _rope(qs, s["pos"], h, hd), _rope(ks, s["pos"], kv, hd)
    k, v, att = s["k"].double(), s["v"].double(), []
    for r, p in enumerate(s["pos"].tolist()):
        k[r, p], v[r, p] = ks[r], vs[r]
        kk, vv = (_split(t[r, :p + 1], kv).repeat_interleave(h // kv, dim=0) for t in (k, v))
        att.append(_attend(_split(qs[r:r + 1], h), kk, vv).reshape(1, q))
    x = x + torch.cat(att) @ _wide(*s["out"]).T + (0 if s["qwen"] else s["out_b"].double())
    u = _norm(x, s["gamma2"], beta2) @ _wide(*s["up"]).T
    if s["qwen"]:
        gate, up = u[:, :s["ffn"]], u[:, s["ffn"]:]
        u = gate / (1.0 + torch.exp(-gate)) * up
    else:
        u = _gelu(u + s["up_b"].double())
    x = x + u @ _wide(*s["down"]).T + (0 if s["qwen"] else s["down_b"].double())
    return {"x": x, "stats": None, "k": k, "v": v}
