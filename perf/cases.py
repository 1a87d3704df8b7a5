"""Timed workloads: what a program that serves a decoder with this library has it do,
each through the public entry points (tessera_amd.rules, tessera_amd.qwen3).

A case is a dict of plain values; `kind` picks the path:

  mlp       one SwiGLU MLP block, gate/up and down: bf16, e4m3 or block-form weights,
            from one decode row to a long prefill; f32 rows as the decoder's residual
            stream (norm before, residual added after) or bf16 rows as standalone products
  head      the unembedding of a batch's last rows and the greedy pick
  attend    decode attention over paged kept rows, one query a sequence
  step      the fused decode step: q/k norm, RoPE, append, attend
  flash     prefill attention over paged kept rows, prompts packed back to back
  moe       one MoE layer: routing, expert products, combine, shared expert
  generate  the whole Qwen3-shaped runner: a prompt prefilled, then greedy decode

Sizes are those of the benchmark's workloads (a Qwen3-0.6B-shaped decoder, Llama-3-8B-like
quantized products, a GLM-style MoE layer, paged GQA attention) and of the ranges around
them.
"""
import math

import numpy as np
import torch

from tessera_amd import rules
from tessera_amd.qwen3 import Qwen3, default_config

EPS = 1e-6
THETA = 1e6
D = 128  # head width of every attention path

# Block forms: codes a block, largest code magnitude, scale kind, code kind.
FORMS = {"q8_0": (32, 127.0, "f16", "i8"), "mxfp8": (32, 448.0, "e8m0", "e4m3"), "int4_g32": (32, 7.0, "f16", "nib"),
         "q4_0": (32, 7.0, "f16", "nib"), "nvfp4": (16, 6.0, "e4m3", "e2m1"), "mxfp4": (32, 6.0, "e8m0", "e2m1"),
         "int4_g128": (128, 7.0, "f16", "nib")}
BLOCK_BYTES = {"q8_0": 34, "mxfp8": 33, "int4_g32": 18, "q4_0": 18, "nvfp4": 9, "mxfp4": 17, "int4_g128": 66}


def listed():
    return [
        # One token through one layer's MLP of the Qwen3-0.6B shape: the smallest call,
        # launches and latency.
        {"name": "mlp_bf16_decode_1", "kind": "mlp", "m": 1, "hidden": 1024, "ffn": 3072, "w": "bf16", "x": "f32"},
        # A small serving batch against 8-bit weights of a Llama-3-8B-like MLP.
        {"name": "mlp_e4m3_decode_8", "kind": "mlp", "m": 8, "hidden": 4096, "ffn": 14336, "w": "e4m3", "x": "bf16"},
        # A serving batch against 4-bit block weights.
        {"name": "mlp_int4_decode_16", "kind": "mlp", "m": 16, "hidden": 4096, "ffn": 14336, "w": "int4_g32",
         "x": "f32"},
        # Prompts batched to 2048 rows, bf16 products of the Qwen3-0.6B shape.
        {"name": "mlp_bf16_prefill_2048", "kind": "mlp", "m": 2048, "hidden": 1024, "ffn": 3072, "w": "bf16",
         "x": "bf16"},
        # A ragged prompt batch through 8-bit weights.
        {"name": "mlp_e4m3_prefill_1000", "kind": "mlp", "m": 1000, "hidden": 4096, "ffn": 14336, "w": "e4m3",
         "x": "bf16"},
        # Logits and greedy picks of 16 sequences' last rows.
        {"name": "head_16", "kind": "head", "m": 16, "hidden": 1024, "vocab": 151936, "w": "bf16"},
        # Decode attention of a loaded server: 32 sequences of 512..8192 kept rows.
        {"name": "attend_32x8192", "kind": "attend", "rows": 32, "least": 512, "most": 8192, "heads": 16,
         "kv_heads": 8, "page": 16, "back": 0},
        # The fused decode step of a few short chats.
        {"name": "step_8x1000", "kind": "step", "rows": 8, "least": 100, "most": 1000, "heads": 16, "kv_heads": 8,
         "page": 16, "back": 0},
        # Prefill attention: four prompts of 2048.
        {"name": "flash_4x2048", "kind": "flash", "seqs": 4, "least": 2048, "most": 2048, "heads": 16, "kv_heads": 8,
         "page": 16, "back": 0, "q": "bf16"},
        # One MoE layer over a prefill batch.
        {"name": "moe_4096", "kind": "moe", "tokens": 4096, "hidden": 4096, "ffn": 1536, "experts": 128, "top": 8,
         "shared": True, "x": "bf16"},
        # The same layer over one decode batch: most experts see a row or two.
        {"name": "moe_16", "kind": "moe", "tokens": 16, "hidden": 4096, "ffn": 1536, "experts": 128, "top": 8,
         "shared": True, "x": "bf16"},
        # The whole decoder: a 1000-token prompt answered with 16 tokens.
        {"name": "generate_1000_16", "kind": "generate", "prompt": 1000, "steps": 16, "hidden": 1024, "ffn": 3072,
         "layers": 28, "heads": 16, "kv_heads": 8, "vocab": 151936},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "mlp", "head", "attend", "step", "flash", "moe", "moe", "generate"])
    if kind == "mlp":
        w = rng.choice(["bf16", "bf16", "e4m3", "e4m3", "q8_0", "mxfp8", "int4_g32", "q4_0", "nvfp4", "mxfp4",
                        "int4_g128"])
        unit = 512 if w == "int4_g128" else 128
        hidden = unit * _log(rng, 1024 // unit, 4096 // unit)
        ffn = unit * _log(rng, 2048 // unit, 14336 // unit)
        return {"kind": kind, "m": _log(rng, 1, 2048 if w in ("bf16", "e4m3") else 512), "hidden": hidden, "ffn": ffn,
                "w": w, "x": rng.choice(["f32", "bf16"])}
    if kind == "head":
        return {"kind": kind, "m": _log(rng, 1, 64), "hidden": 128 * _log(rng, 8, 32),
                "vocab": rng.choice([32000, 49152, 100277, 151936]), "w": rng.choice(["bf16", "bf16", "e4m3"])}
    heads, kv = rng.choice([(16, 8), (32, 8), (16, 2), (8, 8)])
    if kind in ("attend", "step"):
        most = _log(rng, 64, 8192)
        rows = _log(rng, 1, max(1, min(64, 262144 // most)))
        return {"kind": kind, "rows": rows, "least": max(1, int(most * rng.uniform(0.05, 1))), "most": most,
                "heads": heads, "kv_heads": kv, "page": rng.choice([16, 16, 64]),
                "back": rng.choice([0, 0, 0, 1024])}
    if kind == "flash":
        most = _log(rng, 32, 4096)
        seqs = _log(rng, 1, max(1, min(16, 8192 // most)))
        return {"kind": kind, "seqs": seqs, "least": max(1, int(most * rng.uniform(0.1, 1))), "most": most,
                "heads": heads, "kv_heads": kv, "page": rng.choice([16, 16, 64]), "back": rng.choice([0, 0, 0, 1024]),
                "q": rng.choice(["bf16", "f32"])}
    if kind == "moe":
        experts = rng.choice([16, 32, 64, 128])
        return {"kind": kind, "tokens": _log(rng, 1, 4096), "hidden": 128 * _log(rng, 8, 32),
                "ffn": 64 * _log(rng, 8, 24), "experts": experts, "top": rng.choice([2, 4, 8]),
                "shared": rng.choice([True, False]), "x": rng.choice(["bf16", "bf16", "f32"])}
    hidden = rng.choice([512, 1024, 1024, 2048])
    return {"kind": kind, "prompt": _log(rng, 8, 1000), "steps": _log(rng, 1, 16), "hidden": hidden,
            "ffn": hidden * 3, "layers": rng.choice([4, 8, 16]), "heads": 16, "kv_heads": 8,
            "vocab": rng.choice([32000, 151936])}


# --------------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, std=1.0, dtype=torch.float32):
    t = torch.randn(shape, device="cuda", generator=g, dtype=dtype)
    return t.mul_(std) if std != 1.0 else t


def _e2m1_codes(v):
    """Nearest e2m1 code of |v| <= 6, sign in bit 3."""
    mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=v.device)
    return (torch.bucketize(v.abs(), mids) + 8 * (v < 0)).to(torch.uint8)


def _block_pack(form, w):
    """Weights [n, k] as the packed tensor of a block form (absmax scales, nearest codes),
    and the f32 values the packed tensor holds."""
    B, top, scale_kind, code_kind = FORMS[form]
    n, k = w.shape
    v = w.view(n, k // B, B)
    s = v.abs().amax(2, keepdim=True) / top
    head = None
    if scale_kind == "f16":
        s16 = s.to(torch.float16)
        s, sb = s16.float(), s16.view(torch.uint8).view(n, k // B, 2)
    elif scale_kind == "e8m0":
        e = torch.ceil(torch.log2(s.clamp_min(2.0 ** -100))).clamp(-126, 127)
        s, sb = torch.exp2(e), (e + 127).to(torch.uint8)
    else:  # e4m3 scales under one f32 head
        head = (s.amax() / 448.0).view(1)
        s8 = (s / head).to(torch.float8_e4m3fn)
        s, sb = s8.float() * head, s8.view(torch.uint8)
    q = v / s.clamp_min(1e-30)
    if code_kind == "i8":
        c = q.round_().clamp_(-127, 127)
        value, codes = c, c.to(torch.int8).view(torch.uint8)
    elif code_kind == "e4m3":
        c8 = q.clamp_(-448, 448).to(torch.float8_e4m3fn)
        value, codes = c8.float(), c8.view(torch.uint8)
    else:
        if code_kind == "nib":
            value = q.round_().clamp_(-8, 7)
            nib = (value + 8).to(torch.uint8)
        else:
            nib = _e2m1_codes(q)
            table = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], device=w.device)
            value = table[nib.long()]
        lo, hi = (nib[:, :, :B // 2], nib[:, :, B // 2:]) if form == "q4_0" else (nib[:, :, 0::2], nib[:, :, 1::2])
        codes = lo | (hi << 4)
    packed = torch.cat([sb, codes], 2).reshape(-1)
    if head is not None:
        packed = torch.cat([head.view(torch.uint8), packed])
    return packed.contiguous(), (value * s).view(n, k)


def _weight(g, form, n, k, std=0.02):
    """(what the product takes: w, w_scale), (the f32 values it holds)."""
    w = _normal(g, (n, k), std)
    if form == "bf16":
        w = w.to(torch.bfloat16)
        return (w, None), w
    if form == "e4m3":
        scale = (w.abs().amax(1) / 448.0).to(torch.bfloat16)
        codes = (w / scale.float()[:, None]).to(torch.float8_e4m3fn)
        return (codes.view(torch.uint8), scale), (codes, scale)
    return _block_pack(form, w)


def _wide(held):
    """The held weights in 64 bits."""
    if isinstance(held, tuple):
        return held[0].float().double() * held[1].double()[:, None]
    return held.double()


def _spread(case, n):
    """n whole numbers from `most` down to `least`, in no order of size."""
    most, least = case["most"], case["least"]
    v = [most - (most - least) * i // max(1, n - 1) for i in range(n)]
    return [v[(i * 7) % n] if n % 7 else v[i] for i in range(n)]


def _kept(case, g, seed, lens):
    """Paged kept rows: K, V and a shuffled page table for one slot a sequence."""
    page = case["page"]
    kept_pages = -(-case["most"] // page)
    total = len(lens) * kept_pages
    perm = torch.from_numpy(np.random.default_rng(seed).permutation(total).astype(np.int32)).cuda()
    k = _normal(g, (total * page, case["kv_heads"], D), dtype=torch.bfloat16)
    v = _normal(g, (total * page, case["kv_heads"], D), dtype=torch.bfloat16)
    return {"k": k, "v": v, "table": perm, "kept_pages": kept_pages, "page": page, "keys": kept_pages * page}


def _back(case):
    return case.get("back") or 0xFFFFFFFF


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def _config(case):
    return default_config(vocab=case["vocab"], hidden=case["hidden"], ffn=case["ffn"], layers=case["layers"],
                          heads=case["heads"], kv_heads=case["kv_heads"], eps=EPS, theta=THETA,
                          max_prompt=case["prompt"], max_context=case["prompt"] + case["steps"] + 1)


def _prompt(case, seed):
    return np.random.default_rng(seed).integers(0, case["vocab"], case["prompt"]).astype(np.uint32)


def _mlp_inputs(case, seed):
    g, H, F, w = _gen(seed), case["hidden"], case["ffn"], case["w"]
    s = {"x": _normal(g, (case["m"], H), dtype=torch.bfloat16 if case["x"] == "bf16" else torch.float32)}
    s["gain"] = 1.0 + _normal(g, (H,), 0.02)
    held = {}
    if w in FORMS and case["m"] <= 4:  # the few-row block product takes no gate/up pair
        s["gate"], held["gate"] = _weight(g, w, F, H)
        s["up"], held["up"] = _weight(g, w, F, H)
    else:
        s["gate_up"], held["gate_up"] = _weight(g, w, 2 * F, H)
    s["down"], held["down"] = _weight(g, w, H, F)
    return s, held


def _head_inputs(case, seed):
    g = _gen(seed)
    w, held = _weight(g, case["w"], case["vocab"], case["hidden"])
    return {"x": _normal(g, (case["m"], case["hidden"])), "gain": 1.0 + _normal(g, (case["hidden"],), 0.02),
            "w": w}, held


def _moe_inputs(case, seed):
    g, H, F, E = _gen(seed), case["hidden"], case["ffn"], case["experts"]
    bf = torch.bfloat16
    s = {"h": _normal(g, (case["tokens"], H), dtype=bf if case["x"] == "bf16" else torch.float32),
         "router": _normal(g, (E, H), 1.0 / math.sqrt(H), bf),
         "w_in": _normal(g, (E, 2 * F, H), 0.02, bf), "w_out": _normal(g, (E, H, F), 0.02, bf),
         "shared_in": None, "shared_out": None}
    if case["shared"]:
        s["shared_in"], s["shared_out"] = _normal(g, (2 * F, H), 0.02, bf), _normal(g, (H, F), 0.02, bf)
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        return {"case": case, **_mlp_inputs(case, seed)[0]}
    if kind == "head":
        return {"case": case, **_head_inputs(case, seed)[0]}
    if kind == "moe":
        return {"case": case, **_moe_inputs(case, seed)}
    if kind == "generate":
        return {"case": case, "model": Qwen3(_config(case), seed=seed), "prompt": _prompt(case, seed)}
    g = _gen(seed)
    if kind == "flash":
        lens = _spread(case, case["seqs"])
        s = _kept(case, g, seed, lens)
        s["q"] = _normal(g, (sum(lens), case["heads"], D),
                         dtype=torch.bfloat16 if case["q"] == "bf16" else torch.float32)
        s["slots"] = _i32([i for i, n in enumerate(lens) for _ in range(n)])
        s["positions"] = _i32([p for n in lens for p in range(n)])
        return {"case": case, **s}
    lens = _spread(case, case["rows"])
    s = _kept(case, g, seed, lens)
    s["slots"], s["positions"] = _i32(list(range(len(lens)))), _i32([n - 1 for n in lens])
    if kind == "attend":
        s["q"] = _normal(g, (len(lens), case["heads"], D))
    else:
        s["qkv"] = _normal(g, (len(lens), (case["heads"] + 2 * case["kv_heads"]) * D))
        s["q_gain"], s["k_gain"] = 1.0 + _normal(g, (D,), 0.02), 1.0 + _normal(g, (D,), 0.02)
        s["angles"] = rules.rope_table(s["keys"], THETA)
    return {"case": case, **s}


# --------------------------------------------------------------------------- one pass


def _product(s, x, name, **kw):
    w = s["case"]["w"]
    if w in FORMS:
        H, F = s["case"]["hidden"], s["case"]["ffn"]
        return rules.linear(x, s[name], w_form=w, rows={"gate_up": 2 * F, "gate": F, "up": F, "down": H}[name], **kw)
    return rules.linear(x, s[name][0], w_scale=s[name][1], **kw)


def _run_mlp(s):
    case, x = s["case"], s["x"]
    m, out = case["m"], torch.bfloat16 if case["x"] == "bf16" else torch.float32
    rows, res, norm = x, {}, {}
    if case["x"] == "f32":
        res = {"a0": x}
        if case["w"] in FORMS or m > 16:
            rows = rules.rms_norm(x, s["gain"], EPS)
        else:
            norm = {"gain": s["gain"], "eps": EPS}
    if "gate" in s:
        gate, up = _product(s, rows, "gate"), _product(s, rows, "up")
        h = rules.map(gate, ["silu", "mul"], [up])
    else:
        h = _product(s, rows, "gate_up", silu_mul=True, out_dtype=out, **norm)
    return {"h": h, "out": _product(s, h, "down", out_dtype=out, **res)}


def _run_head(s):
    x, (w, scale), m = s["x"], s["w"], s["case"]["m"]
    if m <= 4 and scale is None:
        logits, ids = rules.linear_argmax(x, w, gain=s["gain"], eps=EPS)
        return {"logits": logits, "ids": ids}
    if m <= 16:
        logits = rules.linear(x, w, w_scale=scale, gain=s["gain"], eps=EPS)
    else:
        logits = rules.linear(rules.rms_norm(x, s["gain"], EPS), w, w_scale=scale)
    return {"logits": logits, "ids": rules.argmax(logits)}


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "mlp":
        return _run_mlp(s)
    if kind == "head":
        return _run_head(s)
    if kind == "moe":
        y, ids, gates = rules.moe_layer(s["h"], s["router"], s["w_in"], s["w_out"], top=case["top"],
                                        shared_in=s["shared_in"], shared_out=s["shared_out"])
        return {"y": y, "ids": ids, "gates": gates}
    if kind == "generate":
        s["model"].prefill(s["prompt"])
        tokens = s["model"].decode(case["steps"])
        return {"logits": s["model"].logits(), "tokens": tokens.astype(np.int64)}
    kept = {"keys": s["keys"], "scale": D ** -0.5, "table": s["table"], "kept_pages": s["kept_pages"],
            "page": s["page"], "back": _back(case), "max_position": case["most"] - 1}
    if kind == "attend":
        return rules.attend_rows(s["q"], s["k"], s["v"], s["slots"], s["positions"], **kept)
    if kind == "flash":
        return rules.flash_rows(s["q"], s["k"], s["v"], s["slots"], s["positions"], **kept)
    out = rules.attend_step(s["qkv"], s["q_gain"], s["k_gain"], s["k"], s["v"], s["slots"], s["positions"],
                            heads=case["heads"], eps=EPS, theta=THETA, angles=s["angles"], **kept)
    return {"out": out, "k": s["k"], "v": s["v"]}


# --------------------------------------------------------------------------- what it costs


def _weight_bytes(form, n, k):
    if form == "bf16":
        return 2 * n * k
    if form == "e4m3":
        return n * k + 2 * n
    return n * k // FORMS[form][0] * BLOCK_BYTES[form] + (4 if form == "nvfp4" else 0)


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        m, H, F, e = case["m"], case["hidden"], case["ffn"], 2 if case["x"] == "bf16" else 4
        return {"bytes": _weight_bytes(case["w"], 2 * F, H) + _weight_bytes(case["w"], H, F) + m * (2 * H + F) * e,
                "flops": 6 * m * H * F}
    if kind == "head":
        m, H, V = case["m"], case["hidden"], case["vocab"]
        return {"bytes": _weight_bytes(case["w"], V, H) + 4 * m * (H + V), "flops": 2 * m * H * V}
    if kind == "moe":
        t, H, F, E, top = (case[n] for n in ("tokens", "hidden", "ffn", "experts", "top"))
        met = E * (1 - (1 - top / E) ** t)  # experts that a token picks, on average
        rows = t * top + (t if case["shared"] else 0)
        return {"bytes": (met + case["shared"]) * 6 * H * F + 2 * E * H + t * H * (6 if case["x"] == "bf16" else 8)
                + 8 * t * top,
                "flops": 6 * rows * H * F + 2 * t * E * H}
    heads, kv = case["heads"], case["kv_heads"]
    back = _back(case)
    if kind == "generate":
        H, F, L, V, P, S = (case[n] for n in ("hidden", "ffn", "layers", "vocab", "prompt", "steps"))
        layer = H * (heads + 2 * kv) * D + heads * D * H + 3 * H * F
        ctx = sum(P + i + 1 for i in range(S))
        pairs = P * (P + 1) // 2 + ctx
        # A prefill reads every weight once, each decode step too; kept rows are read per step.
        return {"bytes": (S + 1) * 2 * (L * layer + V * H) + L * 4 * kv * D * (ctx + P + S),
                "flops": 2 * (P + S) * L * layer + 2 * (S + 1) * V * H + 4 * L * heads * D * pairs}
    if kind == "flash":
        lens = _spread(case, case["seqs"])
        pairs = sum(n * (n + 1) // 2 if n <= back else back * (back + 1) // 2 + (n - back) * (back + 1) for n in lens)
        e = 2 if case["q"] == "bf16" else 4
        return {"bytes": sum(lens) * D * (kv * 4 + heads * (e + 4)), "flops": 4 * D * heads * pairs}
    lens = [min(n, back + 1) for n in _spread(case, case["rows"])]
    return {"bytes": sum(lens) * kv * D * 4 + case["rows"] * D * 4 * (2 * heads + (2 * kv if kind == "step" else 0)),
            "flops": 4 * D * heads * sum(lens)}


def tolerance(case):
    """About four times what each path was measured off `exact`, by what it rounds."""
    kind = case["kind"]
    if kind == "mlp":  # bf16 rows: h and out rounded to bf16 (0.0024); f32 rows enter as 16-bit pairs (4e-6)
        return {"rel": 1e-2, "max": 0.05} if case["x"] == "bf16" else {"rel": 1.5e-5, "max": 3e-4}
    if kind == "head":  # 2.5e-6
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "moe":  # silu(g) u is kept in bf16 between the expert products (0.0017); a tied pick may change a row
        return {"rel": 7e-3, "max": 0.5, "differ": 0.002}
    if kind == "generate":  # kept rows are bf16: a rounding that flips travels on (0.0006 to 0.0014)
        return {"rel": 6e-3, "max": 0.1}
    if kind == "flash":  # bf16 q: P rounded to bf16 once (0.0013); f32 q: P in two parts (3e-6)
        return {"rel": 5e-3, "max": 0.1} if case["q"] == "bf16" else {"rel": 1.2e-5, "max": 3e-4}
    if kind == "attend":  # 2.5e-6
        return {"rel": 1e-5, "max": 3e-4}
    # step: f32 angles of positions in the thousands (3.6e-5); a kept row's value may round the other way
    return {"rel": 1.5e-4, "max": 3e-2}


# --------------------------------------------------------------------------- in 64 bits


def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _rms(x, gain, eps=EPS):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * gain.double()


def _rope(x, positions):
    """Halves pairs of x [rows, heads, D]."""
    j = torch.arange(D // 2, device=x.device, dtype=torch.float64)
    a = positions.double()[:, None] * THETA ** (-2 * j / D)
    c, n = a.cos()[:, None], a.sin()[:, None]
    lo, hi = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([lo * c - hi * n, hi * c + lo * n], -1)


def _attention(q, k, v, first, back):
    """Queries [n, heads, D] at positions first.. over keys [t, kv, D], causal and windowed."""
    n, heads, _ = q.shape
    t, kv = k.shape[:2]
    pos = torch.arange(first, first + n, device=q.device)[:, None]
    key = torch.arange(t, device=q.device)[None]
    hidden = (key > pos) | (key < pos - back)
    out = torch.empty_like(q)
    for h in range(heads):
        c = h // (heads // kv)
        p = (q[:, h] @ k[:, c].T * D ** -0.5).masked_fill_(hidden, -math.inf).softmax(1)
        out[:, h] = p @ v[:, c]
    return out


def _kept_rows(s, slot, n):
    """The kept rows of positions 0..n-1 of a slot."""
    page = s["page"]
    p = torch.arange(n, device="cuda")
    return s["table"].long()[slot * s["kept_pages"] + p // page] * page + p % page


def _exact_generate(case, seed):
    """The decoder in 64 bits over the runner's weights; kept rows are bf16, as stored."""
    model = Qwen3(_config(case), seed=seed)
    H, F, heads, kv = case["hidden"], case["ffn"], case["heads"], case["kv_heads"]

    def get(name, layer=0, shape=None):
        a = torch.from_numpy(model.read(name, layer))
        a = a.view(torch.int16).view(torch.bfloat16) if a.dtype == torch.uint16 else a
        a = a.cuda().double()
        return a.view(shape) if shape else a

    names = {"ln1": None, "qkv": (-1, H), "q_norm": None, "k_norm": None, "o": (H, -1), "ln2": None,
             "gate_up": (-1, H), "down": (H, F)}
    layers = [{n: get(n, l, sh) for n, sh in names.items()} for l in range(case["layers"])]
    embed, norm = get("embed", 0, (-1, H)), get("norm")
    model.close()
    kept = [None] * case["layers"]

    def forward(tokens, first):
        x = embed[torch.from_numpy(np.asarray(tokens, np.int64)).cuda()]
        pos = torch.arange(first, first + len(tokens), device="cuda")
        for l, w in enumerate(layers):
            qkv = (_rms(x, w["ln1"]) @ w["qkv"].T).view(len(tokens), heads + 2 * kv, D)
            q = _rope(_rms(qkv[:, :heads], w["q_norm"]), pos)
            new = [_rope(_rms(qkv[:, heads:heads + kv], w["k_norm"]), pos), qkv[:, heads + kv:]]
            new = [a.float().to(torch.bfloat16).double() for a in new]
            kept[l] = new if first == 0 else [torch.cat(p) for p in zip(kept[l], new)]
            x = x + _attention(q, *kept[l], first, 1 << 40).reshape(len(tokens), -1) @ w["o"].T
            gu = _rms(x, w["ln2"]) @ w["gate_up"].T
            x = x + _silu(gu[:, :F]) * gu[:, F:] @ w["down"].T
        return (_rms(x[-1:], norm) @ embed.T)[0]

    tokens = _prompt(case, seed).tolist()
    logits = forward(tokens, 0)
    picked = []
    for i in range(case["steps"]):
        token = int(logits.argmax())
        logits = forward([token], case["prompt"] + i)
        picked.append(int(logits.argmax()))
    return {"logits": logits, "tokens": np.array(picked, np.int64)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "generate":
        return _exact_generate(case, seed)
    if kind == "mlp":
        s, held = _mlp_inputs(case, seed)
        x = s["x"].double()
        rows = _rms(x, s["gain"]) if case["x"] == "f32" else x
        if "gate" in held:
            h = _silu(rows @ _wide(held["gate"]).T) * (rows @ _wide(held["up"]).T)
        else:
            gu = rows @ _wide(held["gate_up"]).T
            h = _silu(gu[:, :case["ffn"]]) * gu[:, case["ffn"]:]
        out = h @ _wide(held["down"]).T
        return {"h": h, "out": out + x if case["x"] == "f32" else out}
    if kind == "head":
        s, held = _head_inputs(case, seed)
        logits = _rms(s["x"].double(), s["gain"]) @ _wide(held).T
        return {"logits": logits, "ids": None}
    if kind == "moe":
        s = _moe_inputs(case, seed)
        h, F = s["h"].double(), case["ffn"]
        scores = h @ s["router"].double().T
        top, ids = scores.topk(case["top"], 1)
        gates = top.softmax(1)
        y = torch.zeros_like(h)
        for e in range(case["experts"]):
            row, pick = (ids == e).nonzero(as_tuple=True)
            if len(row):
                gu = h[row] @ s["w_in"][e].double().T
                y.index_add_(0, row, gates[row, pick, None] * ((_silu(gu[:, :F]) * gu[:, F:]) @ s["w_out"][e].double().T))
        if case["shared"]:
            gu = h @ s["shared_in"].double().T
            y += (_silu(gu[:, :F]) * gu[:, F:]) @ s["shared_out"].double().T
        return {"y": y, "ids": None, "gates": gates}
    s, back = prepare(case, seed), _back(case)
    if kind == "flash":
        out, at = [], 0
        for i, n in enumerate(_spread(case, case["seqs"])):
            r = _kept_rows(s, i, n)
            out.append(_attention(s["q"][at:at + n].double(), s["k"][r].double(), s["v"][r].double(), 0, back))
            at += n
        return torch.cat(out)
    heads, kv = case["heads"], case["kv_heads"]
    k, v = s["k"].double(), s["v"].double()
    q = s["q"].double() if kind == "attend" else None
    lens = _spread(case, case["rows"])
    if kind == "step":
        qkv = s["qkv"].double().view(len(lens), heads + 2 * kv, D)
        q = _rope(_rms(qkv[:, :heads], s["q_gain"]), s["positions"])
        new = _rope(_rms(qkv[:, heads:heads + kv], s["k_gain"]), s["positions"])
        for i, n in enumerate(lens):
            at = _kept_rows(s, i, n)[-1]
            k[at] = new[i].float().to(torch.bfloat16).double()
            v[at] = qkv[i, heads + kv:].float().to(torch.bfloat16).double()
    out = torch.empty(len(lens), heads, D, dtype=torch.float64, device="cuda")
    for i, n in enumerate(lens):
        r = _kept_rows(s, i, n)
        out[i] = _attention(q[i:i + 1], k[r], v[r], n - 1, back)[0]
    return out if kind == "attend" else {"out": out, "k": k, "v": v}
