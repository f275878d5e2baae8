"""What a user of this framework has it do, as cases that can be timed.

The engine that this framework serves runs, per transformer layer and call: the
norms, the rotary embedding and the router logits ("glue"), the W4A16
projections of the attention and of the shared MLP ("dense"), the Token-Union
MoE ("moe"), and once per call the lm_head with the final softcap ("lm_head").
Each of these is a case kind here, through the public entry points of
gemmainfer_amd.ops and the drop-in module gemmainfer_csrc.

The row count M of a call is 1 for a decoded token, up to 8 when draft tokens
are verified, a few tens for a batch of sequences or a short prompt, and
hundreds to thousands for a prompt's prefill.  Shapes are those of the
benchmark and the tests: hidden 2816, 128 experts, top-8, expert width 704,
vocabulary 262144, group sizes 64 (checkpoints) and 128 (benchmark).
"""
import math

import torch

import gemmainfer_csrc
from gemmainfer_amd import ops

DEV = "cuda:0"
H, E, I, TOP_K = 2816, 128, 704, 8
VOCAB = 262144
CAP = 30.0
EPS = 1e-6
MLP = 2112
# attention shapes: (heads, kv heads, head width); a global layer's values are its keys
ATTN = {"sliding": (16, 8, 256), "global": (16, 2, 512)}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
SCALE_STD = 0.02


def listed():
    return [
        # the norms, the rotary embedding and the router logits of one layer for a prompt of ordinary length
        {"name": "glue_prompt", "kind": "glue", "M": 300, "layer": "sliding"},
        # one decoded token: the projections of one layer, where launches and latency are all there is
        {"name": "dense_decode", "kind": "dense", "M": 1, "layer": "sliding", "gs": 64, "dtype": "bf16"},
        # six draft tokens and one more, verified in one call
        {"name": "dense_verify", "kind": "dense", "M": 7, "layer": "sliding", "gs": 64, "dtype": "bf16"},
        # a short prompt of a ragged length
        {"name": "dense_short_prompt", "kind": "dense", "M": 61, "layer": "global", "gs": 64, "dtype": "bf16"},
        # a long prompt
        {"name": "dense_prefill", "kind": "dense", "M": 2048, "layer": "sliding", "gs": 64, "dtype": "bf16"},
        # one decoded token through the experts
        {"name": "moe_decode", "kind": "moe", "M": 1, "gs": 64, "dtype": "bf16", "entry": "layer", "noise": 0.0},
        # a verify call through the drop-in module: seven tokens whose experts overlap
        {"name": "moe_verify", "kind": "moe", "M": 7, "gs": 64, "dtype": "bf16", "entry": "dropin", "noise": 0.5},
        # a batch of decoded tokens, or a short prompt
        {"name": "moe_batch", "kind": "moe", "M": 29, "gs": 64, "dtype": "bf16", "entry": "layer", "noise": 0.0},
        # a prompt of 512 tokens, the benchmark's prefill
        {"name": "moe_prefill", "kind": "moe", "M": 512, "gs": 128, "dtype": "bf16", "entry": "layer", "noise": 0.0},
        # a long prompt of an odd length
        {"name": "moe_long_prefill", "kind": "moe", "M": 1999, "gs": 64, "dtype": "bf16", "entry": "layer",
         "noise": 0.0},
        # a prompt of an engine that runs in fp16, through the drop-in module
        {"name": "moe_fp16_prompt", "kind": "moe", "M": 200, "gs": 64, "dtype": "fp16", "entry": "dropin",
         "noise": 0.0},
        # the logits of a verify call, softcapped
        {"name": "lm_head_verify", "kind": "lm_head", "M": 6, "N": VOCAB, "gs": 128, "cap": CAP},
    ]


def _rows(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["glue", "dense", "dense", "dense", "moe", "moe", "moe", "moe", "lm_head"])
    layer = rng.choice(["sliding", "global"])
    if kind == "glue":
        return {"kind": kind, "M": _rows(rng, 1, 2048), "layer": layer}
    gs = rng.choice([64, 64, 128])
    if kind == "lm_head":
        return {"kind": kind, "M": _rows(rng, 1, 48), "N": VOCAB, "gs": gs, "cap": rng.choice([CAP, CAP, 0.0])}
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    m = _rows(rng, 1, 256 if dtype == "fp16" else 1500)
    if kind == "dense":
        return {"kind": kind, "M": m, "layer": layer, "gs": gs, "dtype": dtype}
    entry = "dropin" if dtype == "fp16" else rng.choice(["layer", "dropin"])
    return {"kind": kind, "M": m, "gs": gs, "dtype": dtype, "entry": entry,
            "noise": 0.5 if m <= 8 and rng.random() < 0.5 else 0.0}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _words(g, *shape):
    return torch.randint(-(2 ** 31), 2 ** 31, shape, generator=g, dtype=torch.int64, device=DEV).to(torch.int32)


def _scales(g, dtype, *shape):
    return (_randn(g, *shape).abs() * SCALE_STD).to(dtype)


def _linear(g, k, n, gs, dtype):
    return _words(g, k // 8, n), _scales(g, dtype, math.ceil(k / gs), n)


def _projections(layer):
    heads, kv, width = ATTN[layer]
    p = {"q": (H, heads * width), "k": (H, kv * width)}
    if layer == "sliding":
        p["v"] = (H, kv * width)
    p.update({"o": (heads * width, H), "gate": (H, MLP), "up": (H, MLP), "down": (MLP, H)})
    return p


def _logits(g, m, noise):
    if noise > 0:
        return _randn(g, 1, E) + noise * _randn(g, m, E)
    return _randn(g, m, E)


def prepare(case, seed):
    g, m = _gen(seed), case["M"]
    dt = DTYPES[case.get("dtype", "bf16")]
    if case["kind"] == "glue":
        heads, kv, width = ATTN[case["layer"]]
        pos = torch.arange(m, device=DEV)
        inv = 10000.0 ** (-torch.arange(0, width, 2, device=DEV, dtype=torch.float64) / width)
        ang = pos.double()[:, None] * inv[None]
        ang = torch.cat([ang, ang], -1)
        return {"case": case, "x": _randn(g, m, H).to(dt), "w": (1 + 0.1 * _randn(g, H)).to(dt),
                "y": torch.empty(m, H, dtype=dt, device=DEV),
                "router_scale": (1 + 0.25 * _randn(g, H)).to(dt), "gate": (2 * _randn(g, E, H)).to(dt),
                "q": _randn(g, 1, heads, m, width).to(dt), "k": _randn(g, 1, kv, m, width).to(dt),
                "cos": ang.cos().to(dt), "sin": ang.sin().to(dt), "pos": pos[None]}
    gs = case["gs"]
    if case["kind"] == "lm_head":
        return {"case": case, "x": _randn(g, m, H).to(dt), "head": _linear(g, H, case["N"], gs, dt)}
    if case["kind"] == "dense":
        proj = _projections(case["layer"])
        s = {"case": case, "x": _randn(g, m, H).to(dt), "attn": _randn(g, m, proj["o"][0]).to(dt)}
        s["w"] = {n: _linear(g, k, c, gs, dt) for n, (k, c) in proj.items()}
        return s
    s = {"case": case, "x": _randn(g, m, H).to(dt), "logits": _logits(g, m, case["noise"])}
    s["gu"], s["gu_s"] = _words(g, E, H // 8, 2 * I), _scales(g, dt, E, math.ceil(H / gs), 2 * I)
    s["dn"], s["dn_s"] = _words(g, E, I // 8, H), _scales(g, dt, E, math.ceil(I / gs), H)
    if case["entry"] == "dropin":
        top = torch.topk(s.pop("logits"), TOP_K, dim=-1)
        s["idx"], s["wt"] = top.indices.to(torch.int32), torch.softmax(top.values, -1).to(dt)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    if case["kind"] == "glue":
        gemmainfer_csrc.rmsnorm(s["x"], s["w"], s["y"], EPS, True)
        gemmainfer_csrc.fused_rope_inplace(s["q"], s["k"], s["cos"], s["sin"], s["pos"])
        return {"norm": s["y"], "q": s["q"], "k": s["k"],
                "logits": ops.moe_router_logits(s["x"], s["router_scale"], s["gate"], EPS)}
    if case["kind"] == "lm_head":
        return ops.w4a16_linear(s["x"], *s["head"], case["gs"], softcap=case["cap"])
    if case["kind"] == "dense":
        return _run_dense(s, case)
    gs = case["gs"]
    if case["entry"] == "dropin":
        out = torch.zeros_like(s["x"])
        gemmainfer_csrc.fused_batched_moe(s["x"], s["gu"], s["gu_s"], s["dn"], s["dn_s"], s["idx"], s["wt"], out, gs)
        return out
    out, idx, wt = ops.moe_layer(s["x"], s["logits"], s["gu"], s["gu_s"], s["dn"], s["dn_s"], TOP_K, gs)
    return {"out": out, "idx": idx, "weights": wt}


def _run_dense(s, case):
    w, x, gs = s["w"], s["x"], case["gs"]
    if case["dtype"] == "bf16":
        names = [n for n in ("q", "k", "v") if n in w]
        r = dict(zip(names, ops.w4a16_linear_multi(x, [w[n] for n in names], gs)))
        r["o"] = ops.w4a16_linear(s["attn"], *w["o"], gs)
        r["act"] = ops.gated_mlp_act(x, w["gate"], w["up"], gs)
        r["down"] = ops.w4a16_linear(r["act"], *w["down"], gs)
        return r
    # the fused calls take bf16 rows; an fp16 engine calls the drop-in once per projection
    r = {}
    for n in ("q", "k", "v", "o", "gate", "up"):
        if n in w:
            a = s["attn"] if n == "o" else x
            r[n] = torch.empty(a.shape[0], w[n][0].shape[1], dtype=a.dtype, device=a.device)
            gemmainfer_csrc.marlin_w4a16(a, *w[n], r[n], gs)
    return r


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how close two right answers are
# ---------------------------------------------------------------------------
def _linear_bytes(k, n, gs):
    return k * n // 2 + math.ceil(k / gs) * n * 2


def _experts(case):
    """Mean number of distinct experts that M tokens select."""
    m, tries = case["M"], 32 if case["M"] <= 64 else 2
    g = torch.Generator().manual_seed(1)
    total = 0
    for _ in range(tries):
        rows = torch.randn(m, E, generator=g)
        if case["noise"] > 0:
            rows = torch.randn(1, E, generator=g) + case["noise"] * rows
        total += torch.topk(rows, TOP_K, dim=-1).indices.unique().numel()
    return total / tries


def work(case):
    m = case["M"]
    if case["kind"] == "glue":
        heads, kv, width = ATTN[case["layer"]]
        rope = 2 * 2 * m * (heads + kv) * width
        return {"bytes": 2 * 2 * m * H + rope + 2 * E * H + 2 * m * E, "flops": 2 * m * H * E}
    if case["kind"] == "lm_head":
        n = case["N"]
        return {"bytes": _linear_bytes(H, n, case["gs"]) + 2 * m * (H + n), "flops": 2 * m * H * n}
    if case["kind"] == "dense":
        p = _projections(case["layer"])
        if case["dtype"] != "bf16":
            del p["down"]
        words = sum(_linear_bytes(k, n, case["gs"]) for k, n in p.values())
        rows = H + p["o"][0] + sum(n for _, n in p.values()) - (MLP if case["dtype"] == "bf16" else 0)
        return {"bytes": words + 2 * m * rows, "flops": 2 * m * sum(k * n for k, n in p.values())}
    expert = _linear_bytes(H, 2 * I, case["gs"]) + _linear_bytes(I, H, case["gs"])
    return {"bytes": _experts(case) * expert + 2 * 2 * m * H + 4 * m * E, "flops": 2 * m * TOP_K * 3 * H * I}


def tolerance(case):
    # four times the distance to 64 bits: one rounding of each output, and of the activations between two products
    if case.get("dtype") == "fp16":
        return {"rel": 1.2e-3, "max": 0.015}
    return {"rel": 8e-3, "max": 0.1}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _dequant(words, scales, gs):
    """float64 [K, N] of packed [K/8, N] int4 codes (zero point 8) and [groups, N] scales."""
    kp, n = words.shape
    shift = torch.arange(0, 32, 4, device=words.device, dtype=torch.int32)
    q = ((words[:, None, :] >> shift[None, :, None]) & 15).reshape(kp * 8, n).double() - 8
    return q * scales.double().repeat_interleave(gs, 0)[: kp * 8]


def _gelu(v):
    return torch.nn.functional.gelu(v, approximate="tanh")


def exact(case, seed):
    s = prepare(case, seed)
    x = s["x"].double()
    if case["kind"] == "glue":
        n = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
        half = s["q"].shape[-1] // 2
        r = {"norm": n * (1 + s["w"].double())}
        for name in ("q", "k"):
            v = s[name].double()
            turned = torch.cat([-v[..., half:], v[..., :half]], -1)
            r[name] = v * s["cos"].double() + turned * s["sin"].double()
        r["logits"] = (n * (s["router_scale"].double() * H ** -0.5)) @ s["gate"].double().t()
        return r
    gs = case["gs"]
    if case["kind"] == "lm_head":
        words, scales = s["head"]
        y = torch.cat([x @ _dequant(words[:, c:c + 16384], scales[:, c:c + 16384], gs)
                       for c in range(0, case["N"], 16384)], 1)
        return case["cap"] * torch.tanh(y / case["cap"]) if case["cap"] > 0 else y
    if case["kind"] == "dense":
        w = s["w"]
        mul = lambda a, n: a @ _dequant(*w[n], gs)  # noqa: E731
        r = {n: mul(s["attn"].double() if n == "o" else x, n) for n in ("q", "k", "v", "o", "gate", "up") if n in w}
        if case["dtype"] == "bf16":
            r["act"] = _gelu(r.pop("gate")) * r.pop("up")
            r["down"] = mul(r["act"], "down")
        return r
    if case["entry"] == "dropin":
        idx, wt = s["idx"].long(), s["wt"].double()
    else:
        top = torch.topk(s["logits"].double(), TOP_K, dim=-1)
        idx, wt = top.indices, torch.softmax(top.values, -1)
    out = torch.zeros_like(x)
    for e in range(E):
        t, slot = torch.nonzero(idx == e, as_tuple=True)
        if t.numel():
            gu = x[t] @ _dequant(s["gu"][e], s["gu_s"][e], gs)
            y = (_gelu(gu[:, :I]) * gu[:, I:]) @ _dequant(s["dn"][e], s["dn_s"][e], gs)
            out.index_add_(0, t, wt[t, slot][:, None] * y)
    return out if case["entry"] == "dropin" else {"out": out, "idx": idx.to(torch.int32), "weights": wt}
