"""The work that programs built on this library have it do, as measurable cases.

A case is a dict of plain values. Three kinds, by what a program calls:

  "moe"     one GPT-OSS MoE block (or a captured step of several layers) over
            `rows` token rows: gossmx_moe_forward / _residual in device memory,
            gossmx_moe_forward in host memory, or a HIP graph of such calls;
  "matmul"  the kernel boundary, gossmx_mxfp4_matmul, on quantized records;
  "model"   whole model steps: a prompt and a few decode steps to logits.

Shapes are GPT-OSS-20B's (32 experts) and 120B's (128 experts): hidden and
intermediate 2880, top-4, with random weights. Every output is bit-exact by
contract, so every tolerance is "exact". `exact` restates the mathematics in
float64 with plain torch; of the path's bf16 boundaries it keeps only those that
decide the routing (the normalized row and the router logits) and, in the
model, the bf16 residual stream.
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

G = importlib.import_module("gpt-oss-rs_amd.gossmx")

HIDDEN = INTER = 2880
BLOCKS = HIDDEN // 32
TOP_K = 4
EPS = 1e-5
ALPHA, LIMIT = 1.702, 7.0
DEV = "cuda:0"
PROJECTIONS = {"residual_q8": G.PROJECTION_RESIDUAL_Q8, "q8": G.PROJECTION_Q8, "exact_bf16": G.PROJECTION_EXACT_BF16}
MODEL_LAYERS, MODEL_THREADS, MODEL_CAP = 2, 16, 1024

# ---------------------------------------------------------------------------
# The cases.


def _moe(name, rows, experts, skew, **more):
    """One MoE call. skew: expert popularity falls as rank^-skew (0: near
    uniform). norm: the decoder layer's half on its residual stream
    (post-attention RMSNorm in front, residual add behind)."""
    case = dict(kind="moe", rows=rows, experts=experts, skew=skew, projection="residual_q8", memory="device", norm=True,
                logits="computed", layers=1, graph=False)
    case.update(more)
    return dict(case, name=name) if name else case


def listed():
    return [
        # Interactive decode of one sequence: the smallest call, where latency and launches count.
        _moe("decode_1", 1, 32, 0.0),
        # A handful of sequences decoding together (one work item per expert).
        _moe("decode_5", 5, 32, 0.0, norm=False),
        # A small server's decode batch, popular experts shared by several rows.
        _moe("decode_24", 24, 32, 0.8),
        # The benchmark's decode step: 64 rows through resident layers with Zipf routing, replayed as a HIP graph.
        _moe("step_64", 64, 32, 1.1, norm=False, logits="given", layers=8, graph=True),
        # A loaded server's decode batch on the large model: 128 experts, skewed routing.
        _moe("decode_256_wide", 256, 128, 1.2),
        # Chunked prefill of odd length in the plain-Q8 projection mode.
        _moe("prefill_777_q8", 777, 32, 0.0, projection="q8", norm=False),
        # Prefill of a prompt on the small and the large model (the benchmark's sizes).
        _moe("prefill_2048", 2048, 32, 0.0),
        _moe("prefill_4096_wide", 4096, 128, 0.0, norm=False),
        # The drop-in host-memory call (rows in and every CpuMoeStep output back in host slices).
        _moe("host_17", 17, 32, 0.8, memory="host", norm=False),
        # An accuracy comparison in the exact-BF16 projection mode, a short prompt's rows.
        _moe("exact_bf16_40", 40, 32, 0.0, projection="exact_bf16", norm=False),
        # The kernel boundary: one expert's gate_up on quantized rows, ragged count, padded output rows.
        dict(name="matmul_129", kind="matmul", rows=129, n=5760, activation="residual_q8", pad=8),
        # A prompt and eight decode steps to logits through a two-layer cut of the 20B model.
        dict(name="model_63_8", kind="model", prompt=63, steps=8),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    u = rng.random()
    experts = rng.choice((32, 32, 128))
    skew = rng.choice((0.0, round(rng.uniform(0.3, 1.3), 2)))
    norm = rng.random() < 0.5
    if u < 0.50:
        return _moe(None, _log_int(rng, 1, 4096), experts, skew, norm=norm)
    if u < 0.60:
        return _moe(None, _log_int(rng, 1, 2048), experts, skew, norm=norm, projection="q8")
    if u < 0.68:
        return _moe(None, _log_int(rng, 1, 64), 32, skew, norm=norm, projection="exact_bf16")
    if u < 0.78:
        return _moe(None, _log_int(rng, 1, 256), experts, skew, norm=False, memory="host")
    if u < 0.86:
        return _moe(None, _log_int(rng, 1, 128), 32, skew, norm=norm, layers=rng.randint(2, 8), graph=True,
                    logits=rng.choice(("given", "computed")))
    if u < 0.94:
        return dict(kind="matmul", rows=_log_int(rng, 1, 1024), n=rng.choice((2880, 5760)),
                    activation=rng.choice(("residual_q8", "residual_q8", "q8")), pad=rng.choice((0, 8)))
    return dict(kind="model", prompt=_log_int(rng, 1, 128), steps=rng.randint(0, 8))


# ---------------------------------------------------------------------------
# Inputs.

_ctx = None


def _context():
    """The program's one context."""
    global _ctx
    if _ctx is None:
        torch.cuda.init()
        _ctx = G.Context(0)
    return _ctx


class State:
    """What a program holds between calls; its device objects are released with it."""

    def __init__(self):
        self.owned = []

    def own(self, obj):
        self.owned.append(obj)
        return obj

    def __del__(self):
        for obj in reversed(self.owned):
            obj.close()


def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _normal(seed, salt, shape, std=1.0, dtype=torch.float32):
    """N(0, std) rounded to bf16."""
    t = torch.randn(shape, generator=_gen(seed, salt), device=DEV).mul_(std).to(torch.bfloat16)
    return t if dtype == torch.bfloat16 else t.to(dtype)


def _rows(seed, salt, m, norm):
    """Hidden rows bf16 [m][hidden]: RMS-normalized, or a residual stream to be normalized by the call."""
    x = torch.randn((m, HIDDEN), generator=_gen(seed, salt), device=DEV)
    if not norm:
        x = x * torch.rsqrt(x.square().mean(1, keepdim=True) + EPS)
    return x.to(torch.bfloat16)


def _bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def _popularity(seed, salt, experts, skew):
    """log p of each expert, p falling as rank^-skew over a random order."""
    order = torch.randperm(experts, generator=_gen(seed, salt), device=DEV)
    return -skew * torch.log(1.0 + order.to(torch.float32))


def _layer_tensors(seed, layer, experts, skew):
    s = 100 * layer
    return dict(router_w=_normal(seed, s + 1, (experts, HIDDEN), 0.02, torch.bfloat16),
                router_b=(_normal(seed, s + 2, (experts,), 0.02) + _popularity(seed, s + 3, experts, skew)).to(torch.bfloat16).float(),
                gate_up_b=_normal(seed, s + 4, (experts, 2 * INTER), 0.02),
                down_b=_normal(seed, s + 5, (experts, HIDDEN), 0.02))


def _layer(state, seed, layer, experts, skew, projection):
    ctx, t = _context(), _layer_tensors(seed, layer, experts, skew)
    gate_up = state.own(G.Weights.generate(ctx, seed, 16 * layer + 4, experts, 2 * INTER, BLOCKS))
    down = state.own(G.Weights.generate(ctx, seed, 16 * layer + 5, experts, HIDDEN, INTER // 32))
    return state.own(G.MoeLayer(ctx, experts, HIDDEN, INTER, TOP_K, _bits(t["router_w"]), t["router_b"].cpu().numpy(),
                                gate_up, t["gate_up_b"].cpu().numpy(), down, t["down_b"].cpu().numpy(), ALPHA, LIMIT,
                                PROJECTIONS[projection]))


def _given_logits(case, seed, layer):
    """Router logits in hand (bf16 values) with the case's expert popularity."""
    u = torch.rand((case["rows"], case["experts"]), generator=_gen(seed, 100 * layer + 50), device=DEV)
    gumbel = -torch.log(-torch.log(u.clamp(1e-6, 1.0 - 1e-6)))
    return (gumbel + _popularity(seed, 100 * layer + 3, case["experts"], case["skew"])).to(torch.bfloat16).float()


def _norm_weight(seed, layer):
    return 1.0 + 0.25 * torch.randn((HIDDEN,), generator=_gen(seed, 100 * layer + 60), device=DEV)


def _prepare_moe(case, seed):
    s, m, E = State(), case["rows"], case["experts"]
    s.case, s.ctx = case, _context()
    s.x = _rows(seed, 7, m, case["norm"])
    s.layers = [_layer(s, seed, i, E, case["skew"], case["projection"]) for i in range(case["layers"])]
    s.logits = [_given_logits(case, seed, i) if case["logits"] == "given" else None for i in range(case["layers"])]
    if case["memory"] == "host":
        s.host_x = _bits(s.x)
        s.logits = [None if t is None else t.cpu().numpy() for t in s.logits]
        return s
    s.norm_w = [_norm_weight(seed, i) for i in range(case["layers"])]
    s.out = []
    for _ in s.layers:
        o = {"selected": torch.empty((m, TOP_K), dtype=torch.int32, device=DEV)}
        if case["norm"]:
            o["next"] = torch.empty((m, HIDDEN), dtype=torch.bfloat16, device=DEV)
        else:
            o["output"] = torch.empty((m, HIDDEN), dtype=torch.float32, device=DEV)
            o["weights"] = torch.empty((m, TOP_K), dtype=torch.float32, device=DEV)
            o["logits"] = torch.empty((m, E), dtype=torch.float32, device=DEV)
        s.out.append(o)
    s.graph = None
    if case["graph"]:
        torch.cuda.synchronize()
        _run_moe_device(s)  # sizes the context's buffers
        s.ctx.synchronize()
        s.ctx.capture_begin()
        _run_moe_device(s)
        s.graph = s.own(s.ctx.capture_end())
    return s


def _records(x, activation):
    """Q8Block / ResidualQ8Block records of f32 rows, as bytes [m][blocks][36 or 72]."""
    def block(v):
        scale = v.abs().amax(-1, keepdim=True) / 127.0
        q = torch.where(scale == 0, torch.zeros_like(v), torch.round(v / scale)).clamp(-127, 127)
        raw = torch.cat([scale.contiguous().view(torch.uint8), q.to(torch.int8).view(torch.uint8)], -1)
        return raw, v - q * scale
    raw, rest = block(x.view(x.shape[0], -1, 32))
    return (torch.cat([raw, block(rest)[0]], -1) if activation == "residual_q8" else raw).contiguous()


def _prepare_matmul(case, seed):
    s, m, n = State(), case["rows"], case["n"]
    s.case, s.ctx = case, _context()
    s.records = _records(_rows(seed, 7, m, False).float(), case["activation"])
    s.bias = _normal(seed, 4, (n,), 0.02)
    s.weights = s.own(G.Weights.generate(s.ctx, seed, 4, 1, n, BLOCKS))
    s.out = torch.zeros((m, n + case["pad"]), dtype=torch.float32, device=DEV)
    return s


def _model_config():
    return dict(G.GPT_OSS_20B, layers=MODEL_LAYERS)


def _model_tensors(seed):
    c = _model_config()
    H, QW, KW = c["hidden"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    layers = []
    for i in range(MODEL_LAYERS):
        s, t = 1000 + 100 * i, {}
        for k, (name, rows, cols) in enumerate((("q", QW, H), ("k", KW, H), ("v", KW, H), ("o", H, QW))):
            t[name + "_weight"] = _normal(seed, s + 2 * k, (rows, cols), 0.02, torch.bfloat16)
            t[name + "_bias"] = _normal(seed, s + 2 * k + 1, (rows,), 0.02)
        t["input_norm"] = 1.0 + _normal(seed, s + 10, (H,), 0.02)
        t["post_attention_norm"] = 1.0 + _normal(seed, s + 11, (H,), 0.02)
        t["sinks"] = _normal(seed, s + 12, (c["heads"],), 0.02)
        layers.append(t)
    # One matrix serves as embedding and head.
    return dict(layers=layers, head=_normal(seed, 900, (c["vocab"], H), 0.02, torch.bfloat16),
                final_norm=1.0 + _normal(seed, 901, (H,), 0.02))


def _model_tokens(case, seed):
    n = case["prompt"] + case["steps"]
    return torch.randint(0, G.GPT_OSS_20B["vocab"], (n,), generator=_gen(seed, 70), device=DEV)


def _prepare_model(case, seed):
    s, c = State(), _model_config()
    s.case, s.ctx = case, _context()
    t = _model_tensors(seed)
    layers = []
    for i, L in enumerate(t["layers"]):
        d = {k: (_bits(v) if v.dtype == torch.bfloat16 else v.cpu().numpy()) for k, v in L.items()}
        layers.append(dict(d, sliding=i % 2 == 0, moe=_layer(s, seed, i, 32, 0.0, "residual_q8")))
    head = _bits(t["head"])
    s.model = s.own(G.Model(s.ctx, G.model_config(context_cap=MODEL_CAP, threads=MODEL_THREADS, **c), head,
                            t["final_norm"].cpu().numpy(), head, layers))
    s.tokens = _model_tokens(case, seed).cpu().numpy().astype(np.uint32)
    return s


def prepare(case, seed):
    return {"moe": _prepare_moe, "matmul": _prepare_matmul, "model": _prepare_model}[case["kind"]](case, seed)


# ---------------------------------------------------------------------------
# One pass.


def _run_moe_device(s):
    m = s.case["rows"]
    for layer, o, logits, w in zip(s.layers, s.out, s.logits, s.norm_w):
        if s.case["norm"]:
            layer.forward_residual_device(s.x, m, w, EPS, o["next"], injected_logits=logits, selected=o["selected"])
        else:
            layer.forward_device(s.x, m, o["output"], injected_logits=logits, router_logits=o["logits"],
                                 selected=o["selected"], routing_weights=o["weights"])


def run(s):
    case = s.case
    if case["kind"] == "matmul":
        kind = G.ACT_RESIDUAL_Q8 if case["activation"] == "residual_q8" else G.ACT_Q8
        G.mxfp4_matmul_device(s.ctx, s.weights, 0, s.records, case["rows"] * BLOCKS, case["rows"], s.bias, s.out,
                              s.out.numel(), s.out.shape[1], kind)
        return {"output": s.out}
    if case["kind"] == "model":
        logits = [s.model.prefill(s.tokens[:case["prompt"]])]
        for t in s.tokens[case["prompt"]:]:
            logits.append(s.model.decode(int(t)))
        return {"logits": logits}
    if case["memory"] == "host":
        r = s.layers[0].forward(s.host_x, s.logits[0])
        return {"output": r["output"], "weights": r["routing_weights"], "logits": r["router_logits"],
                "selected": r["selected"].view(np.int32)}
    if s.graph is not None:
        s.graph.launch()
    else:
        _run_moe_device(s)
    return s.out


# ---------------------------------------------------------------------------
# What a pass cannot do without.


def _touched(rows, experts, skew):
    """Expected number of experts that `rows` rows of top-4 routing reach."""
    p = np.arange(1, experts + 1, dtype=np.float64) ** -skew
    lo, hi = 0.0, 1e9
    for _ in range(100):  # inclusion of expert e in a row: 1 - exp(-t p_e), four in all
        t = 0.5 * (lo + hi)
        lo, hi = (t, hi) if (1.0 - np.exp(-t * p)).sum() < TOP_K else (lo, t)
    return float((1.0 - np.exp(-t * p * rows)).sum())


def _moe_work(rows, experts, skew, norm, computed, bytes_out):
    per_expert = 3 * INTER * BLOCKS * 17 + (2 * INTER + HIDDEN) * 4
    b = _touched(rows, experts, skew) * per_expert + rows * HIDDEN * 2 + bytes_out
    f = 2.0 * rows * TOP_K * 3 * INTER * HIDDEN
    if computed:
        b += experts * (HIDDEN * 2 + 4)
        f += 2.0 * rows * experts * HIDDEN
    else:
        b += rows * experts * 4
    return b + (HIDDEN * 4 if norm else 0), f


def work(case):
    if case["kind"] == "matmul":
        rec = 72 if case["activation"] == "residual_q8" else 36
        return {"bytes": case["n"] * (BLOCKS * 17 + 4) + case["rows"] * (BLOCKS * rec + case["n"] * 4),
                "flops": 2.0 * case["rows"] * case["n"] * HIDDEN}
    if case["kind"] == "model":
        c = _model_config()
        H, QW, KW = c["hidden"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        total_b = total_f = 0.0
        for i in range(case["steps"] + 1):
            rows = case["prompt"] if i == 0 else 1
            seen = case["prompt"] + i
            b, f = _moe_work(rows, 32, 0.0, True, True, rows * H * 2)
            proj = 2 * QW * H + 2 * KW * H
            pairs = rows * seen - rows * (rows - 1) / 2
            total_b += MODEL_LAYERS * (b + 2 * proj + 4 * KW * seen) + 2 * c["vocab"] * H + 4 * c["vocab"]
            total_f += MODEL_LAYERS * (f + 2 * rows * proj + 4 * pairs * QW) + 2 * c["vocab"] * H
        return {"bytes": total_b, "flops": total_f}
    m, E = case["rows"], case["experts"]
    out = m * TOP_K * 4 + (m * HIDDEN * 2 if case["norm"] else m * (HIDDEN + E + TOP_K) * 4)
    b, f = _moe_work(m, E, case["skew"], case["norm"], case["logits"] == "computed", out)
    return {"bytes": case["layers"] * b, "flops": case["layers"] * f}


def tolerance(case):
    return "exact"  # every output is bit-identical to the scalar definition of the path


# ---------------------------------------------------------------------------
# The same in float64.


def _splitmix64(x):
    def shr(v, n):
        return (v >> n) & ((1 << (64 - n)) - 1)
    z = x + (0x9E3779B97F4A7C15 - (1 << 64))
    z = (z ^ shr(z, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
    z = (z ^ shr(z, 27)) * (0x94D049BB133111EB - (1 << 64))
    return z ^ shr(z, 31)


def _expert(seed, stream, rows, blocks, e):
    """Expert e of a generated MXFP4 tensor, [rows][32 * blocks] float64 (the rule gossmx_weights_generate documents)."""
    key = (int(seed) ^ ((stream * 0xD1B54A32D192ED03) & ((1 << 64) - 1))) & ((1 << 64) - 1)
    key = _splitmix64(torch.tensor(key - (1 << 64) if key >> 63 else key, dtype=torch.int64, device=DEV))
    i = torch.arange(e * rows * blocks, (e + 1) * rows * blocks, dtype=torch.int64, device=DEV)
    h0, h1 = _splitmix64(key + 2 * i), _splitmix64(key + 2 * i + 1)
    scale = torch.exp2((119 + ((h1 >> 61) & 7) % 5 - 127).double())
    shifts = torch.arange(0, 64, 4, dtype=torch.int64, device=DEV)
    codes = torch.cat([(h0[:, None] >> shifts) & 15, (h1[:, None] >> shifts) & 15], 1)
    table = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0],
                         dtype=torch.float64, device=DEV)
    return (table[codes] * scale[:, None]).view(rows, blocks * 32)


def _bf16(t):
    return t.to(torch.float32).to(torch.bfloat16).double()


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _moe64(x, t, seed, layer, experts, logits=None):
    """(output, weights, logits, margin) of one block on float64 rows; margin: how far each row's routing is from
    another choice of experts."""
    if logits is None:
        logits = _bf16(x @ t["router_w"].double().T + t["router_b"].double())
    # Descending value, the lower index first on ties.
    top = torch.sort(logits, dim=1, descending=True, stable=True)
    sel, weights = top.indices[:, :TOP_K], torch.softmax(top.values[:, :TOP_K], 1)
    out = torch.zeros_like(x)
    for e in torch.unique(sel).tolist():
        r, k = torch.nonzero(sel == e, as_tuple=True)
        gu = x[r] @ _expert(seed, 16 * layer + 4, 2 * INTER, BLOCKS, e).T + t["gate_up_b"][e].double()
        gate, up = gu[:, 0::2].clamp(max=LIMIT), gu[:, 1::2].clamp(-LIMIT, LIMIT)
        act = gate * torch.sigmoid(ALPHA * gate) * (up + 1.0)
        y = act @ _expert(seed, 16 * layer + 5, HIDDEN, INTER // 32, e).T + t["down_b"][e].double()
        out.index_add_(0, r, y * weights[r, k][:, None])
    return out, weights, logits, top.values[:, TOP_K - 1] - top.values[:, TOP_K]


def _exact_moe(case, seed):
    outs = []
    for i in range(case["layers"]):
        t = _layer_tensors(seed, i, case["experts"], case["skew"])
        x = _rows(seed, 7, case["rows"], case["norm"]).double()
        h = _bf16(_rms(x, _norm_weight(seed, i))) if case["norm"] else x
        given = _given_logits(case, seed, i).double() if case["logits"] == "given" else None
        out, weights, logits, _ = _moe64(h, t, seed, i, case["experts"], given)
        o = {"next": x + out, "selected": None} if case["norm"] else {
            "output": out, "weights": weights, "logits": logits, "selected": None}
        outs.append(o)
    return outs[0] if case["memory"] == "host" else outs


def _exact_matmul(case, seed):
    raw = _records(_rows(seed, 7, case["rows"], False).float(), case["activation"])
    x = 0.0
    for o in range(0, raw.shape[2], 36):
        scale = raw[:, :, o:o + 4].contiguous().view(torch.float32).double()
        x = x + scale * raw[:, :, o + 4:o + 36].contiguous().view(torch.int8).double()
    out = torch.zeros((case["rows"], case["n"] + case["pad"]), dtype=torch.float64, device=DEV)
    out[:, :case["n"]] = (x.view(case["rows"], -1) @ _expert(seed, 4, case["n"], BLOCKS, 0).T
                          + _normal(seed, 4, (case["n"],), 0.02).double())
    return {"output": out}


def _rope64(c, x):
    """YaRN rotary embedding of [positions][heads][head_dim] rows at positions 0..."""
    dim = c["head_dim"]
    freq = c["rope_theta"] ** (torch.arange(0, dim, 2, dtype=torch.float64, device=DEV) / dim)

    def correction(rotations):
        return dim * math.log(c["rope_original_max_positions"] / (rotations * 2 * math.pi)) / (2 * math.log(c["rope_theta"]))
    low, high = max(correction(c["rope_beta_fast"]), 0.0), min(correction(c["rope_beta_slow"]), dim - 1.0)
    ramp = ((torch.arange(dim // 2, dtype=torch.float64, device=DEV) - low) / max(high - low, 0.001)).clamp(0, 1)
    inv = ramp / (c["rope_factor"] * freq) + (1 - ramp) / freq
    angle = torch.arange(x.shape[0], dtype=torch.float64, device=DEV)[:, None] * inv
    scale = 0.1 * math.log(c["rope_factor"]) + 1.0
    cos, sin = (torch.cos(angle) * scale)[:, None], (torch.sin(angle) * scale)[:, None]
    a, b = x[..., :dim // 2], x[..., dim // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _exact_model(case, seed):
    c, t, tokens = _model_config(), _model_tensors(seed), _model_tokens(case, seed)
    n, heads, kv, dim = tokens.numel(), c["heads"], c["kv_heads"], c["head_dim"]
    h = t["head"][tokens].double()
    pos = torch.arange(n, device=DEV)
    margin = torch.full((n,), math.inf, dtype=torch.float64, device=DEV)
    for i, L in enumerate(t["layers"]):
        x = _bf16(_rms(h, L["input_norm"]))
        q, k, v = (_bf16(x @ L[p + "_weight"].double().T + L[p + "_bias"].double()).view(n, -1, dim) for p in "qkv")
        q, k = _bf16(_rope64(c, q)), _bf16(_rope64(c, k))
        k, v = (a.repeat_interleave(heads // kv, 1) for a in (k, v))
        s = torch.matmul(q.transpose(0, 1).contiguous(), k.permute(1, 2, 0).contiguous()) / math.sqrt(dim)
        back = pos[:, None] - pos[None, :]
        seen = (back >= 0) & (back < (c["sliding_window"] if i % 2 == 0 else MODEL_CAP))
        s = torch.where(seen, s, torch.full_like(s, -math.inf))
        s = torch.cat([s, L["sinks"].double()[:, None, None].expand(heads, n, 1)], 2)
        a = torch.matmul(torch.softmax(s, 2)[:, :, :n].contiguous(), v.transpose(0, 1).contiguous())
        a = _bf16(a.transpose(0, 1).reshape(n, heads * dim))
        h = _bf16(h + _bf16(a @ L["o_weight"].double().T + L["o_bias"].double()))
        out, _, _, near = _moe64(_bf16(_rms(h, L["post_attention_norm"])), _layer_tensors(seed, i, 32, 0.0), seed, i, 32)
        margin = torch.minimum(margin, near)
        h = _bf16(h + _bf16(out))
    last = _bf16(_rms(h[case["prompt"] - 1:], t["final_norm"]))
    logits = torch.cat([last @ w.double().T for w in t["head"].split(16384)], 1)
    # A token whose experts hang on the last bits of its bf16 router logits has no one value (2^-5: four spacings of
    # bf16 at a logit of 2 to 4).
    clear = (margin[case["prompt"] - 1:] > 2.0 ** -5).tolist()
    return {"logits": [row if ok else None for row, ok in zip(logits, clear)]}


def exact(case, seed):
    return {"moe": _exact_moe, "matmul": _exact_matmul, "model": _exact_model}[case["kind"]](case, seed)
