"""The work that a program using this framework has it do, as measurable cases.

A case is a dict of plain values.  ``prepare`` makes what the program holds
before the call (inputs from the seed, weights in the layout the framework
keeps them in, caches), ``run`` makes the call or calls of one pass through
the public entry points, ``exact`` gives the same outputs from plain torch in
64 bits.  Weights follow the gpt-oss-style MXFP4 distribution of the
repository's own synthetic layers: uniform E2M1 codes, E8M0 scale bytes
118..124, router weight N(0, 0.02), biases N(0, 0.01), activations N(0, 1).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = Path(__file__).resolve().parents[1] / "kcapw-klcquant_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

LIMIT = 7.0  # SwiGLU clamp
EPS = 1e-5
HEADS, KV_HEADS, HEAD_DIM = 64, 8, 64
WINDOW = 128
FP4 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _moe(name, tokens, experts, precision="fp32", skew=0.0, layers=1, kind="moe", top_k=4, hidden=2880, inter=2880):
    case = {"name": name} if name else {}
    case.update(kind=kind, tokens=tokens, experts=experts, top_k=top_k, hidden=hidden, inter=inter,
                precision=precision, skew=skew, layers=layers)
    return case


def listed() -> list[dict]:
    return [
        # one sequence decoding: a token through consecutive layers, the lowest-latency use
        _moe("moe_decode_1", 1, 128, layers=4),
        # the drop-in call of the executor's token loop, its bookkeeping and routing logs included
        _moe("route_1", 1, 128, kind="route"),
        # 64 sequences decoding: norm, routed experts and the residual add of one layer
        _moe("block_decode_64", 64, 128, kind="block"),
        # a large decode batch, or a short prompt, at an odd size
        _moe("moe_batch_300", 300, 128),
        # a prompt of the smaller model, at an odd size, in the default precision
        _moe("moe_prefill_777", 777, 32),
        # a prefill chunk with the skewed routing of real text, in the reference's bf16 matmul mode
        _moe("moe_prefill_2048", 2048, 128, precision="bf16", skew=1.1),
        # decode attention of one token through alternating sliding and full layers
        {"name": "attention_4096", "kind": "attention", "context": 4096, "layers": 4, "kv": "fp16"},
        # the same at a long context
        {"name": "attention_32768", "kind": "attention", "context": 32768, "layers": 2, "kv": "fp16"},
        # the vocabulary logits and greedy token that end every decode step
        {"name": "lm_head_201088", "kind": "lm_head", "vocab": 201088, "hidden": 2880},
        # a whole layer's down projections from the checkpoint to dense bfloat16
        {"name": "dequant_down_128", "kind": "dequant", "matrices": 128, "rows": 2880, "groups": 90, "dtype": "bf16"},
        # one expert's gate_up from the checkpoint, in the default output type
        {"name": "dequant_gate_up_1", "kind": "dequant", "matrices": 1, "rows": 5760, "groups": 90, "dtype": "fp16"},
        # the dense matrices of a token's experts out of a resident layer
        _moe("load_experts_4", 4, 32, kind="load"),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(("moe", "moe", "moe", "moe", "block", "route", "attention", "attention", "lm_head", "dequant",
                       "dequant", "load"))
    if kind in ("moe", "block", "route", "load"):
        hidden, inter = rng.choice(((2880, 2880), (2880, 2880), (2880, 2880), (2048, 2048), (2048, 1024), (1536, 2496)))
        experts = rng.choice((128, 128, 32, 64))
        top_k = rng.choice((4, 4, 4, 2, 8))
        tokens = {"moe": _log(rng, 1, 8000 // top_k), "block": _log(rng, 1, 600), "route": _log(rng, 1, 48),
                  "load": rng.randint(1, 16)}[kind]
        precision = rng.choice(("fp32", "fp32", "bf16"))
        skew = rng.choice((0.0, round(rng.uniform(0.3, 1.2), 2)))
        return _moe("", tokens, experts, precision, skew, 1, kind, top_k, hidden, inter)
    if kind == "attention":
        return {"kind": kind, "context": _log(rng, 64, 32768), "layers": 2, "kv": rng.choice(("fp16", "fp16", "bf16"))}
    if kind == "lm_head":
        return {"kind": kind, "vocab": _log(rng, 8000, 201088), "hidden": rng.choice((2880, 2880, 2048, 1024, 4096))}
    dtype = rng.choice(("bf16", "fp16", "fp32"))
    rows = rng.choice((64 * rng.randint(8, 90), rng.randint(300, 5760)))
    groups = rng.randint(16, 90)
    most = 128 * 2880 * 90 * 66 // (rows * groups * (66 if dtype != "fp32" else 130))
    return {"kind": kind, "matrices": _log(rng, 1, min(128, most)), "rows": rows, "groups": groups, "dtype": dtype}


# ---- inputs ---------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _bytes(g, *shape) -> torch.Tensor:
    n = math.prod(shape)
    words = torch.randint(-2 ** 63, 2 ** 63 - 1, ((n + 7) // 8,), dtype=torch.int64, device="cuda", generator=g)
    return words.view(torch.uint8)[:n].reshape(shape)


def _scales(g, *shape) -> torch.Tensor:
    return torch.randint(118, 125, shape, dtype=torch.uint8, device="cuda", generator=g)


def _normal(g, shape, std=1.0, mean=0.0) -> torch.Tensor:
    return (torch.randn(shape, device="cuda", generator=g) * std + mean).to(torch.bfloat16)


def _skewed_bias(g, x, w, k, skew, bias) -> torch.Tensor:
    """Router bias that makes the experts' loads follow rank^-skew on these inputs (a few fitting steps)."""
    n_exp = w.shape[0]
    rank = torch.randperm(n_exp, device="cuda", generator=g).float() + 1
    share = rank ** -skew
    target = share / share.sum() * x.shape[0] * k
    logits = x.float() @ w.float().T
    b = -skew * torch.log(rank) + bias.float()
    for _ in range(40):
        top = torch.topk(logits + b, k, dim=1).indices
        count = torch.zeros(n_exp, device="cuda").index_add_(0, top.reshape(-1), torch.ones(top.numel(), device="cuda"))
        b += 0.25 * (torch.log(target + 0.5) - torch.log(count + 0.5))
    return b.to(torch.bfloat16)


def _layer_host(case: dict, seed: int, layer: int) -> dict:
    """One layer's input and checkpoint tensors, on the GPU."""
    g = _gen(seed * 1009 + layer)
    e, h, i, k = case["experts"], case["hidden"], case["inter"], case["top_k"]
    t = {"x": _normal(g, (case["tokens"], h)), "router_w": _normal(g, (e, h), 0.02),
         "router_b": _normal(g, (e,), 0.01),
         "gu_blocks": _bytes(g, e, 2 * i, h // 32, 16), "gu_scales": _scales(g, e, 2 * i, h // 32),
         "gu_bias": _normal(g, (e, 2 * i), 0.01),
         "d_blocks": _bytes(g, e, h, i // 32, 16), "d_scales": _scales(g, e, h, i // 32),
         "d_bias": _normal(g, (e, h), 0.01)}
    t["norm"] = _normal(g, (h,), 0.05, 1.0)
    if case["skew"] > 0:
        x = _norm_exact(t["x"], t["norm"]) if case["kind"] == "block" else t["x"]
        t["router_b"] = _skewed_bias(g, x, t["router_w"], k, case["skew"], t["router_b"])
    return t


def _attention_host(case: dict, seed: int, layer: int) -> dict:
    g = _gen(seed * 1009 + layer)
    q, kv, h = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM, 2880
    return {"x": _normal(g, (h,)),
            "q_w": _normal(g, (q, h), 0.02), "q_b": _normal(g, (q,), 0.01),
            "k_w": _normal(g, (kv, h), 0.02), "k_b": _normal(g, (kv,), 0.01),
            "v_w": _normal(g, (kv, h), 0.02), "v_b": _normal(g, (kv,), 0.01),
            "o_w": _normal(g, (h, q), 0.02), "o_b": _normal(g, (h,), 0.01),
            "sinks": _normal(g, (HEADS,)),
            "keys": torch.randn((case["context"], KV_HEADS, HEAD_DIM), device="cuda", generator=g).to(DTYPES[case["kv"]]),
            "values": torch.randn((case["context"], KV_HEADS, HEAD_DIM), device="cuda", generator=g).to(DTYPES[case["kv"]])}


def _attention_config():
    from klcquant_amd.attention import AttentionConfig

    return AttentionConfig(hidden_size=2880, num_heads=HEADS, num_kv_heads=KV_HEADS, head_dim=HEAD_DIM,
                           rope_factor=32.0, sliding_window=None)


def _windows(case: dict) -> list:
    # alternating sliding and full layers
    return [WINDOW if layer % 2 == 0 else None for layer in range(case["layers"])]


# ---- the framework's side ---------------------------------------------------------------


def prepare(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("moe", "block", "route", "load"):
        from klcquant_amd import moe

        xs, weights, norms = [], [], []
        for layer in range(case["layers"]):
            t = _layer_host(case, seed, layer)
            weights.append(moe.MoELayerWeights.from_checkpoint(
                t["router_w"], t["router_b"], t["gu_blocks"], t["gu_scales"], t["gu_bias"], t["d_blocks"],
                t["d_scales"], t["d_bias"]))
            xs.append(t["x"])
            norms.append(t["norm"])
        state = {"case": case, "xs": xs}
        if kind == "moe":
            state["layers"] = [moe.MoELayer(w, case["top_k"], LIMIT, case["precision"]) for w in weights]
        elif kind == "block":
            state["stack"] = moe.MoEStack(weights, norms, case["top_k"], LIMIT, case["precision"], EPS)
        else:
            from klcquant_amd.mxfp4_expert import ResidentExpertStore
            from klcquant_amd.streamed_moe_router import StreamedMoERouter

            w = weights[0]
            p = "model.layers.0.mlp"
            state["store"] = ResidentExpertStore({0: w})
            state["router"] = StreamedMoERouter(case["top_k"], LIMIT, matmul_precision=case["precision"])
            state["tensors"] = {f"{p}.router.weight": w.router_weight, f"{p}.router.bias": w.router_bias,
                                f"{p}.experts.gate_up_proj_bias": w.gate_up_bias,
                                f"{p}.experts.down_proj_bias": w.down_bias}
            state["position"] = 0
            state["experts"] = sorted({(7 * seed + 5 * j) % case["experts"] for j in range(case["tokens"])})
        return state
    if kind == "attention":
        from klcquant_amd.attention import DeviceKVCache, StreamedAttention

        cache = DeviceKVCache(torch.device("cuda"), max_tokens=case["context"], precision=case["kv"])
        tensors, xs = {}, []
        for layer in range(case["layers"]):
            t = _attention_host(case, seed, layer)
            p = f"model.layers.{layer}.self_attn"
            for n in "qkvo":
                tensors[f"{p}.{n}_proj.weight"], tensors[f"{p}.{n}_proj.bias"] = t[f"{n}_w"], t[f"{n}_b"]
            tensors[f"{p}.sinks"] = t["sinks"]
            ring, _ = cache.next_slot(layer, KV_HEADS, HEAD_DIM)
            ring["k"].copy_(t["keys"])
            ring["v"].copy_(t["values"])
            ring["total"] = case["context"]
            xs.append(t["x"])
        return {"case": case, "attention": StreamedAttention(_attention_config()), "cache": cache, "xs": xs,
                "tensors": tensors, "position": case["context"], "windows": _windows(case)}
    g = _gen(seed)
    if kind == "lm_head":
        from klcquant_amd.lm_head import LmHead

        w = _normal(g, (case["vocab"], case["hidden"]), 0.02)
        return {"case": case, "head": LmHead(w), "x": _normal(g, (case["hidden"],))}
    n, rows, groups = case["matrices"], case["rows"], case["groups"]
    shape = (n, rows, groups) if n > 1 else (rows, groups)
    return {"case": case, "blocks": _bytes(g, *shape, 16), "scales": _scales(g, *shape)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "moe":
        return [layer.forward(x) for layer, x in zip(state["layers"], state["xs"])]
    if kind == "block":
        return state["stack"].forward(state["xs"][0])
    if kind == "route":
        x = state["xs"][0]
        n = case["tokens"]
        at = state["position"]
        state["position"] = at + n
        hidden, position = (x[0], at) if n == 1 else (x, list(range(at, at + n)))
        out, route = state["router"].route(0, hidden, state["tensors"], state["store"], position=position)
        logs = [route["expert_logs"]] if n == 1 else route["expert_logs"]
        return {"out": out, "experts": torch.tensor(route["experts"]), "weights": torch.tensor(route["weights"]),
                "norms": torch.tensor([[[e["gate_up_norm"], e["output_norm"]] for e in row] for row in logs])}
    if kind == "load":
        store = state["store"]
        return [store.load_expert_matrix(0, e, proj) for e in state["experts"] for proj in ("gate_up_proj", "down_proj")]
    if kind == "attention":
        at = state["position"]
        state["position"] = at + 1
        outs = []
        for layer, (x, window) in enumerate(zip(state["xs"], state["windows"])):
            out, info = state["attention"].forward(layer, x, state["tensors"], at, state["cache"], window)
            outs.append([out, torch.tensor([info["q_pre_rope_norm"], info["k_pre_rope_norm"], info["q_post_rope_norm"],
                                            info["k_post_rope_norm"], info["q_rope_delta_norm"],
                                            info["k_rope_delta_norm"]]),
                         info["q_post_rope_nonfinite_count"] + info["k_post_rope_nonfinite_count"]])
        return outs
    if kind == "lm_head":
        logits, token = state["head"].logits_device(state["x"])
        return [logits, token]
    from klcquant_amd.mxfp4_expert import dequantize_mxfp4_matrix

    return dequantize_mxfp4_matrix(state["blocks"], state["scales"], DTYPES[case["dtype"]])


# ---- what a pass cannot do without --------------------------------------------------------


def _touched(experts: int, k: int, tokens: int, skew: float) -> float:
    """Expected distinct experts of ``tokens`` top-k selections."""
    p = [r ** -skew for r in range(1, experts + 1)]
    total = sum(p)
    return sum(1.0 - (1.0 - min(1.0, k * v / total)) ** tokens for v in p)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("moe", "block", "route"):
        t, e, k, h, i = case["tokens"], case["experts"], case["top_k"], case["hidden"], case["inter"]
        per_expert = 3 * i * h // 32 * 17 + (2 * i + h) * 2
        per_layer = _touched(e, k, t, case["skew"]) * per_expert + e * (h + 1) * 2 + t * h * 4
        if kind == "block":
            per_layer += h * 2
        flops = t * k * 6 * h * i + 2 * t * h * e
        return {"bytes": case["layers"] * per_layer, "flops": case["layers"] * flops}
    if kind == "load":
        n = min(case["tokens"], case["experts"])
        return {"bytes": n * 3 * case["inter"] * (case["hidden"] // 32) * (17 + 64), "flops": 0}
    if kind == "attention":
        weights = 2 * 2880 * (2 * HEADS + 2 * KV_HEADS) * HEAD_DIM
        total = flops = 0
        for window in _windows(case):
            keys = min(window or case["context"], case["context"])
            total += weights + 2 * keys * KV_HEADS * HEAD_DIM * 2
            flops += weights + 4 * keys * HEADS * HEAD_DIM
        return {"bytes": total, "flops": flops}
    if kind == "lm_head":
        v, h = case["vocab"], case["hidden"]
        return {"bytes": v * h * 2 + v * 4 + h * 2, "flops": 2 * v * h}
    size = 4 if case["dtype"] == "fp32" else 2
    return {"bytes": case["matrices"] * case["rows"] * case["groups"] * (17 + 32 * size), "flops": 0}


def tolerance(case: dict):
    kind = case["kind"]
    if kind in ("load", "dequant"):
        return "exact"  # every MXFP4 value is exact in the output types, or rounded once
    if kind == "lm_head":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}  # float32 dot products, correctly rounded or nearly
    # bfloat16 outputs that hold a few bfloat16 roundings each
    return {"rel": 6e-3, "max": 6e-2, "differ": 0.0}


# ---- the same outputs in 64 bits ----------------------------------------------------------


def _dense(blocks, scales) -> torch.Tensor:
    """[rows, G, 16] codes and [rows, G] scales -> float64 [rows, 32 G]."""
    table = torch.tensor(FP4, dtype=torch.float64, device=blocks.device)
    pair = torch.stack((blocks & 15, blocks >> 4), dim=-1).long()  # low nibble first
    return (table[pair].reshape(*scales.shape, 32) * torch.exp2(scales.double() - 127.0).unsqueeze(-1)).flatten(-2)


def _norm_exact(x, w) -> torch.Tensor:
    """The model's RMSNorm with its bfloat16 rounding points, the mean in 64 bits."""
    r = ((x.double() ** 2).mean(dim=-1, keepdim=True).float() + EPS).double().rsqrt().float().to(torch.bfloat16)
    return x * r * w


def _select(x, t, k) -> tuple[torch.Tensor, torch.Tensor]:
    """Experts and bfloat16 softmax weights of bfloat16 logits, in torch's CPU order for ties."""
    logits = (x.double() @ t["router_w"].double().T).float() + t["router_b"].float()
    values, ids = torch.topk(logits.to(torch.bfloat16).float().cpu(), k, dim=-1)
    return ids.cuda(), torch.softmax(values, dim=-1).to(torch.bfloat16).cuda()


def _experts_exact(x, t, ids) -> tuple[torch.Tensor, torch.Tensor]:
    """Every pair's SwiGLU and expert output in float64, ``[T, k, I]`` and ``[T, k, H]``."""
    n, k = ids.shape
    gated = torch.empty((n * k, t["d_blocks"].shape[2] * 32), dtype=torch.float64, device="cuda")
    out = torch.empty((n * k, x.shape[1]), dtype=torch.float64, device="cuda")
    flat = ids.reshape(-1)
    for e in flat.unique().tolist():
        pairs = (flat == e).nonzero()[:, 0]
        gu = x[pairs // k].double() @ _dense(t["gu_blocks"][e], t["gu_scales"][e]).T + t["gu_bias"][e].double()
        gate = gu[:, 0::2].clamp(max=LIMIT)
        up = gu[:, 1::2].clamp(-LIMIT, LIMIT)
        gated[pairs] = (up + 1) * gate * torch.sigmoid(1.702 * gate)
        out[pairs] = gated[pairs] @ _dense(t["d_blocks"][e], t["d_scales"][e]).T + t["d_bias"][e].double()
    return gated.reshape(n, k, -1), out.reshape(n, k, -1)


def _attention_exact(case, t, window, position):
    x = t["x"].double()
    q, k, v = (t[f"{n}_w"].double() @ x + t[f"{n}_b"].double() for n in "qkv")
    q, k, v = (y.to(torch.bfloat16).double().view(-1, HEAD_DIM) for y in (q, k, v))
    half = HEAD_DIM // 2
    pos = 150000.0 ** (torch.arange(half, dtype=torch.float64, device="cuda") * 2 / HEAD_DIM)
    corr = [HEAD_DIM * math.log(4096 / (b * 2 * math.pi)) / (2 * math.log(150000.0)) for b in (32.0, 1.0)]
    ramp = ((torch.arange(half, dtype=torch.float64, device="cuda") - corr[0]) / (corr[1] - corr[0])).clamp(0, 1)
    inv = (1 / (32.0 * pos)) * ramp + (1 / pos) * (1 - ramp)
    # the angle is float32 in the model: at long contexts its rounding is the result's
    ang = inv.float() * float(position)
    scale = 0.1 * math.log(32.0) + 1.0
    cos, sin = ((f(ang.double()) * scale).to(torch.bfloat16).double() for f in (torch.cos, torch.sin))

    def rot(y):
        a, b = y[:, :half], y[:, half:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=1)

    qr, kr = rot(q), rot(k)
    keys = torch.cat((t["keys"][1:].double(), kr[None]))[-(window or case["context"]):]
    values = torch.cat((t["values"][1:].double(), v[None]))[-(window or case["context"]):]
    group = HEADS // KV_HEADS
    scores = torch.einsum("gjd,tgd->gjt", qr.view(KV_HEADS, group, HEAD_DIM), keys).reshape(HEADS, -1)
    scores = torch.cat((scores / math.sqrt(HEAD_DIM), t["sinks"].double()[:, None]), dim=1)
    p = torch.softmax(scores, dim=1)[:, :-1].view(KV_HEADS, group, -1)
    ctx = torch.einsum("gjt,tgd->gjd", p, values).reshape(-1)
    out = t["o_w"].double() @ ctx + t["o_b"].double()
    norms = torch.stack([y.norm() for y in (q, k, qr, kr, qr - q, kr - k)])
    return [out, norms, None]


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("moe", "block", "route"):
        outs = []
        for layer in range(case["layers"]):
            t = _layer_host(case, seed, layer)
            x = _norm_exact(t["x"], t["norm"]) if kind == "block" else t["x"]
            ids, w = _select(x, t, case["top_k"])
            gated, eo = _experts_exact(x, t, ids)
            outs.append((w.double().unsqueeze(-1) * eo).sum(dim=1))
            del t
        if kind == "moe":
            return outs
        if kind == "block":
            return outs[0] + _layer_host(case, seed, 0)["x"].double()
        one = case["tokens"] == 1
        norms = torch.stack((gated.norm(dim=-1), eo.norm(dim=-1)), dim=-1)
        return {"out": outs[0][0] if one else outs[0], "experts": None, "weights": (w[0] if one else w).double(),
                "norms": norms}
    if kind == "load":
        t = _layer_host(case, seed, 0)
        experts = sorted({(7 * seed + 5 * j) % case["experts"] for j in range(case["tokens"])})
        return [_dense(t[f"{p}_blocks"][e], t[f"{p}_scales"][e]).T.contiguous() for e in experts for p in ("gu", "d")]
    if kind == "attention":
        return [_attention_exact(case, _attention_host(case, seed, layer), window, case["context"])
                for layer, window in enumerate(_windows(case))]
    g = _gen(seed)
    if kind == "lm_head":
        w = _normal(g, (case["vocab"], case["hidden"]), 0.02)
        x = _normal(g, (case["hidden"],)).double()
        return [torch.cat([part.double() @ x for part in w.split(16384)]), None]
    n, rows, groups = case["matrices"], case["rows"], case["groups"]
    shape = (n, rows, groups) if n > 1 else (rows, groups)
    blocks, scales = _bytes(g, *shape, 16), _scales(g, *shape)
    return _dense(blocks, scales).transpose(-1, -2).contiguous()
