"""Decode attention on the device KV ring against the oracle.

Cases cover the single-split path (at most 256 keys) and the split path
with its statistics and combine launches (up to 4500 keys, 18 splits).  RoPE
and the stored keys/values are bit-exact (every bfloat16 op rounded as
torch rounds it, then the cache type's rounding); the context is within a
few cache-type ulps of |ref| plus 2^-9 of the head's largest |ref| of the
oracle (probabilities rounded to the cache type can land one unit apart when
the softmax sum is taken in another order).
"""

from __future__ import annotations

import copy
import ctypes
import threading

import numpy as np
import pytest
import torch

from klcquant_amd import _native, attention
from klcquant_amd.attention import AttentionConfig, DeviceKVCache, StreamedAttention, rope_cos_sin
from oracle import attention as oat
from oracle.numerics import bf16_to_f32, f32_to_bf16

pytestmark = pytest.mark.gpu
P = ctypes.c_void_p
CFG = dict(hidden_size=2880, num_heads=64, num_kv_heads=8, head_dim=64, rope_theta=150000.0, rope_factor=32.0,
           rope_beta_fast=32.0, rope_beta_slow=1.0, rope_original_max_position_embeddings=4096)


def bits(t: torch.Tensor) -> np.ndarray:
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def dev(b: np.ndarray, gpu) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(b).view(np.int16)).view(torch.bfloat16).to(gpu)


def context_tolerance(ref: np.ndarray, kv: str) -> np.ndarray:
    """Per-element bound for the context [heads, head_dim]: the context is rounded twice (cache
    type, then bfloat16) and a probability rounded to the cache type may land one unit off, which
    moves the head's weighted sum by at most that unit times its largest values; so a few cache-type
    ulps of |ref| plus 2^-9 of the head's largest |ref|."""
    ulp = 2.0 ** -10 if kv == "fp16" else 2.0 ** -7
    head_max = np.abs(ref).max(axis=-1, keepdims=True)
    return 4 * ulp * np.abs(ref) + 2.0 ** -8 * np.abs(ref) + 2.0 ** -9 * head_max


@pytest.mark.parametrize("kv", ["fp16", "bf16"])
@pytest.mark.parametrize("steps,cap,window,sinks", [(1, 64, None, True), (300, 512, None, True), (300, 512, 128, False),
                                                    (700, 512, None, True), (700, 1024, None, False),
                                                    (1000, 1024, 128, True), (4500, 8192, None, True),
                                                    (4500, 8192, None, False)])
def test_rope_append_and_decode_match_oracle(gpu, kv, steps, cap, window, sinks):
    cfg = AttentionConfig(**CFG)
    nh, nkv, d = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    rng = np.random.default_rng(steps * 3 + cap + (window or 0) + len(kv))
    code = 1 if kv == "fp16" else 0
    kdt = torch.float16 if kv == "fp16" else torch.bfloat16
    kc = torch.empty((cap, nkv, d), dtype=kdt, device=gpu)
    vc = torch.empty((cap, nkv, d), dtype=kdt, device=gpu)
    keys_rot, vals = [], []
    stream = P(torch.cuda.current_stream(gpu).cuda_stream)
    for pos in range(steps):
        q = f32_to_bf16(rng.standard_normal((nh, d)).astype(np.float32))
        k = f32_to_bf16(rng.standard_normal((nkv, d)).astype(np.float32))
        v = f32_to_bf16(rng.standard_normal((nkv, d)).astype(np.float32))
        cos, sin = rope_cos_sin(cfg, pos, gpu, torch.bfloat16)
        qd, kd, vd = dev(q, gpu), dev(k, gpu), dev(v, gpu)
        q_out, k_out = torch.empty_like(qd), torch.empty_like(kd)
        _native.call("klc_rope_append", P(qd.data_ptr()), P(kd.data_ptr()), P(vd.data_ptr()), P(cos.data_ptr()),
                     P(sin.data_ptr()), P(q_out.data_ptr()), P(k_out.data_ptr()), P(kc.data_ptr()), P(vc.data_ptr()),
                     pos % cap, cap, nh, nkv, d, code, stream)
        cb, sb = bits(cos), bits(sin)
        k_rot = oat.rope_rotate(k, cb, sb)
        keys_rot.append(k_rot)
        vals.append(v)
    q_rot = oat.rope_rotate(q, cb, sb)
    assert np.array_equal(bits(q_out), q_rot) and np.array_equal(bits(k_out), k_rot)
    slot = (steps - 1) % cap
    assert np.array_equal(kc[slot].float().cpu().numpy(), oat.to_kv(bf16_to_f32(k_rot), kv))
    assert np.array_equal(vc[slot].float().cpu().numpy(), oat.to_kv(bf16_to_f32(v), kv))
    held = min(steps, cap)
    count = min(held, window) if window else held
    first = (steps - count) % cap
    sk = f32_to_bf16(rng.standard_normal(nh).astype(np.float32)) if sinks else None
    skd = dev(sk, gpu) if sinks else None
    ws = torch.empty(_native.call("klc_attn_workspace_bytes", nh, d, count), dtype=torch.uint8, device=gpu)
    ctx = torch.empty((nh, d), dtype=torch.bfloat16, device=gpu)
    _native.call("klc_attn_decode", P(q_out.data_ptr()), P(kc.data_ptr()), P(vc.data_ptr()),
                 P(0 if skd is None else skd.data_ptr()), cap, first, count, nh, nkv, d, code, P(ws.data_ptr()),
                 ws.numel(), P(ctx.data_ptr()), stream)
    want, _ = oat.decode_attention(q_rot, np.stack(keys_rot[-count:]), np.stack(vals[-count:]), sk, kv=kv)
    got, ref = bf16_to_f32(bits(ctx)), bf16_to_f32(want)
    assert np.all(np.abs(got - ref) <= context_tolerance(ref, kv)), np.abs(got - ref).max()


@pytest.mark.parametrize("kv", ["fp16", "bf16"])
def test_streamed_attention_forward_matches_oracle(gpu, kv):
    """Eight decode steps through StreamedAttention.forward (sliding window 4):
    torch's projections, then the oracle's RoPE and attention."""
    cfg = AttentionConfig(**CFG, sliding_window=4)
    nh, nkv, d, h = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.hidden_size
    g = torch.Generator(device=gpu).manual_seed(11)
    pre = "model.layers.0.self_attn"

    def w(*s, scale=0.02):
        return (torch.randn(s, generator=g, device=gpu) * scale).to(torch.bfloat16)

    tensors = {f"{pre}.q_proj.weight": w(nh * d, h), f"{pre}.q_proj.bias": w(nh * d),
               f"{pre}.k_proj.weight": w(nkv * d, h), f"{pre}.k_proj.bias": w(nkv * d),
               f"{pre}.v_proj.weight": w(nkv * d, h), f"{pre}.v_proj.bias": w(nkv * d),
               f"{pre}.o_proj.weight": w(h, nh * d), f"{pre}.o_proj.bias": w(h), f"{pre}.sinks": w(nh, scale=1.0)}
    attn, cache = StreamedAttention(cfg), DeviceKVCache(gpu, precision=kv, capacity=4)
    keys, vals = [], []
    lin = torch.nn.functional.linear
    for pos in range(8):
        x = w(h, scale=1.0)
        out, diag = attn.forward(0, x, tensors, pos, cache)
        q = bits(lin(x, tensors[f"{pre}.q_proj.weight"], tensors[f"{pre}.q_proj.bias"]).view(nh, d))
        k = bits(lin(x, tensors[f"{pre}.k_proj.weight"], tensors[f"{pre}.k_proj.bias"]).view(nkv, d))
        v = bits(lin(x, tensors[f"{pre}.v_proj.weight"], tensors[f"{pre}.v_proj.bias"]).view(nkv, d))
        cos, sin = rope_cos_sin(cfg, pos, gpu, torch.bfloat16)
        q_rot, k_rot = oat.rope_rotate(q, bits(cos), bits(sin)), oat.rope_rotate(k, bits(cos), bits(sin))
        keys.append(k_rot)
        vals.append(v)
        ctx, _ = oat.decode_attention(q_rot, np.stack(keys[-4:]), np.stack(vals[-4:]), bits(tensors[f"{pre}.sinks"]), kv=kv)
        want = lin(dev(ctx, gpu).reshape(-1), tensors[f"{pre}.o_proj.weight"], tensors[f"{pre}.o_proj.bias"]).float()
        assert torch.allclose(out.float(), want, rtol=2e-2, atol=1e-2)
        assert diag["rope_position"] == pos and diag["q_post_rope_nonfinite_count"] == 0
        assert np.isclose(diag["k_post_rope_norm"], np.linalg.norm(bf16_to_f32(k_rot)), rtol=1e-5)
    assert cache.stats().tokens == 8 and cache.get(0, 4)[0].shape == (4, nkv, d)


def test_device_kv_cache_api(gpu):
    """append/get/max_tokens/snapshot/restore as kv_cache_manager.py:39-97 keep them."""
    c = DeviceKVCache(gpu, max_tokens=3, precision="bf16")
    ks = [torch.full((2, 8), float(i), dtype=torch.bfloat16, device=gpu) for i in range(5)]
    for i, k in enumerate(ks):
        c.append(1, k, -k)
    keys, values = c.get(1)
    assert keys[:, 0, 0].tolist() == [2.0, 3.0, 4.0] and values[:, 0, 0].tolist() == [-2.0, -3.0, -4.0]
    assert c.get(1, window=2)[0][:, 0, 0].tolist() == [3.0, 4.0] and c.get(7) == (None, None)
    assert c.stats().tokens == 3 and c.stats().resident_bytes == 2 * 3 * 16 * 2
    snap = c.snapshot()
    c.clear()
    assert c.get(1) == (None, None)
    c.restore(snap)
    assert c.get(1)[0][:, 0, 0].tolist() == [2.0, 3.0, 4.0]
    g = DeviceKVCache(gpu, precision="fp16", capacity=2)  # unbounded: grows past its capacity
    for i, k in enumerate(ks):
        g.append(0, k, k)
    assert g.get(0)[0].dtype == torch.float16 and g.get(0)[0][:, 0, 0].tolist() == [0.0, 1.0, 2.0, 3.0, 4.0]
    with pytest.raises(ValueError):
        DeviceKVCache(gpu, precision="q8")


@pytest.mark.parametrize("nh,nkv,d", [(32, 2, 128), (8, 8, 8), (12, 4, 24)])
@pytest.mark.parametrize("window", [None, 100])
def test_other_head_shapes(gpu, nh, nkv, d, window):
    """Group sizes 16, 1 and 3 and head dims 128, 8 and 24 (a value-slice
    count that does not divide the workgroup), bf16 cache, 300 steps."""
    cfg = AttentionConfig(hidden_size=nh * d, num_heads=nh, num_kv_heads=nkv, head_dim=d, rope_factor=8.0)
    rng = np.random.default_rng(nh * 1000 + d + (window or 0))
    cap, steps = 512, 300
    kc = torch.empty((cap, nkv, d), dtype=torch.bfloat16, device=gpu)
    vc = torch.empty((cap, nkv, d), dtype=torch.bfloat16, device=gpu)
    stream = P(torch.cuda.current_stream(gpu).cuda_stream)
    keys, vals = [], []
    for pos in range(steps):
        q = f32_to_bf16(rng.standard_normal((nh, d)).astype(np.float32))
        k = f32_to_bf16(rng.standard_normal((nkv, d)).astype(np.float32))
        v = f32_to_bf16(rng.standard_normal((nkv, d)).astype(np.float32))
        cos, sin = rope_cos_sin(cfg, pos, gpu, torch.bfloat16)
        qd, kd, vd = dev(q, gpu), dev(k, gpu), dev(v, gpu)
        q_out = torch.empty_like(qd)
        _native.call("klc_rope_append", P(qd.data_ptr()), P(kd.data_ptr()), P(vd.data_ptr()), P(cos.data_ptr()),
                     P(sin.data_ptr()), P(q_out.data_ptr()), None, P(kc.data_ptr()), P(vc.data_ptr()), pos % cap,
                     cap, nh, nkv, d, 0, stream)
        keys.append(oat.rope_rotate(k, bits(cos), bits(sin)))
        vals.append(v)
    q_rot = oat.rope_rotate(q, bits(cos), bits(sin))
    assert np.array_equal(bits(q_out), q_rot)
    count = min(steps, window) if window else steps
    sk = f32_to_bf16(rng.standard_normal(nh).astype(np.float32))
    skd = dev(sk, gpu)
    ws = torch.empty(_native.call("klc_attn_workspace_bytes", nh, d, count), dtype=torch.uint8, device=gpu)
    ctx = torch.empty((nh, d), dtype=torch.bfloat16, device=gpu)
    _native.call("klc_attn_decode", P(q_out.data_ptr()), P(kc.data_ptr()), P(vc.data_ptr()), P(skd.data_ptr()), cap,
                 steps - count, count, nh, nkv, d, 0, P(ws.data_ptr()), ws.numel(), P(ctx.data_ptr()), stream)
    want, _ = oat.decode_attention(q_rot, np.stack(keys[-count:]), np.stack(vals[-count:]), sk, kv="bf16")
    got, ref = bf16_to_f32(bits(ctx)), bf16_to_f32(want)
    assert np.all(np.abs(got - ref) <= context_tolerance(ref, "bf16")), np.abs(got - ref).max()


def decode_direct(gpu, q, k, v, sk, cap, first, count, kv):
    """klc_attn_decode on ready tensors with a workspace of exactly the stated size, dirty."""
    (nh, d), nkv = q.shape, k.shape[1]
    ws = torch.full((_native.call("klc_attn_workspace_bytes", nh, d, count),), 255, dtype=torch.uint8, device=gpu)
    ctx = torch.empty((nh, d), dtype=torch.bfloat16, device=gpu)
    _native.call("klc_attn_decode", P(q.data_ptr()), P(k.data_ptr()), P(v.data_ptr()),
                 P(0 if sk is None else sk.data_ptr()), cap, first, count, nh, nkv, d, 1 if kv == "fp16" else 0,
                 P(ws.data_ptr()), ws.numel(), P(ctx.data_ptr()), P(torch.cuda.current_stream(gpu).cuda_stream))
    return ctx


@pytest.mark.parametrize("nh,nkv,d,count,kv", [
    (64, 8, 64, 257, "fp16"), (64, 8, 64, 321, "bf16"), (64, 8, 64, 8192, "fp16"), (64, 8, 64, 8193, "fp16"),
    (32, 2, 128, 8449, "bf16"), (32, 2, 128, 400, "fp16"), (12, 4, 24, 1000, "bf16"), (5, 1, 40, 8195, "fp16"),
    (8, 8, 8, 700, "bf16"), (3, 3, 104, 9001, "bf16")])
def test_split_decode_matches_oracle(gpu, nh, nkv, d, count, kv):
    """Both score-block and value-split sizes (the line is at 8,192 keys), partial blocks, group
    sizes 1 to 16, head dims that leave dim quarters and threads idle, a wrapped span."""
    g = torch.Generator(device=gpu).manual_seed(count + d)
    dt = torch.float16 if kv == "fp16" else torch.bfloat16
    cap, first = count + 9, count - 3  # the span wraps after 12 keys
    q = torch.randn(nh, d, generator=g, device=gpu).to(torch.bfloat16)
    k, v = (torch.randn(cap, nkv, d, generator=g, device=gpu).to(dt) for _ in range(2))
    sk = torch.randn(nh, generator=g, device=gpu).to(torch.bfloat16)
    ctx = decode_direct(gpu, q, k, v, sk, cap, first, count, kv)
    idx = (torch.arange(count, device=gpu) + first) % cap
    kd, vd = k[idx].double(), v[idx].double()
    s = torch.einsum("gjd,tgd->gjt", q.double().cpu().view(nkv, nh // nkv, d), kd.cpu()).reshape(nh, count)
    s = torch.cat((s.float() / np.float32(np.sqrt(d)), sk.float().cpu()[:, None]), dim=1)
    p = torch.softmax(s.double(), dim=1)[:, :-1].float().to(dt).double().view(nkv, nh // nkv, count)
    ref = torch.einsum("gjt,tgd->gjd", p, vd.cpu()).reshape(nh, d)
    ref = ref.float().to(dt).to(torch.bfloat16).float().numpy()
    got = ctx.float().cpu().numpy()
    assert np.all(np.abs(got - ref) <= context_tolerance(ref, kv)), np.abs(got - ref).max()


@pytest.mark.parametrize("nh,nkv,d,count,kv", [
    (8, 1, 64, 65537, "fp16"), (2, 1, 128, 66001, "bf16"), (16, 1, 128, 65800, "fp16"), (3, 1, 64, 131073, "bf16"),
    (8, 1, 64, 65536, "fp16")])
def test_long_split_decode_matches_oracle(gpu, nh, nkv, d, count, kv):
    """Score blocks of 256 keys (past 65,536 keys), more of them than a value workgroup holds statistics of."""
    test_split_decode_matches_oracle(gpu, nh, nkv, d, count, kv)


def test_split_decode_infinite_scores(gpu):
    """A score block that is -inf throughout weighs nothing; a NaN key makes its KV head's queries NaN."""
    nh, nkv, d, count = 16, 2, 64, 600
    g = torch.Generator(device=gpu).manual_seed(1)
    q = torch.full((nh, d), 3e38, device=gpu).to(torch.bfloat16)
    k = torch.zeros(count, nkv, d, device=gpu, dtype=torch.bfloat16)
    k[64:256] = -3e38
    v = torch.randn(count, nkv, d, generator=g, device=gpu).to(torch.bfloat16)
    ctx = decode_direct(gpu, q, k, v, None, count, 0, count, "bf16").float()
    keep = torch.cat((v[:64], v[256:])).float()
    p = torch.tensor(1.0 / keep.shape[0]).to(torch.bfloat16).item()
    ref = (p * keep.sum(dim=0)).repeat_interleave(nh // nkv, dim=0)
    assert torch.allclose(ctx, ref, rtol=2.0 ** -7, atol=2.0 ** -9)
    k[300, 1, 5] = float("nan")
    ctx = decode_direct(gpu, q, k, v, None, count, 0, count, "bf16").float()
    assert torch.isfinite(ctx[: nh // 2]).all() and torch.isnan(ctx[nh // 2:]).all()


def step_tensors(gpu, g, nh, nkv, d, h, rows, pre, sinks=True):
    def w(*s, scale=0.02):
        return (torch.randn(s, generator=g, device=gpu) * scale).to(torch.bfloat16)

    t = {f"{pre}.{n}_proj.weight": w(r, c) for n, r, c in (("q", nh * d, h), ("k", nkv * d, h), ("v", nkv * d, h),
                                                           ("o", rows, nh * d))}
    t |= {f"{pre}.{n}_proj.bias": w(r) for n, r in (("q", nh * d), ("k", nkv * d), ("v", nkv * d), ("o", rows))}
    if sinks:
        t[f"{pre}.sinks"] = w(nh, scale=1.0)
    return t


@pytest.mark.parametrize("nh,nkv,d,h,rows,count,position,kv,sinks", [
    (64, 8, 64, 2880, 2880, 128, 131071, "fp16", True), (64, 8, 64, 2880, 2880, 900, 0, "bf16", True),
    (4, 4, 8, 8, 1, 1, 5, "fp16", False), (32, 2, 128, 4096, 33, 257, 99999, "bf16", True),
    (6, 2, 24, 520, 77, 300, 4095, "fp16", True), (16, 1, 40, 1544, 512, 256, 70000, "bf16", False)])
def test_attention_step_matches_oracle(gpu, nh, nkv, d, h, rows, count, position, kv, sinks):
    """klc_attn_step's stages, each exactly from the one before: correctly rounded projections (the
    float64 sum rounded to float32 and bfloat16), RoPE with torch's own tables and the stored key and
    value bit for bit, the context and output within their bounds, the diagnostics."""
    g = torch.Generator(device=gpu).manual_seed(nh * d + h)
    pre = "model.layers.3.self_attn"
    cfg = AttentionConfig(hidden_size=h, num_heads=nh, num_kv_heads=nkv, head_dim=d, rope_factor=32.0)
    t = step_tensors(gpu, g, nh, nkv, d, h, rows, pre, sinks)
    x = torch.randn(h, generator=g, device=gpu).to(torch.bfloat16)
    cache = DeviceKVCache(gpu, max_tokens=count, precision=kv)
    ring, _ = cache.next_slot(3, nkv, d)
    ring["k"].copy_(torch.randn(ring["k"].shape, generator=g, device=gpu))
    ring["v"].copy_(torch.randn(ring["v"].shape, generator=g, device=gpu))
    ring["total"] = count + 1  # the token goes to slot 1 % count
    attn = StreamedAttention(cfg)
    assert attn._step(3, x, t, position, cache, None) is not None, "the one-call path did not take these tensors"
    ring["total"] = count + 1
    out, diag = attn.forward(3, x, t, position, cache)
    assert ring["total"] == count + 2

    def proj(n, heads):
        y = t[f"{pre}.{n}_proj.weight"].double().cpu() @ x.double().cpu() + t[f"{pre}.{n}_proj.bias"].double().cpu()
        return f32_to_bf16(y.float().numpy()).reshape(heads, d)

    q, k, v = proj("q", nh), proj("k", nkv), proj("v", nkv)
    cos, sin = rope_cos_sin(cfg, position, gpu, torch.bfloat16)
    q_rot, k_rot = oat.rope_rotate(q, bits(cos), bits(sin)), oat.rope_rotate(k, bits(cos), bits(sin))
    slot = (count + 1) % count
    assert np.array_equal(ring["k"][slot].float().cpu().numpy(), oat.to_kv(bf16_to_f32(k_rot), kv))
    assert np.array_equal(ring["v"][slot].float().cpu().numpy(), oat.to_kv(bf16_to_f32(v), kv))
    order = [(slot + 1 + i) % count for i in range(count)]  # the appended token last
    sk = t[f"{pre}.sinks"] if sinks else None
    ctx = decode_direct(gpu, dev(q_rot, gpu), ring["k"], ring["v"], sk, count, order[0], count, kv)
    want = t[f"{pre}.o_proj.weight"].double() @ ctx.reshape(-1).double() + t[f"{pre}.o_proj.bias"].double()
    assert torch.equal(out, want.float().to(torch.bfloat16))
    ref = {"q_pre_rope_norm": q, "k_pre_rope_norm": k, "q_post_rope_norm": q_rot, "k_post_rope_norm": k_rot}
    for name, rows_ in ref.items():
        assert np.isclose(diag[name], np.linalg.norm(bf16_to_f32(rows_).astype(np.float64)), rtol=1e-6)
    for name, a, b in (("q_rope_delta_norm", q_rot, q), ("k_rope_delta_norm", k_rot, k)):
        assert np.isclose(diag[name], np.linalg.norm((bf16_to_f32(a) - bf16_to_f32(b)).astype(np.float64)), rtol=1e-6)
    assert diag["q_post_rope_nonfinite_count"] == diag["k_post_rope_nonfinite_count"] == 0
    assert diag["rope_position"] == position and diag["sliding_window"] is None


def test_attention_step_and_general_path_agree(gpu):
    """The same step through the one call and, with gradients asked for, through F.linear; non-finite
    values are counted by both."""
    nh, nkv, d, h = 64, 8, 64, 2880
    g = torch.Generator(device=gpu).manual_seed(5)
    pre = "model.layers.0.self_attn"
    t = step_tensors(gpu, g, nh, nkv, d, h, h, pre)
    cfg = AttentionConfig(**CFG, sliding_window=4)
    for poison in (False, True):
        x = torch.randn(h, generator=g, device=gpu).to(torch.bfloat16)
        if poison:
            x[7] = float("inf")
        outs, diags = [], []
        for grad in (False, True):
            w = {n: v.clone().requires_grad_(grad and n.endswith("o_proj.weight")) for n, v in t.items()}
            cache = DeviceKVCache(gpu, precision="fp16", capacity=4)
            attn = StreamedAttention(cfg)
            assert (attn._step(0, x, w, 3, DeviceKVCache(gpu, capacity=4), None) is None) == grad
            for pos in range(3):
                out, diag = attn.forward(0, x, w, pos, cache)
                attn = copy.deepcopy(attn)  # with its records and tables
            outs.append(out)
            diags.append(diag)
        assert outs[1].requires_grad and not outs[0].requires_grad
        assert torch.allclose(outs[0].float(), outs[1].float(), rtol=2e-2, atol=1e-2, equal_nan=True)
        assert diags[0].keys() == diags[1].keys()
        for name in diags[0]:
            assert diags[0][name] == diags[1][name] or np.isclose(diags[0][name], diags[1][name], rtol=1e-4, equal_nan=True)
        if poison:
            assert diags[0]["q_post_rope_nonfinite_count"] > 0


def test_attention_step_interrupted_wait_keeps_the_record(gpu, monkeypatch):
    """An exception in the wait leaves only after the stream is done with the record (whose memory could
    otherwise be another tensor's by then), and the next step, with a tag of its own, reads its own values."""
    nh, nkv, d, h = 64, 8, 64, 2880
    g = torch.Generator(device=gpu).manual_seed(9)
    pre = "model.layers.0.self_attn"
    t = step_tensors(gpu, g, nh, nkv, d, h, h, pre)
    attn, cache = StreamedAttention(AttentionConfig(**CFG)), DeviceKVCache(gpu, capacity=8)
    x = torch.randn(h, generator=g, device=gpu).to(torch.bfloat16)
    busy = torch.randn(4096, 4096, generator=g, device=gpu)
    seen = []

    def interrupted(record, dev, limit_s):
        seen.append((record, int(record.words[8])))
        raise KeyboardInterrupt

    with monkeypatch.context() as m:
        m.setattr(attention._HostRecord, "wait", interrupted)
        for _ in range(40):
            busy = busy @ busy * 1e-4  # a queue ahead of the step
        with pytest.raises(KeyboardInterrupt):
            attn.forward(0, x, t, 0, cache)
    (record, before), = seen
    assert before == 0 and record.words[8] == record.tag == 1 and attention._UNSETTLED == []
    attn._records.append(record)
    _, diag = attn.forward(0, 2 * x, t, 1, cache)
    assert record.words[8] == record.tag == 2
    q = torch.nn.functional.linear(2 * x, t[f"{pre}.q_proj.weight"], t[f"{pre}.q_proj.bias"])
    assert np.isclose(diag["q_pre_rope_norm"], q.float().norm().item(), rtol=1e-3)


def test_attention_step_wait_past_its_limit(gpu, monkeypatch):
    """Behind a queue longer than the wait's limit the step synchronises its stream: the same results."""
    nh, nkv, d, h = 8, 2, 64, 256
    g = torch.Generator(device=gpu).manual_seed(10)
    t = step_tensors(gpu, g, nh, nkv, d, h, h, "model.layers.0.self_attn")
    cfg = AttentionConfig(hidden_size=h, num_heads=nh, num_kv_heads=nkv, head_dim=d)
    x = torch.randn(h, generator=g, device=gpu).to(torch.bfloat16)
    want = StreamedAttention(cfg).forward(0, x, t, 5, DeviceKVCache(gpu, capacity=8))
    busy = torch.randn(4096, 4096, generator=g, device=gpu)
    monkeypatch.setattr(StreamedAttention, "_RECORD_WAIT_S", 0.0)
    monkeypatch.setattr(attention._HostRecord, "_SLICE_US", 1)
    for _ in range(40):
        busy = busy @ busy * 1e-4
    out, diag = StreamedAttention(cfg).forward(0, x, t, 5, DeviceKVCache(gpu, capacity=8))
    assert torch.equal(out, want[0]) and diag == want[1]


def test_attention_step_keeps_a_caches_own_span(gpu):
    """A cache class that chooses the keys itself (here the last two) is asked for them."""
    class LastTwo(DeviceKVCache):
        @staticmethod
        def _span(r, window):
            return DeviceKVCache._span(r, min(window or 2, 2))

    nh, nkv, d, h = 8, 2, 64, 256
    g = torch.Generator(device=gpu).manual_seed(11)
    t = step_tensors(gpu, g, nh, nkv, d, h, h, "model.layers.0.self_attn")
    attn = StreamedAttention(AttentionConfig(hidden_size=h, num_heads=nh, num_kv_heads=nkv, head_dim=d))
    xs = torch.randn(6, h, generator=g, device=gpu).to(torch.bfloat16)
    own, windowed = LastTwo(gpu, capacity=16), DeviceKVCache(gpu, capacity=16)
    for pos in range(6):
        got, _ = attn.forward(0, xs[pos], t, pos, own)
        want, _ = attn.forward(0, xs[pos], t, pos, windowed, sliding_window=2)
        assert torch.allclose(got.float(), want.float(), rtol=2e-2, atol=1e-2)


def small_step(gpu, seed, capacity=8, kv="fp16"):
    """A small layer: (attention, hidden, tensors, a fresh cache)."""
    nh, nkv, d, h = 8, 2, 64, 256
    g = torch.Generator(device=gpu).manual_seed(seed)
    t = step_tensors(gpu, g, nh, nkv, d, h, h, "model.layers.0.self_attn")
    attn = StreamedAttention(AttentionConfig(hidden_size=h, num_heads=nh, num_kv_heads=nkv, head_dim=d))
    return attn, torch.randn(h, generator=g, device=gpu).to(torch.bfloat16), t, DeviceKVCache(gpu, capacity=capacity,
                                                                                            precision=kv)


def test_attention_step_leaves_watched_calls_to_torch(gpu):
    """Under anything that watches or replaces torch calls the one-call step declines, touching neither the
    cache nor the stream (a capture holds nothing of it)."""
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    attn, x, t, cache = small_step(gpu, 12)
    declined = []

    def step(y=None):
        declined.append(attn._step(0, x, t, 0, cache, None) is None)
        return None if y is None else y + 1

    with torch.autocast("cuda", dtype=torch.bfloat16):
        step()
    with Functions():
        step()
    with Dispatch():
        step()
    with forward_ad.dual_level():
        step()
    torch.func.vmap(step)(torch.zeros(2, device=gpu))
    torch.jit.trace(step, (torch.zeros(2, device=gpu),), check_trace=False)
    y = torch.zeros(4, device=gpu)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        z = step(y)
    for n in range(3):
        y.fill_(n)
        graph.replay()
        torch.cuda.synchronize()
        assert z.tolist() == [n + 1.0] * 4
    assert len(declined) >= 7 and all(declined) and not cache.layers
    assert attn._step(0, x, t, 0, cache, None) is not None


def test_attention_step_leaves_other_tensors_to_torch(gpu):
    """Weights and inputs that the one call does not take as they lie give the general path's results:
    the same values in another layout, type or class."""
    class Sub(torch.Tensor):
        pass

    pre = "model.layers.0.self_attn"
    attn, x, t, cache = small_step(gpu, 13)
    want, _ = attn.forward(0, x, t, 7, cache)
    strided = torch.empty(512, device=gpu, dtype=torch.bfloat16)[::2]
    strided.copy_(x)
    shifted_x = torch.empty(257, device=gpu, dtype=torch.bfloat16)[1:]
    shifted_x.copy_(x)
    q = t[f"{pre}.q_proj.weight"]
    shifted = torch.empty(q.numel() + 1, device=gpu, dtype=torch.bfloat16)[1:].view(q.shape)
    shifted.copy_(q)
    for hidden, change in (
            (strided, {}), (shifted_x, {}), (x.as_subclass(Sub), {}),
            (x, {"q_proj.weight": shifted}), (x, {"q_proj.weight": q.t().contiguous().t()}),
            (x, {"k_proj.weight": t[f"{pre}.k_proj.weight"].as_subclass(Sub)}),
            (x, {"sinks": t[f"{pre}.sinks"].float()}),
            (x, {"o_proj.weight": torch.nn.Parameter(t[f"{pre}.o_proj.weight"])})):
        tensors = t | {f"{pre}.{n}": v for n, v in change.items()}
        assert attn._step(0, hidden, tensors, 7, DeviceKVCache(gpu, capacity=8), None) is None, change.keys()
        out, _ = attn.forward(0, hidden, tensors, 7, DeviceKVCache(gpu, capacity=8))
        assert torch.allclose(out.float().detach(), want.float(), rtol=2e-2, atol=1e-2)
    with torch.no_grad():  # nothing for autograd to see
        p = t | {n: torch.nn.Parameter(v) for n, v in t.items()}
        assert torch.equal(attn._step(0, x, p, 7, DeviceKVCache(gpu, capacity=8), None)[0], want)
    # biases and sinks are read two bytes at a time, so they may lie anywhere; no bias tensor: the general path
    def odd(v):
        w = torch.empty(v.numel() + 1, device=gpu, dtype=torch.bfloat16)[1:]
        w.copy_(v)
        return w

    moved = {n: odd(v) if v.dim() == 1 else v for n, v in t.items()}
    assert torch.equal(attn._step(0, x, moved, 7, DeviceKVCache(gpu, capacity=8), None)[0], want)
    out, _ = attn.forward(0, x, t | {f"{pre}.q_proj.bias": None}, 7, DeviceKVCache(gpu, capacity=8))
    zero = torch.zeros_like(t[f"{pre}.q_proj.bias"])
    ref, _ = attn.forward(0, x, t | {f"{pre}.q_proj.bias": zero}, 7, DeviceKVCache(gpu, capacity=8))
    assert torch.allclose(out.float(), ref.float(), rtol=2e-2, atol=1e-2)


def test_attention_step_on_streams_and_threads(gpu):
    """Two threads with a stream and a cache each, on one StreamedAttention, give a single thread's bits."""
    attn, _, t, _ = small_step(gpu, 14)
    g = torch.Generator(device=gpu).manual_seed(15)
    xs = torch.randn(2, 300, 256, generator=g, device=gpu).to(torch.bfloat16)
    torch.cuda.synchronize()

    def run(i, results):
        with torch.cuda.stream(torch.cuda.Stream(gpu)):
            cache = DeviceKVCache(gpu, capacity=512)
            results[i] = [attn.forward(0, xs[i, pos], t, pos, cache) for pos in range(300)]
            torch.cuda.current_stream(gpu).synchronize()

    alone, together = {}, {}
    for i in range(2):
        run(i, alone)
    threads = [threading.Thread(target=run, args=(i, together)) for i in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for i in range(2):
        for (a, da), (b, db) in zip(alone[i], together[i]):
            assert torch.equal(a, b) and da == db
    assert len(attn._records) <= 16


def test_attention_rejects_bad_shapes(gpu):
    x = torch.zeros(4096, dtype=torch.bfloat16, device=gpu)
    ws = torch.zeros(1 << 16, dtype=torch.uint8, device=gpu)
    stream = P(torch.cuda.current_stream(gpu).cuda_stream)

    def decode(nh, nkv, d, count=4, cap=8, first=0):
        with pytest.raises(_native.KlcError) as exc:
            _native.call("klc_attn_decode", P(x.data_ptr()), P(x.data_ptr()), P(x.data_ptr()), None, cap, first,
                         count, nh, nkv, d, 0, P(ws.data_ptr()), ws.numel(), P(x.data_ptr()), stream)
        return exc.value.status

    assert decode(34, 2, 64) == -2      # group of 17 > 16
    assert decode(8, 8, 136) == -2      # head_dim above 128
    assert decode(8, 8, 12) == -2       # head_dim not a multiple of 8
    assert decode(8, 3, 64) == -2       # heads not a multiple of KV heads
    assert decode(8, 8, 64, count=9) == -1   # more keys than the ring holds
    assert decode(8, 8, 64, first=8) == -1   # first slot outside the ring
    with pytest.raises(_native.KlcError) as exc:
        _native.call("klc_rope_append", P(x.data_ptr()), P(x.data_ptr()), P(x.data_ptr()), P(x.data_ptr()),
                     P(x.data_ptr()), P(x.data_ptr()), None, P(x.data_ptr()), P(x.data_ptr()), 8, 8, 8, 8, 64, 0,
                     stream)
    assert exc.value.status == -1       # slot == cap
