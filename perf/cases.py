"""Measured workloads of the library: what its users run, over the sizes they run it at.

    listed()              the named cases
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   what a user's program holds before the call
    run(state)            one pass through the public entry points
    work(case)            bytes and operations one pass cannot do without
    tolerance(case)       how far two correct implementations may lie apart
    exact(case, seed)     the same results in 64 bits, in plain torch

The operations ("op" of a case):
    call     lb.gemm_*(x, D): numpy in, numpy out, weights resident (the drop-in Python call)
    gemm     y = x . w^T on device pointers: decode (M <= 4), batched decode and prompts,
             with the kernel and weight layout that a resident program takes for the shape
    attend   causal attention of a prompt's T tokens behind `past` cached ones
    step     one decode token: rotary embedding, cache write and attention over the cache
    pack     fp32 weights -> packed int4 / MXFP4 on the device
    answer   the decoder: a prompt, then greedy tokens, then the next token's logits
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import torch

import lowbit_amd as lb
from lowbit_amd import kernels as K
from lowbit_amd import model as M

KINDS = {"w4a16": 0, "mxfp4": 1, "w4a8": 2}


# ---------------------------------------------------------------- cases

def listed() -> list[dict]:
    return [
        # the drop-in call with host activations, at one token: latency and launches
        {"name": "call-w4a8-1", "op": "call", "fmt": "w4a8", "asym": True, "m": 1, "n": 4096, "k": 4096},
        # one decode token through the up projection of a 7B MLP: the headline shape
        {"name": "decode-w4a8-1", "op": "gemm", "fmt": "w4a8", "asym": True, "m": 1, "n": 11008, "k": 4096},
        # three sequences decoded together, down projection (long rows)
        {"name": "decode-mxfp4-3", "op": "gemm", "fmt": "mxfp4", "asym": False, "m": 3, "n": 4096, "k": 11008},
        # a batch of 16 sequences, up projection
        {"name": "batch-w4a16-16", "op": "gemm", "fmt": "w4a16", "asym": True, "m": 16, "n": 11008, "k": 4096},
        # a batch of 64 sequences
        {"name": "batch-w4a8-64", "op": "gemm", "fmt": "w4a8", "asym": True, "m": 64, "n": 11008, "k": 4096},
        # prompts: a square projection, a ragged prompt through the down projection, a long one
        {"name": "prompt-w4a16-512", "op": "gemm", "fmt": "w4a16", "asym": True, "m": 512, "n": 4096, "k": 4096},
        {"name": "prompt-mxfp4-777", "op": "gemm", "fmt": "mxfp4", "asym": False, "m": 777, "n": 4096, "k": 11008},
        {"name": "prompt-w4a8-2048", "op": "gemm", "fmt": "w4a8", "asym": False, "m": 2048, "n": 11008, "k": 4096},
        # attention of the 0.5B decoder (14 heads on 2, 64 wide): a prompt, and a late decode token
        {"name": "attend-1000", "op": "attend", "t": 1000, "past": 0, "h": 14, "kv": 2, "d": 64},
        {"name": "step-4096", "op": "step", "past": 3500, "cap": 4096, "h": 14, "kv": 2, "d": 64},
        # quantizing one 7B MLP matrix when a model is loaded
        {"name": "pack-int4", "op": "pack", "fmt": "int4", "asym": True, "group": 128, "n": 4096, "k": 11008},
        # four layers of the 0.5B decoder answering: prompt, then greedy decoding
        {"name": "answer-w4a16", "op": "answer", "fmt": "w4a16", "shape": "qwen", "layers": 4, "t": 384, "new": 16},
    ]


def _spread(rng, lo: int, hi: int, step: int = 1) -> int:
    """A multiple of `step` between lo and hi, even over the logarithm."""
    v = lo * (hi / lo) ** rng.random()
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng) -> dict:
    op = rng.choice(["gemm"] * 6 + ["attend", "attend", "step", "pack", "pack", "call", "answer"])
    if op in ("gemm", "call"):
        fmt = rng.choice(["w4a16", "mxfp4", "w4a8"])
        m = _spread(rng, 1, 2048) if op == "gemm" else _spread(rng, 1, 32)
        n = _spread(rng, 256, 14336) if rng.random() < 0.5 else _spread(rng, 256, 14336, 128)
        k = _spread(rng, 256, 11008, 32 if fmt == "mxfp4" else 128)
        while m * n * k > 30e9:
            m = (m + 1) // 2
        case = {"op": op, "fmt": fmt, "asym": fmt != "mxfp4" and rng.random() < 0.6, "m": m, "n": n, "k": k}
        if op == "gemm" and fmt != "mxfp4" and m <= 4 and rng.random() < 0.3:
            case["group"] = 32  # finer scales: a decode option
        return case
    if op in ("attend", "step"):
        d = rng.choice([32, 64, 64, 128, 128])
        kv = rng.choice([1, 2, 4, 8])
        h = kv * rng.choice([1, 2, 4, 7])
        if op == "attend":
            t = _spread(rng, 16, 1536)
            past = rng.choice([0, 0, _spread(rng, 16, 1024)])
            return {"op": op, "t": t, "past": past, "h": min(h, kv * (32 // kv)), "kv": kv, "d": d}
        cap = _spread(rng, 64, 8192)
        return {"op": op, "past": rng.randrange(cap // 4, cap), "cap": cap, "h": h, "kv": kv, "d": d}
    if op == "pack":
        fmt = rng.choice(["int4", "mxfp4"])
        group = rng.choice([128, 128, 32]) if fmt == "int4" else 32
        n, k = _spread(rng, 128, 11008), _spread(rng, 200, 11008, rng.choice([1, 32, 128]))
        return {"op": op, "fmt": fmt, "asym": fmt == "int4" and rng.random() < 0.5, "group": group, "n": n, "k": k}
    return {"op": "answer", "fmt": rng.choice(["w4a16", "mxfp4"]), "shape": rng.choice(["qwen", "wide"]),
            "layers": rng.choice([2, 3, 4]), "t": _spread(rng, 8, 512), "new": rng.randrange(2, 17)}


# ---------------------------------------------------------------- inputs, in plain torch

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _acts(g, m: int, k: int) -> torch.Tensor:
    """Hidden states: normal, with the few large channels decoders have."""
    x = torch.randn(m, k, generator=g, device="cuda")
    big = torch.rand(k, generator=g, device="cuda") < 1 / 256
    return torch.where(big, x * 8, x)


def _pad(t: torch.Tensor, block: int) -> torch.Tensor:
    return torch.nn.functional.pad(t, (0, -t.shape[1] % block))


def _nibbles(codes: torch.Tensor, block: int) -> torch.Tensor:
    """uint8 codes [N, Kp] -> bytes: element j of a block in the low nibble of byte j,
    element j + block/2 in the high one."""
    c = codes.reshape(codes.shape[0], -1, 2, block // 2)
    return (c[:, :, 0] | (c[:, :, 1] << 4)).reshape(codes.shape[0], -1)


def _int4(w: torch.Tensor, asym: bool, group: int = 128):
    """(codes uint8 [N, Kp], scales [N, G], zeros [N, G] or None) of fp32 w [N, K]."""
    n, k = w.shape
    b = _pad(w, group).reshape(n, -1, group)
    if asym:
        hi, lo = b.amax(2).clamp(min=0), b.amin(2).clamp(max=0)
        s = (hi - lo) / 15
        s = torch.where(s > 0, s, torch.ones_like(s))
        z = torch.round(-lo / s).clamp(0, 15)
        q = (torch.round(b / s[:, :, None]) + z[:, :, None]).clamp(0, 15)
        real = (torch.arange(b.shape[1] * group, device=w.device) < k).reshape(1, -1, group)
        q = torch.where(real, q, z[:, :, None].expand_as(q))
    else:
        s = b.abs().amax(2) / 7
        s = torch.where(s > 0, s, torch.ones_like(s))
        z = None
        q = torch.round(b / s[:, :, None]).clamp(-8, 7) + 8
    return q.to(torch.uint8).reshape(n, -1), s, None if z is None else z.to(torch.uint8)


def _mxfp4(w: torch.Tensor):
    """(E2M1 codes uint8 [N, Kp], E8M0 exponents uint8 [N, Kp/32]) of fp32 w [N, K]."""
    n = w.shape[0]
    b = _pad(w, 32).reshape(n, -1, 32)
    amax = b.abs().amax(2)
    e = torch.floor(torch.log2(amax.double()).float()) - 2 + 127
    e = torch.where(amax > 0, e, torch.full_like(e, 127)).clamp(0, 254)
    v = b / torch.pow(2.0, e.double() - 127)[:, :, None]
    a = v.abs()
    mag = sum((a >= t if up else a > t).to(torch.uint8)
              for t, up in ((.25, 0), (.75, 1), (1.25, 0), (1.75, 1), (2.5, 0), (3.5, 1), (5.0, 0)))
    codes = mag | (((v < 0) & (mag > 0)).to(torch.uint8) << 3)
    return codes.reshape(n, -1), e.to(torch.uint8)


def _dense(fmt: str, packed, group: int = 128) -> torch.Tensor:
    """float64 [N, Kp] that the packed weights stand for."""
    if fmt == "mxfp4":
        codes, e = packed
        val = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], device=codes.device, dtype=torch.float64)
        v = val[(codes & 7).long()] * torch.where(codes & 8 > 0, -1.0, 1.0)
        s = torch.pow(2.0, e.double() - 127)
        return (v.reshape(v.shape[0], -1, 32) * s[:, :, None]).reshape(v.shape)
    codes, s, z = packed
    q = codes.double().reshape(codes.shape[0], -1, group)
    zero = 8.0 if z is None else z.double()[:, :, None]
    return ((q - zero) * s.double()[:, :, None]).reshape(codes.shape)


def _packed(case: dict, w: torch.Tensor):
    return _mxfp4(w) if case["fmt"] == "mxfp4" else _int4(w, case["asym"], case.get("group", 128))


def _gemm_inputs(case: dict, seed: int):
    g = _gen(seed)
    w = torch.randn(case["n"], case["k"], generator=g, device="cuda") * 0.02
    return _packed(case, w), _acts(g, case["m"], case["k"])


def _attn_inputs(case: dict, seed: int):
    """qkv rows of the new tokens (q widened: scores spread over several units), the
    caches and the rotary tables."""
    g = _gen(seed)
    h, kv, d, past = case["h"], case["kv"], case["d"], case["past"]
    t = case.get("t", 1)
    cap = case.get("cap", past + t)
    qkv = torch.randn(t, (h + 2 * kv) * d, generator=g, device="cuda")
    qkv[:, : h * d] *= 2
    kc = torch.randn(kv, cap, d, generator=g, device="cuda")
    vc = torch.randn(kv, cap, d, generator=g, device="cuda")
    inv = 1.0 / 1e6 ** (torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    ang = torch.arange(cap, device="cuda", dtype=torch.float64)[:, None] * inv
    return qkv, kc, vc, ang.cos().float(), ang.sin().float()


def _config(case: dict) -> M.ModelConfig:
    if case["shape"] == "qwen":
        return M.qwen2_config(num_layers=case["layers"], vocab_size=32768, max_position=2048)
    return M.ModelConfig(vocab_size=32000, hidden_size=1024, intermediate_size=2816, num_layers=case["layers"],
                         num_heads=8, num_kv_heads=2, head_dim=128, max_position=2048)


def _model_weights(cfg: M.ModelConfig, seed: int) -> dict:
    g = _gen(seed)
    h, i, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    r = lambda *s: torch.randn(*s, generator=g, device="cuda") * 0.05  # noqa: E731
    w = {"model.embed_tokens.weight": r(cfg.vocab_size, h) * 20, "model.norm.weight": 1 + r(h)}
    for li in range(cfg.num_layers):
        p = f"model.layers.{li}."
        w[p + "input_layernorm.weight"], w[p + "post_attention_layernorm.weight"] = 1 + r(h), 1 + r(h)
        for nm, heads in (("q", cfg.num_heads), ("k", cfg.num_kv_heads), ("v", cfg.num_kv_heads)):
            w[p + f"self_attn.{nm}_proj.weight"] = r(heads * d, h)
            if cfg.qkv_bias:
                w[p + f"self_attn.{nm}_proj.bias"] = r(heads * d)
        w[p + "self_attn.o_proj.weight"] = r(h, cfg.num_heads * d)
        w[p + "mlp.gate_proj.weight"], w[p + "mlp.up_proj.weight"] = r(i, h), r(i, h)
        w[p + "mlp.down_proj.weight"] = r(h, i)
    if not cfg.tie_word_embeddings:
        w["lm_head.weight"] = r(cfg.vocab_size, h)
    return w


def _prompt(case: dict, cfg: M.ModelConfig, seed: int) -> list[int]:
    return np.random.default_rng(seed).integers(0, cfg.vocab_size, case["t"]).tolist()


# ---------------------------------------------------------------- prepare, run

def _resident(case: dict, packed):
    """The device handle a program makes of packed weights (lb.to_device)."""
    if case["fmt"] == "mxfp4":
        codes, e = packed
        return lb.to_device(lb.MXFP4Weights(_nibbles(codes, 32).cpu().numpy(), e.cpu().numpy(), case["k"]))
    (codes, s, z), group = packed, case.get("group", 128)
    return lb.to_device(lb.Int4Weights(_nibbles(codes, group).cpu().numpy(), s.cpu().numpy(),
                                       None if z is None else z.cpu().numpy(), case["k"], group))


def _prepare_gemm(case: dict, seed: int) -> dict:
    packed, x = _gemm_inputs(case, seed)
    w = _resident(case, packed)
    if case["op"] == "call":
        fn = {"w4a16": lb.gemm_w4a16, "mxfp4": lb.gemm_mxfp4, "w4a8": lb.gemm_w4a8}[case["fmt"]]
        xh = x.cpu().numpy()
        fn(xh, w)  # a warm handle, as in a serving loop
        return {"call": lambda: fn(xh, w)}
    L, fmt, m, n = K.lib(), case["fmt"], case["m"], case["n"]
    x = torch.nn.functional.pad(x, (0, w.kp - case["k"])).contiguous()
    y = torch.empty(m, n, device="cuda")
    prm = K._Params(-1, 0, 0, 0, 0, 0, 0)
    tiles = L.lbd_gemm_path(KINDS[fmt], m, w.kp, C.byref(prm)) == K.ISA_GFX950_MFMA
    need = (L.lbd_w4a8_workspace_bytes(m, w.kp) if fmt == "w4a8"
            else L.lbd_bf16x3_workspace_bytes_split(KINDS[fmt], m, n, w.kp))
    ws = torch.empty(max(256, need), dtype=torch.uint8, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    dx, dy, dw = x.data_ptr(), y.data_ptr(), ws.data_ptr()
    zp = getattr(getattr(w, "zeros", None), "ptr", None)
    if case.get("group") == 32:
        fn = L.lbd_gemm_w4a16_g32 if fmt == "w4a16" else L.lbd_gemm_w4a8_g32
        call = lambda: fn(dx, m, w.kp, w.qw.ptr, w.scales.ptr, zp, n, dy, s)  # noqa: E731
    elif fmt == "w4a16" and tiles:
        (w.tiles_f8 if K.w4a16_uses_t16f8(w, m) else w.tiles)()
        call = lambda: K.gemm_w4a16_tiles(w, dx, m, dy, prm, dw, need, s)  # noqa: E731
    elif fmt == "w4a16":
        call = lambda: L.lbd_gemm_w4a16(dx, m, w.kp, w.qw.ptr, w.scales.ptr, zp, n, dy, C.byref(prm), s)  # noqa: E731
    elif fmt == "mxfp4" and tiles:
        qt, et = w.tiles()
        call = lambda: L.lbd_gemm_mxfp4_t16(dx, m, w.kp, qt.ptr, et.ptr, n, dy, C.byref(prm), dw, need, s)  # noqa: E731
    elif fmt == "mxfp4":
        call = lambda: L.lbd_gemm_mxfp4(dx, m, w.kp, w.qw.ptr, w.e8m0.ptr, n, dy, C.byref(prm), s)  # noqa: E731
    elif tiles:
        qt, st, zt = w.tiles()
        zt = None if zt is None else zt.ptr
        call = lambda: L.lbd_gemm_w4a8_t16(dx, m, w.kp, qt.ptr, st.ptr, zt, n, dy, C.byref(prm),  # noqa: E731
                                           dw, need, s)
    else:
        call = lambda: L.lbd_gemm_w4a8(dx, m, w.kp, w.qw.ptr, w.scales.ptr, zp, n, dy, C.byref(prm),  # noqa: E731
                                       dw, need, s)

    def go():
        K._check(call(), fmt)
        return y
    return {"call": go, "keep": (w, x, ws)}


def _prepare_attention(case: dict, seed: int) -> dict:
    qkv, kc, vc, cos, sin = _attn_inputs(case, seed)
    L, h, kv, d = K.lib(), case["h"], case["kv"], case["d"]
    pos = torch.tensor([case["past"]], dtype=torch.int32, device="cuda")
    out = torch.empty(qkv.shape[0], h * d, device="cuda")
    s, cap, width = torch.cuda.current_stream().cuda_stream, kc.shape[1], qkv.shape[1]
    if case["op"] == "attend":
        def go():
            K._check(L.lbd_attention(qkv.data_ptr(), width, kc.data_ptr(), vc.data_ptr(), case["t"], h, kv, d,
                                     pos.data_ptr(), cap, out.data_ptr(), s), "attention")
            return out
        return {"call": go}
    work = torch.empty(L.lbd_attention_decode_work_bytes(h, d, cap), dtype=torch.uint8, device="cuda")

    def go():
        K._check(L.lbd_attention_decode_ws(qkv.data_ptr(), h, kv, d, cos.data_ptr(), sin.data_ptr(), pos.data_ptr(),
                                           cap, kc.data_ptr(), vc.data_ptr(), cap, out.data_ptr(), work.data_ptr(),
                                           work.numel(), s), "attention step")
        return {"out": out, "k": kc, "v": vc}
    return {"call": go}


def _prepare_pack(case: dict, seed: int) -> dict:
    n, k, group = case["n"], case["k"], case["group"]
    w = torch.randn(n, k, generator=_gen(seed), device="cuda") * 0.02
    L, s, kp = K.lib(), torch.cuda.current_stream().cuda_stream, -(-k // group) * group
    u8 = lambda *shape: torch.empty(*shape, dtype=torch.uint8, device="cuda")  # noqa: E731
    qw, per = u8(n, kp // 2), kp // group
    if case["fmt"] == "mxfp4":
        e = u8(n, per)

        def go():
            K._check(L.lbd_quantize_mxfp4(w.data_ptr(), n, k, qw.data_ptr(), e.data_ptr(), s), "pack")
            return {"qw": qw, "e8m0": e}
        return {"call": go}
    scales, zeros = torch.empty(n, per, device="cuda"), u8(n, per) if case["asym"] else None
    fn = L.lbd_quantize_int4 if group == 128 else L.lbd_quantize_int4_g32

    def go():
        K._check(fn(w.data_ptr(), n, k, int(case["asym"]), 0, qw.data_ptr(), scales.data_ptr(),
                    None if zeros is None else zeros.data_ptr(), s), "pack")
        return {"qw": qw, "scales": scales, "zeros": zeros}
    return {"call": go}


def _prepare_answer(case: dict, seed: int) -> dict:
    cfg = _config(case)
    weights = {k: v.cpu().numpy() for k, v in _model_weights(cfg, seed).items()}
    model = M.Model(cfg, weights, case["fmt"], max_tokens=case["t"])
    prompt, cache = _prompt(case, cfg, seed), model.new_cache(case["t"] + case["new"] + 1)
    model.forward(prompt, cache)  # the prompt kernels' weight layouts exist once a model has answered

    def go():
        cache.length = 0
        tokens = model.generate(prompt, case["new"], cache)
        return {"tokens": np.array(tokens, np.int64), "logits": model.forward(tokens[-1:], cache)}
    return {"call": go}


def prepare(case: dict, seed: int) -> dict:
    make = {"call": _prepare_gemm, "gemm": _prepare_gemm, "attend": _prepare_attention, "step": _prepare_attention,
            "pack": _prepare_pack, "answer": _prepare_answer}[case["op"]]
    return make(case, seed)


def run(state: dict):
    return state["call"]()


# ---------------------------------------------------------------- work, tolerance

def _weight_bytes(fmt: str, asym: bool, n: int, k: int, group: int = 128) -> float:
    return n * k / 2 + (n * k / 32 if fmt == "mxfp4" else n * k / group * (5 if asym else 4))


def work(case: dict) -> dict:
    op = case["op"]
    if op in ("call", "gemm"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _weight_bytes(case["fmt"], case["asym"], n, k, case.get("group", 128)) + 4 * m * (n + k),
                "flops": 2 * m * n * k}
    if op in ("attend", "step"):
        t, h, kv, d, past = case.get("t", 1), case["h"], case["kv"], case["d"], case["past"]
        pairs = t * past + t * (t + 1) / 2
        return {"bytes": 4 * (2 * t * h * d + 2 * kv * (past + t) * d), "flops": 4 * pairs * h * d}
    if op == "pack":
        fmt, n, k = case["fmt"], case["n"], case["k"]
        per = 1 if fmt == "mxfp4" else 5 if case["asym"] else 4
        return {"bytes": n * k * 4.5 + n * k / case["group"] * per, "flops": 4 * n * k}
    cfg, t, new = _config(case), case["t"], case["new"]
    h, d = cfg.hidden_size, cfg.head_dim
    widths = [((cfg.num_heads + 2 * cfg.num_kv_heads) * d, h), (h, cfg.num_heads * d),
              (2 * cfg.intermediate_size, h), (h, cfg.intermediate_size)]
    layer, head = sum(n * k for n, k in widths), cfg.vocab_size * h
    per = _weight_bytes(case["fmt"], False, 1, 1)
    attn = 4 * cfg.num_heads * d * cfg.num_layers * (t * t / 2 + new * t)
    return {"bytes": per * (cfg.num_layers * layer + head) * (new + 1),
            "flops": 2 * cfg.num_layers * layer * (t + new) + 2 * head * (new + 1) + attn}


def tolerance(case: dict):
    if case["op"] == "pack":
        return "exact"
    # against 64 bits: GEMMs 0.7-1.8e-7, attention 2-6e-7, the decoder's logits 0.4-3e-4
    # (four layers carry each one's rounding on)
    if case["op"] == "answer":
        return {"rel": 1.5e-3, "differ": 0.0}
    return {"rel": 4e-6 if case["op"] in ("attend", "step") else 2e-6}


# ---------------------------------------------------------------- the results in 64 bits

def _rows_int8(x: torch.Tensor) -> torch.Tensor:
    """The per-token int8 quantization that W4A8 is defined with, as float64 values."""
    amax = x.abs().amax(1, keepdim=True)
    s = torch.where(amax > 0, amax / 127, torch.ones_like(amax))
    return torch.round(x / s).clamp(-127, 127).double() * s.double()


def _softmax_av(q, k, v, past: int):
    """q [H, T, D], k / v [KV, S, D] in float64, causal behind `past` -> [T, H D]."""
    h, t, d = q.shape
    rep = h // k.shape[0]
    out = []
    for i in range(h):
        sc = q[i] @ k[i // rep].t() / d ** 0.5
        at = torch.arange(k.shape[1], device=q.device)[None] > past + torch.arange(t, device=q.device)[:, None]
        out.append(torch.softmax(sc.masked_fill(at, float("-inf")), 1) @ v[i // rep])
    return torch.stack(out, 1).reshape(t, h * d)


def _rotate(x, cos, sin):
    """x [..., D] rotated by angles [..., D/2], halves paired."""
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _exact_answer(case: dict, seed: int) -> dict:
    cfg = _config(case)
    w = _model_weights(cfg, seed)
    h, kv, d = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim
    fmt = case["fmt"]
    lin = lambda t: _dense(fmt, _mxfp4(t) if fmt == "mxfp4" else _int4(t, False))  # noqa: E731
    mats = {k: lin(v) for k, v in w.items() if "_proj.weight" in k}
    head = lin(w["model.embed_tokens.weight" if cfg.tie_word_embeddings else "lm_head.weight"])
    cos, sin = (torch.from_numpy(t).cuda().double() for t in M.rope_tables(d, cfg.max_position, cfg.rope_theta))
    norm = lambda x, n: x / torch.sqrt((x * x).mean(1, keepdim=True) + cfg.rms_norm_eps) * w[n].double()  # noqa: E731
    none = torch.empty(kv, 0, d, device="cuda", dtype=torch.float64)
    keys = [[none, none] for _ in range(cfg.num_layers)]

    def forward(tokens: list[int], past: int):
        x = w["model.embed_tokens.weight"][torch.tensor(tokens, device="cuda")].double()
        t = len(tokens)
        for li in range(cfg.num_layers):
            p = f"model.layers.{li}."
            y = norm(x, p + "input_layernorm.weight")
            q, k, v = (y @ mats[p + f"self_attn.{nm}_proj.weight"].t() + w.get(p + f"self_attn.{nm}_proj.bias", 0)
                       for nm in "qkv")
            q, k, v = (a.double().reshape(t, -1, d).transpose(0, 1) for a in (q, k, v))
            q, k = (_rotate(a, cos[past:past + t], sin[past:past + t]) for a in (q, k))
            keys[li] = [torch.cat([old, new], 1) for old, new in zip(keys[li], (k, v))]
            x = x + _softmax_av(q, *keys[li], past) @ mats[p + "self_attn.o_proj.weight"].t()
            y = norm(x, p + "post_attention_layernorm.weight")
            g, u = y @ mats[p + "mlp.gate_proj.weight"].t(), y @ mats[p + "mlp.up_proj.weight"].t()
            x = x + (g * torch.sigmoid(g) * u) @ mats[p + "mlp.down_proj.weight"].t()
        return (norm(x, "model.norm.weight")[-1:] @ head.t())[0]

    logits = forward(_prompt(case, cfg, seed), 0)
    tokens = [int(logits.argmax())]
    for i in range(case["new"]):
        logits = forward(tokens[-1:], case["t"] + i)
        if i + 1 < case["new"]:
            tokens.append(int(logits.argmax()))
    return {"tokens": None, "logits": logits}


def exact(case: dict, seed: int):
    op = case["op"]
    if op in ("call", "gemm"):
        packed, x = _gemm_inputs(case, seed)
        w = _dense(case["fmt"], packed, case.get("group", 128))[:, : case["k"]]
        y = (_rows_int8(x) if case["fmt"] == "w4a8" else x.double()) @ w.t()
        return y.cpu().numpy() if op == "call" else y
    if op in ("attend", "step"):
        qkv, kc, vc, cos, sin = _attn_inputs(case, seed)
        h, kv, d, past = case["h"], case["kv"], case["d"], case["past"]
        rows = qkv.double().reshape(qkv.shape[0], -1, d).transpose(0, 1)
        q, k, v = rows[:h], rows[h:h + kv], rows[h + kv:]
        kc, vc = kc.double(), vc.double()
        if op == "attend":
            return _softmax_av(q, kc, vc, past)
        q, k = (_rotate(a, cos[past].double(), sin[past].double()) for a in (q, k))
        kc[:, past], vc[:, past] = k[:, 0], v[:, 0]
        return {"out": _softmax_av(q, kc[:, : past + 1], vc[:, : past + 1], past), "k": kc, "v": vc}
    if op == "pack":
        if case["fmt"] == "mxfp4":
            return None
        w = torch.randn(case["n"], case["k"], generator=_gen(seed), device="cuda") * 0.02
        b = _pad(w.double(), case["group"]).reshape(case["n"], -1, case["group"])
        s = (b.amax(2).clamp(min=0) - b.amin(2).clamp(max=0)) / 15 if case["asym"] else b.abs().amax(2) / 7
        return {"qw": None, "scales": torch.where(s > 0, s, torch.ones_like(s)), "zeros": None}
    return _exact_answer(case, seed)
