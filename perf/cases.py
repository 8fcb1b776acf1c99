"""The calls this framework is measured on: decode and prefill work of a
quantized transformer, through the public Python entry points (tenzo_amd.ops
and tenzo_amd.engine).

Sizes are those of the repository's own configurations (the BitNet-2B shape:
hidden 2560, FFN 6912, 20 query / 5 kv heads of 128; GEMVs of 11008 x 4096 and
14336 x 4096) and ragged relatives of them. Each case is a dict of plain values
whose "kind" picks one path:

  proj      RMSNorm + activation quantizer + TL1 product of M token rows: the
            decode GEMV for one row, the int8 contraction for a prompt's rows
  bitlinear executeBitLinearTL1 on fp32 rows (quantizer and product in one call)
  attn      one decode step of INT8-KV attention for B sequences
  tern      the same step over a ternary cache (tl1_fused or popcount_fused)
  paged     the same step over a paged INT8 cache
  q4_0, q8_0, gptq, awq   weight-quantized products of B activation rows
  prefill   a prompt through the engine, then the first decode step's logits
  decode    one greedy decode step of the 30-layer model, with its logits
"""
import ctypes
import math

import numpy as np
import torch

from tenzo_amd import engine, ops, synth

D = 128
THETA = 500000.0
EPS = 1e-5

# rms of an embedding row. In a trained model a layer changes the residual stream by a few
# percent; with random weights and a small embedding every layer would replace it, and the
# flip of one rounded code, which any change of a sum's order brings, would grow with depth.
EMBED_RMS = 64.0
AWQ_ORDER = [0, 2, 4, 6, 1, 3, 5, 7]  # the element of a word's nibble e


def listed():
    return [
        # a decode step's Q|K|V projection through the operators: two launches
        # on a few MB, the smallest call a program makes
        {"name": "proj_m1", "kind": "proj", "M": 1, "N": 3840, "K": 2560},
        # executeBitLinearTL1 on the rows of a small batch (the FFN's down matrix)
        {"name": "bitlinear_m24", "kind": "bitlinear", "M": 24, "N": 2560, "K": 6912},
        # the gate|up product of a prompt pass, a ragged number of tokens
        {"name": "proj_m500", "kind": "proj", "M": 500, "N": 13824, "K": 2560},
        # chat at the start of a conversation: one sequence, a short context
        {"name": "attn_b1_1k", "kind": "attn", "B": 1, "Hq": 20, "Hkv": 5, "ctx": 1000},
        # batched serving over long contexts
        {"name": "attn_b16_30k", "kind": "attn", "B": 16, "Hq": 20, "Hkv": 5, "ctx": 30011},
        # the compressed cache, a few sequences
        {"name": "tern_b4_6k", "kind": "tern", "mode": "tl1_fused", "B": 4, "Hq": 20, "Hkv": 5,
         "ctx": 6001},
        # the paged cache, one sequence of some length
        {"name": "paged_8k", "kind": "paged", "Hq": 20, "Hkv": 5, "ctx": 8100},
        # a GGUF Q4_0 layer in batch-1 decode
        {"name": "q4_0_b1", "kind": "q4_0", "B": 1, "N": 11008, "K": 4096, "half": True},
        # a GGUF Q8_0 layer for a few sequences, fp32 activations as the reference has them
        {"name": "q8_0_b6", "kind": "q8_0", "B": 6, "N": 11008, "K": 4096, "half": False},
        # a GPTQ layer for a batch of eight
        {"name": "gptq_b8", "kind": "gptq", "B": 8, "N": 14336, "K": 4096, "group": 128,
         "half": True},
        # a prompt of ordinary length (a few layers of the model: every layer is alike)
        {"name": "prefill_1500", "kind": "prefill", "n": 1500, "layers": 4},
        # the whole model, one token at a context of 4096
        {"name": "decode_4k", "kind": "decode", "ctx": 4096, "layers": 30},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["proj", "bitlinear", "attn", "tern", "paged", "q4_0", "q8_0", "gptq",
                       "awq", "prefill", "decode"])
    heads = rng.choice([(20, 5), (16, 4), (8, 8), (16, 2)])
    if kind in ("proj", "bitlinear"):
        M = _log(rng, 1, 1100 if kind == "proj" else 300)
        K = rng.choice([64 * rng.randint(10, 108), 2 * _log(rng, 320, 3456)])
        return {"kind": kind, "M": M, "N": 64 * rng.randint(20, 216), "K": K}
    if kind == "attn":
        B, ctx = _log(rng, 1, 16), _log(rng, 60, 30000)
        return {"kind": kind, "B": B, "Hq": heads[0], "Hkv": heads[1],
                "ctx": min(ctx, 16 * 5 * 30000 // (B * heads[1]))}
    if kind == "tern":
        return {"kind": kind, "mode": rng.choice(["tl1_fused", "popcount_fused"]),
                "B": _log(rng, 1, 16), "Hq": heads[0], "Hkv": heads[1], "ctx": _log(rng, 60, 16000)}
    if kind == "paged":
        return {"kind": kind, "Hq": heads[0], "Hkv": heads[1], "ctx": _log(rng, 60, 30000)}
    if kind in ("q4_0", "q8_0"):
        return {"kind": kind, "B": _log(rng, 1, 16), "N": _log(rng, 1000, 14336),
                "K": 32 * rng.choice([64, 80, 100, 128, 160, 216, 344]),
                "half": rng.choice([True, False])}
    if kind in ("gptq", "awq"):
        return {"kind": kind, "B": _log(rng, 1, 8), "N": 8 * _log(rng, 128, 1400),
                "K": 512 * rng.randint(4, 28), "group": rng.choice([32, 64, 128]),
                "half": rng.choice([True, True, False])}
    if kind == "prefill":
        return {"kind": kind, "n": _log(rng, 20, 1500), "layers": 4}
    return {"kind": "decode", "ctx": _log(rng, 100, 8000), "layers": 30}


# ------------------------------------------------------------------ inputs ----

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _tl1_bytes(w):
    """Ternary [N][K] -> the TL1 blocks [N/64][K/2][32] the weight files hold."""
    N, K = w.shape
    u = (w + 1).to(torch.uint8).reshape(N // 64, 2, 32, K // 2, 2)
    nib = u[..., 0] | (u[..., 1] << 2)
    return (nib[:, 0] | (nib[:, 1] << 4)).transpose(1, 2).contiguous().reshape(-1)


def _ternary(g, N, K):
    return torch.randint(-1, 2, (N, K), dtype=torch.int8, device="cuda", generator=g)


def _rows(g, M, K):
    """Activation rows: N(0, 1) with a few large channels, as hidden states have."""
    x = _randn(g, M, K)
    x[:, torch.randint(0, K, (4,), device="cuda", generator=g)] *= 6.0
    return x


def _away(x):
    return torch.sign(x) * torch.floor(x.abs() + 0.5)  # halves away from zero


def _kv_codes(x):
    amax = x.abs().amax(-1).clamp_min(1e-8)
    c = torch.clamp(_away(x * (127.0 / amax)[..., None]), -128, 127).to(torch.int8)
    return c, amax / 127.0


def _angles(pos):
    f = THETA ** (-np.arange(0, D, 2, dtype=np.float64) / D)
    a = (np.float32(pos) * f.astype(np.float32)).astype(np.float32)
    return torch.from_numpy(np.concatenate([np.cos(a), np.sin(a)]).astype(np.float32)).cuda()


def _qkv(g, case, B):
    return (_randn(g, B, case["Hq"] * D), _randn(g, B, case["Hkv"] * D),
            _randn(g, B, case["Hkv"] * D), _angles(case["ctx"]))


def _int8_cache(g, shape):
    """Codes and scales of cached N(0, 1) rows, made a piece at a time."""
    n = math.prod(shape)
    codes = torch.empty((n, D), dtype=torch.int8, device="cuda")
    scales = torch.empty(n, device="cuda")
    for i in range(0, n, 1 << 18):
        c, s = _kv_codes(_randn(g, min(1 << 18, n - i), D))
        codes[i:i + c.shape[0]] = c
        scales[i:i + c.shape[0]] = s
    return codes.reshape(*shape, D), scales.reshape(shape)


def _room(ctx):
    return (ctx + 1 + 63) // 64 * 64  # cache rows of a program that has space for the new token


def _pack_fields(w):
    f = (w + 1).to(torch.uint8).reshape(*w.shape[:-1], 32, 4)
    return f[..., 0] | (f[..., 1] << 2) | (f[..., 2] << 4) | (f[..., 3] << 6)


def _pack_planes(w):
    bit = (2 ** torch.arange(8, device="cuda")).to(torch.int32)

    def plane(m):
        return (m.to(torch.int32).reshape(*m.shape[:-1], 16, 8) * bit).sum(-1).to(torch.uint8)

    return torch.cat([plane(w > 0), plane(w < 0)], -1)


def _inputs(case, seed):
    """The case's inputs as plain tensors (and what the weights stand for)."""
    g = _gen(seed)
    k = case["kind"]
    if k in ("proj", "bitlinear"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"x": _rows(g, M, K), "w": _ternary(g, N, K), "norm": 1.0 + 0.1 * _randn(g, K),
                "scale": 0.0159}
    if k == "attn":
        B, Hkv = case["B"], case["Hkv"]
        q, kn, vn, cs = _qkv(g, case, B)
        S = _room(case["ctx"])
        kc, ks = _int8_cache(g, (B, Hkv, S))
        vc, vs = _int8_cache(g, (B, Hkv, S))
        return {"q": q, "k": kn, "v": vn, "cs": cs, "kc": kc, "vc": vc, "ks": ks.half(),
                "vs": vs.half()}
    if k == "tern":
        B, Hkv = case["B"], case["Hkv"]
        q, kn, vn, cs = _qkv(g, case, B)
        S = _room(case["ctx"])
        out = {"q": q, "k": kn, "v": vn, "cs": cs}
        for name in ("k", "v"):
            u = torch.rand((B, Hkv, S, D), device="cuda", generator=g)
            w = ((u > 0.345).to(torch.int8) + (u > 0.655).to(torch.int8) - 1)
            planes = name == "k" and case["mode"] == "popcount_fused"
            out[name + "w"] = w
            out[name + "b"] = (_pack_planes(w) if planes else _pack_fields(w)).contiguous()
            out[name + "s"] = 0.9 + 0.6 * torch.rand((B, Hkv, S), device="cuda", generator=g)
        return out
    if k == "paged":
        q, kn, vn, cs = _qkv(g, case, 1)
        nb = case["ctx"] // 16 + 1
        pk, pks = _int8_cache(g, (nb + 3, 2, case["Hkv"], 16))
        pv, pvs = _int8_cache(g, (nb + 3, 2, case["Hkv"], 16))
        table = torch.randperm(nb + 3, device="cuda", generator=g)[:nb].to(torch.int32)
        return {"q": q, "k": kn, "v": vn, "cs": cs, "pk": pk, "pv": pv, "pks": pks, "pvs": pvs,
                "table": table.contiguous()}
    B, N, K = case["B"], case["N"], case["K"]
    act = _rows(g, B, K)
    act = act.half() if case["half"] else act
    if k in ("q4_0", "q8_0"):
        d = (0.002 + 0.004 * torch.rand((N, K // 32, 1), device="cuda", generator=g)).half()
        if k == "q4_0":
            c = torch.randint(0, 16, (N, K // 32, 32), dtype=torch.uint8, device="cuda", generator=g)
            body = c[..., :16] | (c[..., 16:] << 4)
        else:
            c = torch.randint(-127, 128, (N, K // 32, 32), dtype=torch.int8, device="cuda",
                              generator=g)
            body = c.view(torch.uint8)
        return {"act": act, "c": c, "d": d, "w": torch.cat([d.view(torch.uint8), body], -1).reshape(-1)}
    G = K // case["group"]
    c = torch.randint(0, 16, (K, N), dtype=torch.uint8, device="cuda", generator=g)
    z = torch.randint(0, 16, (G, N), dtype=torch.uint8, device="cuda", generator=g)
    s = (0.002 + 0.004 * torch.rand((G, N), device="cuda", generator=g)).half()
    sh = (4 * torch.arange(8, device="cuda")).to(torch.int64)
    order = AWQ_ORDER if k == "awq" else list(range(8))
    words = (c.reshape(K // 8, 8, N)[:, order].to(torch.int64) << sh[None, :, None]).sum(1)
    if k == "gptq":
        zp = torch.zeros(((G + 7) // 8 * 8, N), dtype=torch.int64, device="cuda")
        zp[:G] = z
        zw = (zp.reshape(-1, 8, N) << sh[None, :, None]).sum(1)
    else:
        zw = (z.reshape(G, N // 8, 8).to(torch.int64) << sh).sum(-1)
    return {"act": act, "c": c, "z": z, "s": s, "qw": words.to(torch.int32).contiguous(),
            "zw": zw.to(torch.int32).contiguous()}


def _config(case):
    if case["kind"] == "prefill":
        return synth.DecodeConfig(n_layers=case["layers"], vocab=32000,
                                  max_seq=(case["n"] + 64) // 64 * 64)
    return synth.DecodeConfig(n_layers=case["layers"], max_seq=(case["ctx"] + 64) // 64 * 64)


def _engine(case, seed):
    """An engine of the BitNet-2B layer shape with random weights."""
    cfg = _config(case)
    g = _gen(seed)
    rng = np.random.default_rng(seed)
    e = engine.Engine(cfg)
    names = dict(zip(synth.PROJ, ["q", "k", "v", "out", "gate", "up", "down"]))
    for l in range(cfg.n_layers):
        w = engine.LayerWeights()
        hold = []
        for p, field in names.items():
            n, k = cfg.proj_shape(p)
            pair = torch.randint(0, 81, (n * k // 4,), dtype=torch.uint8, device="cuda", generator=g)
            a, b = pair // 9, pair % 9  # two pairs of ternary weights to a byte
            hold.append((a % 3) | ((a // 3) << 2) | ((b % 3) << 4) | ((b // 3) << 6))
            setattr(w, field + "_w", hold[-1].data_ptr())
            setattr(w, field + "_scale", 0.0159)
        for f in ("in_norm", "attn_sub_norm", "post_norm", "ffn_sub_norm"):
            n = cfg.ffn if f == "ffn_sub_norm" else cfg.hidden
            hold.append((1.0 + 0.1 * rng.standard_normal(n)).astype(np.float32))
            setattr(w, f, hold[-1].ctypes.data)
        torch.cuda.synchronize()
        e._check(e.L.tenzo_set_layer_weights(e.h, l, ctypes.byref(w)), "set_layer_weights")
    norm = (1.0 + 0.1 * rng.standard_normal(cfg.hidden)).astype(np.float32)
    e._check(e.L.tenzo_set_final_norm(e.h, norm.ctypes.data), "set_final_norm")
    head = torch.empty((cfg.vocab, cfg.hidden), dtype=torch.int8, device="cuda")
    scales = torch.empty(cfg.vocab, device="cuda")
    for r in range(0, cfg.vocab, 16384):
        c, s = _kv_codes(_randn(g, min(16384, cfg.vocab - r), cfg.hidden))
        head[r:r + c.shape[0]] = c
        scales[r:r + c.shape[0]] = EMBED_RMS * s
    torch.cuda.synchronize()
    e._check(e.L.tenzo_set_lm_head_i8(e.h, head.data_ptr(), scales.data_ptr(), cfg.vocab,
                                      cfg.hidden), "set_lm_head_i8")
    if case["kind"] == "decode":
        shape = (cfg.n_layers, cfg.n_kv_heads, case["ctx"])
        kc, ks = _int8_cache(g, shape)
        vc, vs = _int8_cache(g, shape)
        ks, vs = ks.half(), vs.half()
        torch.cuda.synchronize()
        e.set_kv_device(kc.data_ptr(), vc.data_ptr(), ks.data_ptr(), vs.data_ptr(), case["ctx"])
    e.set_rope_theta(THETA)
    return {"engine": e, "tokens": rng.integers(0, cfg.vocab, size=4096).astype(np.int32)}


def prepare(case, seed):
    k = case["kind"]
    if k in ("prefill", "decode"):
        return dict(_engine(case, seed), case=case)
    s = _inputs(case, seed)
    if k in ("proj", "bitlinear"):
        s["packed"] = ops.tl1_repack(_tl1_bytes(s.pop("w")), case["N"], case["K"])
    for spare in ("c", "d", "z", "kw", "vw"):
        s.pop(spare, None)
    return dict(s, case=case)


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "proj":
        codes, q, _ = ops.rmsnorm_quant31(s["x"], s["norm"], EPS)
        # the GEMV for the rows of a decode step, the contraction for a prompt's
        product = ops.bitlinear_tl1 if case["M"] == 1 else ops.bitlinear_tl1_batch
        y, _ = product(codes, q, s["packed"], s["scale"], case["N"], case["K"])
        return {"y": y, "codes": codes}
    if k == "bitlinear":
        return ops.bitlinear_tl1_f32(s["x"], s["packed"], s["scale"], case["N"], case["K"])
    if k == "attn":
        out = ops.attn_int8_decode(s["q"], s["k"], s["v"], s["kc"], s["vc"], s["ks"], s["vs"],
                                   s["cs"], case["ctx"])
        return {"out": out, "kc": s["kc"], "vc": s["vc"], "ks": s["ks"], "vs": s["vs"]}
    if k == "tern":
        out = ops.attn_tern_decode(case["mode"], s["q"], s["k"], s["v"], s["kb"], s["vb"], s["ks"],
                                   s["vs"], s["cs"], case["ctx"])
        return {"out": out, "kb": s["kb"], "vb": s["vb"], "ks": s["ks"], "vs": s["vs"]}
    if k == "paged":
        out = ops.attn_paged_int8_decode(s["q"], s["k"], s["v"], s["pk"], s["pv"], s["pks"],
                                         s["pvs"], s["table"], 1, s["cs"], case["ctx"])
        return {"out": out, "pk": s["pk"], "pv": s["pv"], "pks": s["pks"], "pvs": s["pvs"]}
    if k in ("q4_0", "q8_0"):
        return getattr(ops, "gemv_" + k)(s["act"], s["w"], case["K"], case["N"])
    if k in ("gptq", "awq"):
        return getattr(ops, "gemv_" + k)(s["act"], s["qw"], s["s"], s["zw"], case["K"], case["N"],
                                         case["group"])
    e, t = s["engine"], s["tokens"]
    if k == "prefill":
        e.reset()
        e.prefill_batch(t[:case["n"] - 1])
        e.step(int(t[case["n"] - 1]))
    else:
        e.rewind(case["ctx"])
        e.step(int(t[0]))
    return {"x": e.buffer("x"), "logits": e.logits()}


# -------------------------------------------------------------------- work ----

def work(case):
    k = case["kind"]
    if k in ("proj", "bitlinear"):
        M, N, K = case["M"], case["N"], case["K"]
        codes = 2 * M * K if k == "proj" else 0  # the codes are an output, and read
        return {"bytes": N * K // 4 + 4 * M * K + codes + 4 * M * N, "flops": 2 * M * N * K}
    if k in ("attn", "tern", "paged"):
        B, Hq, Hkv, n = case.get("B", 1), case["Hq"], case["Hkv"], case["ctx"] + 1
        row = {"attn": 2 * (D + 2), "tern": 2 * (D // 4 + 4), "paged": 2 * (D + 4)}[k]
        return {"bytes": B * (Hkv * n * row + 4 * D * (2 * Hq + 2 * Hkv)),
                "flops": 4 * B * Hq * n * D}
    if k in ("q4_0", "q8_0", "gptq", "awq"):
        B, N, K = case["B"], case["N"], case["K"]
        if k in ("q4_0", "q8_0"):
            w = N * K // 32 * (18 if k == "q4_0" else 34)
        else:
            w = N * K // 2 + K // case["group"] * N * 5 // 2
        return {"bytes": w + B * K * (2 if case["half"] else 4) + 4 * B * N, "flops": 2 * B * N * K}
    cfg = _config(case)
    params = sum(n * kk for n, kk in (cfg.proj_shape(p) for p in synth.PROJ)) * cfg.n_layers
    if k == "decode":
        b = cfg.step_bytes(case["ctx"] + 1)["total"]
        return {"bytes": b + 4 * cfg.vocab, "flops": 2 * (params + cfg.vocab * cfg.hidden)}
    n = case["n"]
    attn = cfg.n_layers * cfg.n_q_heads * 4 * D * n * n // 2
    return {"bytes": cfg.step_bytes(n)["total"] + 4 * cfg.vocab,
            "flops": 2 * n * params + attn + 2 * cfg.vocab * cfg.hidden}


def tolerance(case):
    k = case["kind"]
    if k in ("proj", "bitlinear"):
        # whole-number sums and one product: every implementation gives the same bits
        return "exact"
    # A whole model: four times what its two orders of the attention's sums differ by
    # (prefill: exact against streaming, up to 0.0063 in the logits; decode: the
    # persistent kernel against the stage kernels, 1e-7, and up to 0.014 where a code flips).
    if k == "prefill":
        return {"rel": 0.025}
    if k == "decode":
        return {"rel": 0.03}
    # fp32 sums in another order
    return {"rel": 1e-5, "max": 2e-4, "differ": 0.0}


# ------------------------------------------------------------------- exact ----

def _rope64(x, cs):
    c, s = cs.double()[:64], cs.double()[64:]
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _attend(q, kf, vf):
    """softmax(q k / sqrt(D)) v of one kv head's query rows in float64."""
    return torch.softmax(q @ kf.T / math.sqrt(D), -1) @ vf


def _tern_row(x):
    """A row's ternary codes and scale: threshold at half the mean magnitude."""
    a = x.abs()
    m = a > 0.5 * a.mean(-1, keepdim=True)
    return torch.sign(x) * m, (a * m).sum(-1) / m.sum(-1)


def exact(case, seed):
    k = case["kind"]
    if k in ("prefill", "decode"):
        return None  # a whole model: its rounded codes have no 64-bit value
    s = _inputs(case, seed)
    if k in ("proj", "bitlinear"):
        x = s["x"].double()
        if k == "proj":
            x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * s["norm"].double()
        amax = x.abs().amax(-1, keepdim=True).clamp_min(1e-6)
        codes = _away(x * (31.0 / amax))
        y = (codes @ s["w"].double().T) * (amax / 31.0) * s["scale"]
        return {"y": y, "codes": None} if k == "proj" else y
    if k in ("attn", "tern", "paged"):
        Hq, Hkv, n = case["Hq"], case["Hkv"], case["ctx"]
        G = Hq // Hkv
        B = case.get("B", 1)
        q = _rope64(s["q"].double().reshape(B, Hkv, G, D), s["cs"])
        kn = _rope64(s["k"].double().reshape(B, Hkv, D), s["cs"])
        vn = s["v"].double().reshape(B, Hkv, D)
        out = torch.empty((B, Hkv, G, D), dtype=torch.float64, device="cuda")
        for b in range(B):
            for h in range(Hkv):
                qh = q[b, h]
                if k == "tern":
                    kf = s["kw"][b, h, :n].double() * s["ks"][b, h, :n, None].double()
                    vf = s["vw"][b, h, :n].double() * s["vs"][b, h, :n, None].double()
                    (kt, kts), (vt, vts) = _tern_row(kn[b, h]), _tern_row(vn[b, h])
                    knew, vnew = kt * kts, vt * vts
                    if case["mode"] == "tl1_fused":
                        mx = qh.abs().amax(-1, keepdim=True)
                        qh = _away(qh * (127.0 / mx)) * (mx / 127.0)
                    else:
                        qt, qts = _tern_row(qh)
                        qh = qt * qts[:, None]
                else:
                    (kt, kts), (vt, vts) = _kv_codes(kn[b, h]), _kv_codes(vn[b, h])
                    if k == "attn":
                        kts, vts = kts.half().double(), vts.half().double()
                        kf = s["kc"][b, h, :n].double() * s["ks"][b, h, :n, None].double()
                        vf = s["vc"][b, h, :n].double() * s["vs"][b, h, :n, None].double()
                    else:
                        t = s["table"].long()
                        kf = (s["pk"][t, 1, h].reshape(-1, D)[:n].double()
                              * s["pks"][t, 1, h].reshape(-1, 1)[:n].double())
                        vf = (s["pv"][t, 1, h].reshape(-1, D)[:n].double()
                              * s["pvs"][t, 1, h].reshape(-1, 1)[:n].double())
                    knew, vnew = kt.double() * kts, vt.double() * vts
                out[b, h] = _attend(qh, torch.cat([kf, knew[None]]), torch.cat([vf, vnew[None]]))
        rest = ("pk", "pv", "pks", "pvs") if k == "paged" else (
            ("kb", "vb") if k == "tern" else ("kc", "vc")) + ("ks", "vs")
        return dict({"out": out.reshape(B, Hq * D)}, **{name: None for name in rest})
    act = s["act"].double()
    if k in ("q4_0", "q8_0"):
        w = (s["c"].double() - (8 if k == "q4_0" else 0)) * s["d"].double()
        return act @ w.reshape(case["N"], case["K"]).T
    g = case["group"]
    z = s["z"].double() + (1 if k == "gptq" else 0)
    w = (s["c"].double().reshape(-1, g, case["N"]) - z[:, None]) * s["s"].double()[:, None]
    return act @ w.reshape(case["K"], case["N"])
