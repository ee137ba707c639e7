"""Performance cases: what users of this framework run, through its public entry points.

A case is a plain dict with a "kind":

  matvec     QMat.matvec_dev: one activation row through a quantized projection (a decode step).
  matmul     QMat.matmul_dev: 2 .. 4096 activation rows, bf16 or f32 mode (batched decode, prefill).
  dense      the same two entry points on unquantized F32 / F16 / BF16 weights.
  i8         quantize_q8_act_dev + QMat.matmul_i8_dev: the int8-activation path over Q8_0 weights.
  attention  attention_dev: causal GQA attention of `rows` queries over a K/V cache of earlier rows.
  moe        MoeExperts.layer_dev: router, top-k and the expert FFN of one MoE layer.
  model      DeviceDecoder: prefill of a prompt (and greedy decode of `new` tokens) on a whole model.

Inputs are made from the seed on the GPU: GGUF blocks with uniform quants and scales that give
weights of about zero mean and standard deviation 1/sqrt(K), activations N(0, 1). torch is imported
(and initialises the device) before the library is loaded, so both share one HIP runtime.
"""
import math
import os
import sys

import numpy as np
import torch

torch.cuda.is_available()
sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rusty-engine_amd"))

import rehip  # noqa: E402
from rehip import qwen  # noqa: E402

TYPES = {"Q4_0": rehip.Q4_0, "Q5_0": rehip.Q5_0, "Q8_0": rehip.Q8_0, "Q4_K": rehip.Q4_K, "Q5_K": rehip.Q5_K,
         "Q6_K": rehip.Q6_K}
DENSE = {"F32": (rehip.F32, torch.float32), "F16": (rehip.F16, torch.float16), "BF16": (rehip.BF16, torch.bfloat16)}
MODES = {"bf16": rehip.MODE_BF16, "f32": rehip.MODE_F32}
# root mean square of a block's values at scale 1 (d = 1; dmin = 7.5 d / 15.5 d centres the K-quants)
UNIT = {"Q4_0": 4.64, "Q5_0": 9.25, "Q8_0": 73.9, "Q4_K": 257.2, "Q5_K": 526.9, "Q6_K": 682.4}


def listed():
    return [
        # smallest call: the q / o projection of a small model in a decode step, bound by the launch
        {"name": "matvec_q4k_896", "kind": "matvec", "type": "Q4_K", "m": 896, "n": 896},
        # a batch of 8 sequences decoding together: the down projection on few rows
        {"name": "matmul_q6k_8rows", "kind": "matmul", "type": "Q6_K", "m": 896, "n": 4864, "rows": 8, "mode": "bf16"},
        # prefill of a 961-token prompt, gate / up projection, bf16 mode (ragged row count)
        {"name": "matmul_q5_0_961_bf16", "kind": "matmul", "type": "Q5_0", "m": 4864, "n": 896, "rows": 961,
         "mode": "bf16"},
        # the same prompt's down projection in the f32-accurate mode
        {"name": "matmul_q6k_961_f32", "kind": "matmul", "type": "Q6_K", "m": 896, "n": 4864, "rows": 961,
         "mode": "f32"},
        # largest product: an FFN projection of a large model over a 2048-row prefill chunk
        {"name": "matmul_q4k_large", "kind": "matmul", "type": "Q4_K", "m": 14336, "n": 4096, "rows": 2048,
         "mode": "bf16"},
        # an unquantized (F16) model's projection over the same 961-token prompt, f32 mode
        {"name": "dense_f16_961_f32", "kind": "dense", "type": "F16", "m": 4864, "n": 896, "rows": 961, "mode": "f32"},
        # the int8-activation path over a prompt
        {"name": "i8_q8_0_961", "kind": "i8", "m": 4864, "n": 896, "rows": 961},
        # attention of a prompt chunk over an earlier context, 32 query / 4 KV heads of 128
        {"name": "attention_hd128_1000", "kind": "attention", "rows": 1000, "pos": 1048, "heads": 32, "kv_heads": 4,
         "hd": 128, "max_seq": 4096},
        # one MoE layer (128 experts, top 8) for a decoding batch of 32 tokens
        {"name": "moe_32", "kind": "moe", "tokens": 32, "experts": 128, "top_k": 8, "hidden": 2048, "inter": 768,
         "type": "Q4_K", "down": "Q6_K", "mode": "bf16"},
        # the same layer for a 512-token prefill
        {"name": "moe_512", "kind": "moe", "tokens": 512, "experts": 128, "top_k": 8, "hidden": 2048, "inter": 768,
         "type": "Q4_K", "down": "Q6_K", "mode": "bf16"},
        # a whole 24-layer model: prefill of a 961-token prompt, bf16 GEMMs, to the first logits
        {"name": "model_prefill_961", "kind": "model", "layers": 24, "vocab": 151936, "prompt": 961, "new": 1,
         "mode": "bf16"},
        # the same model answering a short prompt: prefill of 37 tokens, 24 greedy tokens (f32 GEMMs)
        {"name": "model_generate_24", "kind": "model", "layers": 24, "vocab": 151936, "prompt": 37, "new": 24,
         "mode": "f32"},
    ]


def _log(rng, lo, hi, step=1):
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))) // step * step))


def draw(rng):
    kind = rng.choice(["matvec", "matmul", "matmul", "matmul", "dense", "i8", "attention", "attention", "moe", "moe",
                       "model"])
    if kind == "matvec":
        return {"kind": kind, "type": rng.choice(sorted(TYPES)), "m": _log(rng, 64, 32768),
                "n": _log(rng, 128, 4864, 32)}
    if kind in ("matmul", "dense", "i8"):
        c = {"kind": kind}
        if kind != "i8":
            c["type"] = rng.choice(sorted(TYPES if kind == "matmul" else DENSE))
        top = 4096 if kind == "matmul" else 2048
        c["m"], c["n"] = _log(rng, 64, 14336), _log(rng, 256, 14336, 8 if kind == "dense" else 32)
        c["rows"] = _log(rng, 1 if kind == "dense" else 2, top)
        if kind != "i8":
            c["mode"] = rng.choice(sorted(MODES))
        cost = (3 if c.get("mode") == "f32" else 1) * (1 if kind == "matmul" else 4)
        while cost * c["m"] * c["n"] * c["rows"] > 14336 * 4096 * 2048:       # no dearer than the largest listed
            c["m"], c["rows"] = max(64, c["m"] * 2 // 3), max(2, c["rows"] * 2 // 3)
        return c
    if kind == "attention":
        heads, kv, hd = rng.choice([(14, 2, 64), (16, 8, 64), (32, 4, 128), (24, 8, 128), (12, 12, 64)])
        rows, pos = _log(rng, 1, 2048), _log(rng, 1, 4096) - 1
        while rows * (pos + rows // 2) * heads * hd > 1000 * 1548 * 32 * 128:
            rows = max(1, rows * 2 // 3)
        return {"kind": kind, "rows": rows, "pos": pos, "heads": heads, "kv_heads": kv, "hd": hd,
                "max_seq": max(2048, -(-(rows + pos) // 1024) * 1024)}
    if kind == "moe":
        ne, k, hidden, inter = rng.choice([(128, 8, 2048, 768), (64, 8, 2048, 768), (64, 6, 1024, 512),
                                           (16, 4, 1024, 1408), (8, 2, 2048, 2048)])
        return {"kind": kind, "tokens": _log(rng, 1, 512), "experts": ne, "top_k": k, "hidden": hidden,
                "inter": inter, "type": rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q5_0", "Q4_0"]),
                "down": rng.choice(["Q6_K", "Q4_K", "Q8_0"]), "mode": rng.choice(["bf16", "bf16", "f32"])}
    return {"kind": "model", "layers": rng.randint(2, 6), "vocab": 8192, "prompt": _log(rng, 1, 961),
            "new": rng.randint(1, 12), "mode": rng.choice(sorted(MODES))}


# ---- inputs ------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _blocks(g, name, m, n, std=None):
    """GGUF blocks of an m x n matrix: uint8 (m, blocks per row, block bytes)."""
    qk, bb = rehip.GEOM[TYPES[name]]
    std = n ** -0.5 if std is None else std
    nb = -(-n // qk)
    raw = torch.randint(0, 256, (m, nb, bb), generator=g, device="cuda", dtype=torch.uint8)
    d = _randn(g, m, nb) * (std / UNIT[name])
    if name in ("Q4_K", "Q5_K"):
        d = d.abs().to(torch.float16).float()
        raw[..., 0:2], raw[..., 2:4] = _f16_bytes(d), _f16_bytes(d * (7.5 if name == "Q4_K" else 15.5))
    elif name == "Q6_K":
        raw[..., 192:208] = torch.randint(-64, 64, (m, nb, 16), generator=g, device="cuda",
                                          dtype=torch.int8).view(torch.uint8)
        raw[..., 208:210] = _f16_bytes(d)
    else:
        raw[..., 0:2] = _f16_bytes(d)
    return raw


def _host(t):
    return t.contiguous().view(torch.uint8).reshape(-1).cpu().numpy()


def _matmul_inputs(case, g):
    m, n, rows = case["m"], case["n"], case.get("rows", 1)
    if case["kind"] == "dense":
        w = (_randn(g, m, n) * n ** -0.5).to(DENSE[case["type"]][1])
    else:
        w = _blocks(g, case.get("type", "Q8_0"), m, n)
    return w, _randn(g, rows, n)


def _attention_inputs(case, g):
    hd, total = case["hd"], case["pos"] + case["rows"]
    q = 2.0 * _randn(g, case["rows"], case["heads"], hd)
    kc = torch.zeros(case["max_seq"], case["kv_heads"], hd, device="cuda")
    vc = torch.zeros_like(kc)
    kc[:total] = _randn(g, total, case["kv_heads"], hd)
    vc[:total] = _randn(g, total, case["kv_heads"], hd)
    return q, kc, vc


def _moe_inputs(case, g):
    ne, h, i = case["experts"], case["hidden"], case["inter"]
    gate = _blocks(g, case["type"], ne * i, h)
    up = _blocks(g, case["type"], ne * i, h)
    down = _blocks(g, case["down"], ne * h, i)
    return gate, up, down, _randn(g, ne, h) * h ** -0.5, _randn(g, case["tokens"], h)


def _model_inputs(case, g):
    """Blocks of every tensor (Q4_K attention and gate / up, Q6_K down, Q8_0 embedding and head)."""
    geo = qwen.QWEN25_05B
    d, kv, ff = geo.d_model, geo.n_kv_heads * geo.head_dim, geo.d_ff
    layers = []
    for _ in range(case["layers"]):
        b = {"q": _blocks(g, "Q4_K", d, d), "k": _blocks(g, "Q4_K", kv, d), "v": _blocks(g, "Q4_K", kv, d),
             "o": _blocks(g, "Q4_K", d, d), "gate": _blocks(g, "Q4_K", ff, d), "up": _blocks(g, "Q4_K", ff, d),
             "down": _blocks(g, "Q6_K", d, ff)}
        for norm in ("attn_norm", "ffn_norm"):
            b[norm] = 1 + 0.1 * _randn(g, d)
        for bias, width in (("q_bias", d), ("k_bias", kv), ("v_bias", kv)):
            b[bias] = 0.1 * _randn(g, width)
        layers.append(b)
    embed, out = (_blocks(g, "Q8_0", case["vocab"], d, 0.1) for _ in range(2))
    out_norm = 1 + 0.1 * _randn(g, d)
    prompt = torch.randint(0, case["vocab"], (case["prompt"],), generator=g, device="cuda")
    return layers, embed, out, out_norm, prompt


# ---- the calls ---------------------------------------------------------------------------------
def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = {"case": case}
    if kind in ("matvec", "matmul", "dense", "i8"):
        w, s["x"] = _matmul_inputs(case, g)
        m, n, rows = case["m"], case["n"], case.get("rows", 1)
        t = DENSE[case["type"]][0] if kind == "dense" else TYPES[case.get("type", "Q8_0")]
        s["q"] = rehip.QMat.from_bytes(t, _host(w), m, n)
        s["y"] = torch.empty(rows, m, device="cuda")
        if kind == "i8":
            s["scales"] = torch.empty(rows, n // 32, device="cuda")
            s["qs"] = torch.empty(rows, n, device="cuda", dtype=torch.int8)
    elif kind == "attention":
        s["q"], s["kc"], s["vc"] = _attention_inputs(case, g)
        s["pos"] = torch.full((1,), case["pos"], device="cuda", dtype=torch.int32)
        s["ctx"] = torch.empty_like(s["q"])
        # the split workspace of a decoding program; a prefill call has no use for it
        few = case["rows"] < 8
        s["work_bytes"] = rehip.attention_work_bytes(case["rows"], case["heads"], case["hd"],
                                                     case["max_seq"]) if few else 0
        s["work"] = torch.empty(s["work_bytes"] // 4, device="cuda") if few else None
    elif kind == "moe":
        gate, up, down, s["router"], s["x"] = _moe_inputs(case, g)
        t, td = TYPES[case["type"]], TYPES[case["down"]]
        s["e"] = rehip.MoeExperts(t, _host(gate), t, _host(up), td, _host(down), case["experts"], case["hidden"],
                                  case["inter"])
        s["out"] = torch.empty(case["tokens"], case["hidden"], device="cuda")
    else:
        layers, embed, out, out_norm, prompt = _model_inputs(case, g)
        blocks = [qwen.BlockBytes(**{k: v.cpu().numpy() if v.dtype == torch.float32 else _host(v)
                                     for k, v in b.items()}) for b in layers]
        mb = qwen.ModelBytes(qwen.QWEN25_05B, case["vocab"], _host(embed), _host(out), out_norm.cpu().numpy(), blocks)
        s["dec"] = qwen.DeviceDecoder(mb, max_seq=-(-(case["prompt"] + case["new"] + 1) // 128) * 128,
                                      mode=MODES[case["mode"]])
        mb.blocks = []
        s["prompt"] = prompt.cpu().numpy().astype(np.int32)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "matvec":
        s["q"].matvec_dev(s["x"].data_ptr(), s["y"].data_ptr())
        return s["y"]
    if kind in ("matmul", "dense"):
        s["q"].matmul_dev(s["x"].data_ptr(), case["rows"], s["y"].data_ptr(), MODES[case["mode"]])
        return s["y"]
    if kind == "i8":
        rehip.quantize_q8_act_dev(s["x"].data_ptr(), case["rows"], case["n"], s["scales"].data_ptr(),
                                  s["qs"].data_ptr())
        s["q"].matmul_i8_dev(s["scales"].data_ptr(), s["qs"].data_ptr(), case["rows"], s["y"].data_ptr())
        return {"y": s["y"], "scales": s["scales"], "qs": s["qs"]}
    if kind == "attention":
        rehip.attention_dev(s["q"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(), case["rows"], case["heads"],
                            case["kv_heads"], case["hd"], case["max_seq"], s["pos"].data_ptr(), s["ctx"].data_ptr(),
                            work=s["work"].data_ptr() if s["work"] is not None else None,
                            work_bytes=s["work_bytes"])
        return s["ctx"]
    if kind == "moe":
        s["e"].layer_dev(s["x"].data_ptr(), case["tokens"], s["router"].data_ptr(), case["top_k"],
                         rehip.GATE_SOFTMAX, s["out"].data_ptr(), MODES[case["mode"]])
        return s["out"]
    dec = s["dec"]                       # a new conversation: position 0, then prompt and answer
    dec.seq_len = 0
    dec.pos.zero()
    tokens = dec.generate(s["prompt"], case["new"])
    return {"logits": dec.logits(), "tokens": np.asarray(tokens, np.int64)}


# ---- what a pass cannot do without -----------------------------------------------------------------
def _row_bytes(name, n):
    qk, bb = rehip.GEOM[TYPES[name]]
    return -(-n // qk) * bb


def work(case):
    kind = case["kind"]
    if kind in ("matvec", "matmul", "dense", "i8"):
        m, n, rows = case["m"], case["n"], case.get("rows", 1)
        wb = m * n * rehip.DENSE_TYPES[DENSE[case["type"]][0]] if kind == "dense" else \
            m * _row_bytes(case.get("type", "Q8_0"), n)
        extra = rows * n + 4 * rows * (n // 32) if kind == "i8" else 0
        return {"bytes": wb + 4 * rows * (m + n) + extra, "flops": 2 * m * n * rows}
    if kind == "attention":
        h, hd, rows = case["heads"], case["hd"], case["rows"]
        keys = sum(case["pos"] + r + 1 for r in range(rows))
        return {"bytes": 4 * hd * (2 * rows * h + 2 * case["kv_heads"] * (case["pos"] + rows)),
                "flops": 4 * keys * h * hd}
    if kind == "moe":
        t, ne, k, h, i = (case[x] for x in ("tokens", "experts", "top_k", "hidden", "inter"))
        hit = ne * (1 - (1 - k / ne) ** t)
        expert = 2 * i * _row_bytes(case["type"], h) + h * _row_bytes(case["down"], i)
        return {"bytes": int(hit * expert) + 4 * ne * h + 8 * t * h, "flops": 2 * t * h * (3 * k * i + ne)}
    geo, p, new = qwen.QWEN25_05B, case["prompt"], case["new"]
    d, kv, ff = geo.d_model, geo.n_kv_heads * geo.head_dim, geo.d_ff
    layer = (2 * d + 2 * kv + 2 * ff) * _row_bytes("Q4_K", d) + d * _row_bytes("Q6_K", ff)
    head = case["vocab"] * _row_bytes("Q8_0", d)
    params = d * (2 * d + 2 * kv) + 3 * d * ff
    keys = sum(range(1, p + 1)) + sum(range(p + 1, p + new))
    flops = 2 * case["layers"] * params * (p + new - 1) + 4 * case["layers"] * keys * d + 2 * case["vocab"] * d * new
    return {"bytes": new * (case["layers"] * layer + head) + 4 * case["vocab"], "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "i8":
        return "exact"                   # integer dots folded in a fixed order: the same bits
    if kind == "attention" or kind == "matvec":
        return {"rel": 1e-5}             # f32 products and sums
    if kind == "model":
        # a change of rounding passes through every later layer
        return {"rel": 0.03 if case["mode"] == "bf16" else 1e-3, "differ": 0.01}
    if case["mode"] == "bf16" and case.get("rows", 16) > 1:
        return {"rel": 1e-2}             # operands rounded to bf16
    # split operands, each product within about 2^-16 (two products deep in the expert FFN)
    return {"rel": 3e-5 if kind == "moe" else 2e-5}


# ---- the same in 64 bits -----------------------------------------------------------------------
def _f16(raw, at):
    return raw[..., at:at + 2].contiguous().view(torch.float16).double()


def _dequant(name, raw, n):
    """f64 (m, n) values of GGUF blocks (m, blocks, bytes)."""
    m = raw.shape[0]
    lo, hi = (lambda b: b & 15), (lambda b: b >> 4)
    if name in ("Q4_0", "Q5_0"):
        qs = raw[..., 2:18] if name == "Q4_0" else raw[..., 6:22]
        q = torch.cat([lo(qs), hi(qs)], -1)
        if name == "Q5_0":
            bit = torch.arange(8, device=raw.device, dtype=torch.uint8)
            q = q | ((raw[..., 2:6, None] >> bit & 1).reshape(*raw.shape[:2], 32) << 4)
        v = (q.double() - (8 if name == "Q4_0" else 16)) * _f16(raw, 0)
    elif name == "Q8_0":
        v = raw[..., 2:34].contiguous().view(torch.int8).double() * _f16(raw, 0)
    elif name in ("Q4_K", "Q5_K"):
        s = raw[..., 4:16]
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | (s[..., :4] >> 6 << 4)], -1)
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | (s[..., 4:8] >> 6 << 4)], -1)
        qs = raw[..., 16:144] if name == "Q4_K" else raw[..., 48:176]
        qs = qs.reshape(*raw.shape[:2], 4, 1, 32)
        q = torch.cat([lo(qs), hi(qs)], -2).reshape(*raw.shape[:2], 8, 32)
        if name == "Q5_K":
            bit = torch.arange(8, device=raw.device, dtype=torch.uint8)[:, None]
            q = q | ((raw[..., None, 16:48] >> bit & 1) << 4)
        v = q.double() * (sc.double() * _f16(raw, 0))[..., None] - (mn.double() * _f16(raw, 2))[..., None]
    else:
        ql, qh = raw[..., :128].reshape(*raw.shape[:2], 2, 2, 32), raw[..., 128:192].reshape(*raw.shape[:2], 2, 32)
        q = torch.stack([lo(ql[..., 0, :]) | (qh & 3) << 4, lo(ql[..., 1, :]) | (qh >> 2 & 3) << 4,
                         hi(ql[..., 0, :]) | (qh >> 4 & 3) << 4, hi(ql[..., 1, :]) | (qh >> 6) << 4], -2)
        sc = raw[..., 192:208].contiguous().view(torch.int8).double() * _f16(raw, 208)
        v = (q.reshape(*raw.shape[:2], 16, 16).double() - 32) * sc[..., None]
    return v.reshape(m, -1)[:, :n]


def _silu(v):
    return v / (1 + torch.exp(-v))


def _attend(q, k, v, pos):
    """f64 causal attention, q (rows, heads, hd) at positions pos.., k and v (keys, kv_heads, hd)."""
    rows, heads, hd = q.shape
    grp, out = heads // k.shape[1], torch.empty(q.shape, device=q.device, dtype=torch.float64)
    hidden = torch.arange(k.shape[0], device=q.device)[None] > pos + torch.arange(rows, device=q.device)[:, None]
    for h in range(heads):
        s = (q[:, h].double() @ k[:, h // grp].double().T.contiguous()) * hd ** -0.5
        p = torch.softmax(s.masked_fill(hidden, -math.inf), -1)
        out[:, h] = p @ v[:, h // grp].double()
    return out


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind in ("matvec", "matmul", "dense", "i8"):
        w, x = _matmul_inputs(case, g)
        wd = w.double() if kind == "dense" else _dequant(case.get("type", "Q8_0"), w, case["n"])
        if kind == "i8":                 # the activations as their int8 blocks say
            b = x.reshape(case["rows"], -1, 32)
            d = b.abs().amax(-1, keepdim=True) / 127
            r = b / d
            qi = (torch.sign(r) * torch.floor(r.abs() + 0.5)).clamp(-127, 127).double()
            x = (qi * d.double()).reshape(case["rows"], -1)
            return {"y": x @ wd.T.contiguous(), "scales": None, "qs": None}
        return x.double() @ wd.T.contiguous()
    if kind == "attention":
        q, kc, vc = _attention_inputs(case, g)
        total = case["pos"] + case["rows"]
        return _attend(q, kc[:total], vc[:total], case["pos"])
    if kind == "moe":
        gate, up, down, router, x = _moe_inputs(case, g)
        h, i, xd = case["hidden"], case["inter"], x.double()
        w, ids = torch.topk(xd @ router.double().T.contiguous(), case["top_k"], -1)
        w, out = torch.softmax(w, -1), torch.zeros_like(xd)
        for e in range(case["experts"]):
            t, slot = torch.nonzero(ids == e, as_tuple=True)
            if not len(t):
                continue
            gw, uw = (_dequant(case["type"], b[e * i:(e + 1) * i], h).T.contiguous() for b in (gate, up))
            dw = _dequant(case["down"], down[e * h:(e + 1) * h], i).T.contiguous()
            out.index_add_(0, t, ((_silu(xd[t] @ gw) * (xd[t] @ uw)) @ dw) * w[t, slot, None])
        return out
    if case["new"] > 1:                  # greedy tokens of 64-bit logits need not be the model's
        return None
    layers, embed, out, out_norm, prompt = _model_inputs(case, g)
    geo = qwen.QWEN25_05B
    d, hd, ff = geo.d_model, geo.head_dim, geo.d_ff
    norm = lambda v, w: v / torch.sqrt((v * v).mean(-1, keepdim=True) + geo.rms_eps) * w.double()  # noqa: E731
    proj = lambda v, t, w, n: v @ _dequant(t, w, n).T.contiguous()  # noqa: E731
    freq = geo.rope_freq_base ** (-2 * torch.arange(hd // 2, device="cuda", dtype=torch.float64) / hd)
    ang = torch.arange(len(prompt), device="cuda", dtype=torch.float64)[:, None, None] * freq

    def rope(v):
        a, b = v.reshape(len(prompt), -1, hd).split(hd // 2, -1)
        return torch.cat([a * torch.cos(ang) - b * torch.sin(ang), b * torch.cos(ang) + a * torch.sin(ang)], -1)

    x = _dequant("Q8_0", embed[prompt], d)
    for b in layers:
        y = norm(x, b["attn_norm"])
        q, k, v = (proj(y, "Q4_K", b[t], d) + b[t + "_bias"].double() for t in "qkv")
        ctx = _attend(rope(q), rope(k), v.reshape(len(prompt), -1, hd), 0)
        x = x + proj(ctx.reshape(len(prompt), d), "Q4_K", b["o"], d)
        y = norm(x, b["ffn_norm"])
        x = x + proj(_silu(proj(y, "Q4_K", b["gate"], d)) * proj(y, "Q4_K", b["up"], d), "Q6_K", b["down"], ff)
    return {"logits": proj(norm(x[-1:], out_norm), "Q8_0", out, d)[0], "tokens": None}
