"""Workloads of the kernel layer and the engine, called through their public
entry points (include/cactus_hip.h, cactus_amd.engine).

Each case is a dict of plain values with a "kind":

  matmul     grouped INT8 / packed INT4 weights x FP16 activations (the row
             quantization included), with or without the residual add
  dense      FP16 weights x FP16 activations, FP16 accumulation
  head       the end of a sampled decode step: logits over the vocabulary,
             then temperature, top-k, top-p and the draw
  attention  one layer's attention: FP16 keys / values, or the INT8 KV cache
             plus the new FP16 rows; exact order or tolerance ("fast") mode
  pointwise  the non-matmul part of an encoder or decoder block: norm of the
             residual stream, activation of the MLP's hidden rows, residual add
  generate   a whole model: prefill of a prompt, then greedy decode steps

Every FP16 result of the exact entry points is defined bit for bit (integer
group sums, the order of every rounding), so their outputs are compared
exactly; the tolerance-mode attention has a relative error.
"""
import math

import numpy as np
import torch

import cactus_amd as cm
from cactus_amd.engine import Qwen, qwen3_0p6b

DEV = "cuda"


def listed():
    return [
        # one decode projection of a small model: the smallest call, all latency
        {"name": "int8_m1", "kind": "matmul", "bits": 8, "M": 1, "K": 640, "N": 2048, "gs": 32, "add": False},
        # the MLP down projection of a decode step with its residual
        {"name": "int4_m1_add", "kind": "matmul", "bits": 4, "M": 1, "K": 3072, "N": 1024, "gs": 32, "add": True},
        # a chat turn of a few words: the q projection of a short prefill
        {"name": "int8_m19", "kind": "matmul", "bits": 8, "M": 19, "K": 1024, "N": 2048, "gs": 32, "add": False},
        # the gate / up projection of a 512-token prefill
        {"name": "int8_m512", "kind": "matmul", "bits": 8, "M": 512, "K": 1024, "N": 3072, "gs": 32, "add": False},
        # a ragged prompt through a down projection in the converter's default group size
        {"name": "int4_m777_g128", "kind": "matmul", "bits": 4, "M": 777, "K": 3072, "N": 1024, "gs": 128, "add": True},
        # a layer kept in FP16, on a short prompt
        {"name": "f16_m100", "kind": "dense", "M": 100, "K": 1024, "N": 3072},
        # the tail of a sampled decode step over the full vocabulary
        {"name": "sampled_head", "kind": "head", "K": 1024, "V": 151936, "temperature": 0.6, "top_p": 0.95, "top_k": 20},
        # one decode step's attention late in a long conversation
        {"name": "attn_decode_4096", "kind": "attention", "cache": "int8", "fast": False, "S": 1, "ctx": 4096,
         "Hq": 16, "Hkv": 8, "d": 128},
        # one prefill chunk's attention in the middle of a long prompt
        {"name": "attn_prefill_256", "kind": "attention", "cache": "int8", "fast": False, "S": 256, "ctx": 2048,
         "Hq": 16, "Hkv": 8, "d": 128},
        # a prefill chunk of odd length in tolerance mode
        {"name": "attn_fast_333", "kind": "attention", "cache": "int8", "fast": True, "S": 333, "ctx": 3000,
         "Hq": 16, "Hkv": 8, "d": 128},
        # an audio encoder block's 1500 frames
        {"name": "encoder_1500", "kind": "pointwise", "norm": "layer", "act": "gelu_erf", "rows": 1500, "width": 1280,
         "ffn": 5120},
        # a question of 777 tokens and the first 16 tokens of the answer, Qwen3-0.6B shape
        {"name": "generate_777", "kind": "generate", "layers": 28, "prompt": 777, "new": 16},
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, round(v / step) * step)))


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "matmul", "dense", "head", "attention", "attention", "pointwise", "generate"])
    if kind == "matmul":
        gs = rng.choice([32, 32, 32, 64, 128])
        return {"kind": kind, "bits": rng.choice([8, 4]), "M": _log(rng, 1, 1024), "K": _log(rng, 256, 4096, gs), "gs": gs,
                "N": _log(rng, 256, 8192, rng.choice([1, 8, 64])), "add": rng.random() < 0.4}
    if kind == "dense":
        return {"kind": kind, "M": _log(rng, 1, 512), "K": _log(rng, 128, 4096, 8), "N": _log(rng, 128, 4096)}
    if kind == "head":
        return {"kind": kind, "K": _log(rng, 512, 1536, 64), "V": _log(rng, 30000, 152000),
                "temperature": round(rng.uniform(0.3, 1.3), 2), "top_p": round(rng.uniform(0.7, 1.0), 2),
                "top_k": _log(rng, 1, 100)}
    if kind == "attention":
        Hkv, g = rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4])
        S = rng.choice([1, _log(rng, 2, 512)])
        return {"kind": kind, "cache": rng.choice(["int8", "int8", "f16"]), "fast": rng.random() < 0.4, "S": S,
                "ctx": max(S, _log(rng, 16, 4096)), "Hq": Hkv * g, "Hkv": Hkv, "d": rng.choice([64, 128, 128])}
    if kind == "pointwise":
        width = _log(rng, 256, 2048, rng.choice([1, 8, 64]))
        return {"kind": kind, "norm": rng.choice(["layer", "rms"]), "act": rng.choice(["gelu", "gelu_erf", "silu"]),
                "rows": _log(rng, 1, 1500), "width": width, "ffn": width * rng.choice([2, 3, 4])}
    return {"kind": kind, "layers": rng.randint(1, 28), "prompt": _log(rng, 8, 700), "new": rng.randint(1, 15)}


# ------------------------------------------------------------------ inputs
def _normal(g, *shape, sd=1.0, mean=0.0):
    return (torch.randn(*shape, generator=g, device=DEV) * sd + mean).half()


def _quantize_rows(x):
    """Symmetric INT8 codes and scales of the last dimension's rows."""
    x = x.float()
    s = (x.abs().amax(-1, keepdim=True) / 127.0).clamp_min(1e-10)
    return torch.round(x * (1.0 / s)).clamp(-128, 127).to(torch.int8), s


def _inputs(case, seed):
    """What the call gets, in plain torch on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    k = case["kind"]
    if k == "matmul":
        M, K, N, gs = case["M"], case["K"], case["N"], case["gs"]
        q = 127 if case["bits"] == 8 else 7
        codes = torch.randint(-q, q + 1, (N, K), generator=g, device=DEV, dtype=torch.int8)
        return {"x": _normal(g, M, K), "codes": codes, "scales": (torch.randn(N, K // gs, generator=g, device=DEV).abs() * 0.02 / q).half(),
                "res": _normal(g, M, N) if case["add"] else None}
    if k == "dense":
        return {"x": _normal(g, case["M"], case["K"]), "w": _normal(g, case["N"], case["K"], sd=0.03)}
    if k == "head":
        return {"x": _normal(g, 1, case["K"]), "w": _normal(g, case["V"], case["K"], sd=0.05)}
    if k == "attention":
        S, T, Hq, Hkv, d = case["S"], case["ctx"], case["Hq"], case["Hkv"], case["d"]
        i = {"q": _normal(g, S, Hq, d), "k": _normal(g, T, Hkv, d), "v": _normal(g, T, Hkv, d)}
        if case["cache"] == "int8":  # the last S positions are the new rows
            for n in ("k", "v"):
                i[n + "_new"] = i[n][T - S:].contiguous()
                i[n], s = _quantize_rows(i[n][:T - S])
                i[n + "_scales"] = s.contiguous()
        return i
    if k == "pointwise":
        R, W, F = case["rows"], case["width"], case["ffn"]
        return {"x": _normal(g, R, W), "w": _normal(g, W, sd=0.1, mean=1.0), "b": _normal(g, W, sd=0.1),
                "h": _normal(g, R, F), "o": _normal(g, R, W)}
    r = np.random.default_rng(int(seed))
    return {"prompt": r.integers(0, 151936, case["prompt"], dtype=np.uint32)}


def prepare(case, seed):
    """The inputs, the weights in the layout the entry point takes and the
    output buffers, as a program holds them across calls."""
    s = dict(_inputs(case, seed), case=case)
    k = case["kind"]
    if k == "matmul":
        c = s.pop("codes")
        s["B"] = c if case["bits"] == 8 else ((c[:, 0::2] & 15) | (c[:, 1::2] << 4)).contiguous()
        s["C"] = torch.empty(case["M"], case["N"], dtype=torch.float16, device=DEV)
    elif k == "dense":
        s["C"] = torch.empty(case["M"], case["N"], dtype=torch.float16, device=DEV)
    elif k == "head":
        s["logits"] = torch.empty(case["V"], dtype=torch.float16, device=DEV)
        s["token"] = torch.zeros(1, dtype=torch.int32, device=DEV)
        s["seed"] = int(seed) % 100003 + 1
    elif k == "attention":
        s["out"] = torch.empty_like(s["q"])
    elif k == "pointwise":
        s["norm"], s["act"], s["sum"] = (torch.empty_like(s[n]) for n in ("x", "h", "x"))
    else:
        cfg = dict(qwen3_0p6b(max_seq=1024), num_layers=case["layers"])
        s["model"] = Qwen(cfg, seed=int(seed) % 1000003 + 1)
        s["model"].set_decode_mode(1)
    return s


def run(s):
    c = s["case"]
    k = c["kind"]
    if k == "matmul":
        name = "cactus_hip_matmul_int%d_f16act" % c["bits"]
        args = [s["x"].data_ptr(), s["B"].data_ptr(), s["scales"].data_ptr()]
        if c["add"]:
            name += "_add"
            args.append(s["res"].data_ptr())
        cm.call(name, *args, s["C"].data_ptr(), c["M"], c["K"], c["N"], c["gs"], None)
        return s["C"]
    if k == "dense":
        cm.call("cactus_hip_matmul_f16", s["x"].data_ptr(), s["w"].data_ptr(), s["C"].data_ptr(), c["M"], c["K"], c["N"], None)
        return s["C"]
    if k == "head":
        # the first token of a new answer: the repetition history starts empty
        cm.call("cactus_hip_sample_history_reset", None)
        cm.call("cactus_hip_matmul_f16", s["x"].data_ptr(), s["w"].data_ptr(), s["logits"].data_ptr(), 1, c["K"], c["V"], None)
        cm.call("cactus_hip_sample_f16", s["logits"].data_ptr(), s["token"].data_ptr(), c["V"], c["temperature"], c["top_p"],
                c["top_k"], s["seed"], None)
        return {"logits": s["logits"], "token": s["token"]}
    if k == "attention":
        T, S = c["ctx"], c["S"]
        heads = (c["Hq"], c["Hkv"], c["d"], 1.0 / math.sqrt(c["d"]))
        fast = "_fast" if c["fast"] else ""
        if c["cache"] == "int8":
            cm.call("cactus_hip_attention_hybrid_int8_fp16" + fast, s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                    s["k_scales"].data_ptr(), s["v_scales"].data_ptr(), s["k_new"].data_ptr(), s["v_new"].data_ptr(),
                    s["out"].data_ptr(), 1, S, T - S, S, *heads, T - S, 1, 128, None)
        else:
            cm.call("cactus_hip_attention_f16" + fast, s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                    s["out"].data_ptr(), 1, S, T, *heads, None, T - S, 0, 1, None)
        return s["out"]
    if k == "pointwise":
        R, W = c["rows"], c["width"]
        if c["norm"] == "layer":
            cm.call("cactus_hip_layer_norm_f16", s["x"].data_ptr(), s["w"].data_ptr(), s["b"].data_ptr(), s["norm"].data_ptr(),
                    R, W, 1e-5, None)
        else:
            cm.call("cactus_hip_rms_norm_f16", s["x"].data_ptr(), s["w"].data_ptr(), s["norm"].data_ptr(), R, W, 1e-6, None)
        cm.call("cactus_hip_%s_f16" % c["act"], s["h"].data_ptr(), s["act"].data_ptr(), R * c["ffn"], None)
        cm.call("cactus_hip_add_f16", s["x"].data_ptr(), s["o"].data_ptr(), s["sum"].data_ptr(), R * W, None)
        return {"norm": s["norm"], "act": s["act"], "sum": s["sum"]}
    m = s["model"]
    m.reset()
    tokens, _ = m.generate(s["prompt"], c["new"])
    return {"logits": m.last_logits().view(np.float16), "tokens": tokens.astype(np.int64)}


def work(case):
    k = case["kind"]
    if k == "matmul":
        M, K, N, gs = case["M"], case["K"], case["N"], case["gs"]
        return {"bytes": N * K * case["bits"] // 8 + 2 * N * (K // gs) + 2 * M * K + 2 * M * N * (2 if case["add"] else 1),
                "flops": 2 * M * N * K}
    if k == "dense":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 2 * (N * K + M * K + M * N), "flops": 2 * M * N * K}
    if k == "head":
        return {"bytes": 2 * case["V"] * (case["K"] + 2), "flops": 2 * case["V"] * case["K"]}
    if k == "attention":
        S, T, Hq, Hkv, d = case["S"], case["ctx"], case["Hq"], case["Hkv"], case["d"]
        kv = 2 * Hkv * ((T - S) * (d + 4) + S * d * 2) if case["cache"] == "int8" else 2 * Hkv * T * d * 2
        return {"bytes": kv + 4 * S * Hq * d, "flops": 4 * Hq * d * (S * (T - S) + S * (S + 1) // 2)}
    if k == "pointwise":
        R, W, F = case["rows"], case["width"], case["ffn"]
        return {"bytes": 2 * R * (5 * W + 2 * F), "flops": R * (10 * W + 20 * F)}
    c = qwen3_0p6b()
    H, F, hd, L, P, n = c["hidden"], c["ffn"], c["head_dim"], case["layers"], case["prompt"], case["new"]
    qkvo = H * hd * (2 * c["heads"] + 2 * c["kv_heads"])
    weights = L * (qkvo * (1 + 2 / 32) + 3 * H * F * (0.5 + 2 / 32))
    head = 2 * c["vocab"] * H
    kv = L * 2 * c["kv_heads"] * (hd + 4) * (P * n + n * n // 2)
    attn = 4 * L * c["heads"] * hd * (P + n) ** 2 / 2
    return {"bytes": weights * (1 + n) + head * n + kv, "flops": 2 * L * (qkvo + 3 * H * F) * (P + n) + head * n + attn}


def tolerance(case):
    # tolerance mode: 3.3e-4 from the 64-bit result (measured), so two correct
    # forms lie up to 4.7e-4 apart; four times that
    if case["kind"] == "attention" and case["fast"]:
        return {"rel": 2e-3}
    return "exact"


# ------------------------------------------------------------------ 64 bits
def _attention64(case, i):
    S, T, Hq, Hkv, d = case["S"], case["ctx"], case["Hq"], case["Hkv"], case["d"]
    kv = {}
    for n in ("k", "v"):
        x = i[n].double()
        if case["cache"] == "int8":
            x = torch.cat([x * i[n + "_scales"].double(), i[n + "_new"].double()])
        kv[n] = x.transpose(0, 1).repeat_interleave(Hq // Hkv, 0).contiguous()      # [Hq][T][d]
    q = i["q"].double().transpose(0, 1).contiguous()                                # [Hq][S][d]
    pos = torch.arange(T - S, T, device=DEV)
    out = torch.empty(Hq, S, d, dtype=torch.float64, device=DEV)
    for h in range(Hq):
        s = (q[h] @ kv["k"][h].t().contiguous()) / math.sqrt(d)
        s = s.masked_fill(torch.arange(T, device=DEV)[None] > pos[:, None], -math.inf)
        if case["cache"] == "int8":
            p = torch.softmax(s, -1)
        else:
            # blocks of 32 keys; the weights of a block's first floor(n/4)*4
            # keys are the second-order 2^x of kernel_attention.cpp:174-195
            nb = -(-T // 32)
            sb = torch.nn.functional.pad(s, (0, nb * 32 - T), value=-math.inf).view(S, nb, 32)
            bm = sb.amax(-1, keepdim=True)
            x = (sb - torch.where(torch.isinf(bm), torch.zeros_like(bm), bm)) * 1.442695
            f = x - torch.trunc(x)
            poly = (1 + 0.6931472 * f + 0.2402265 * f * f) * torch.exp2(torch.trunc(x))
            n = (pos[:, None] + 1 - 32 * torch.arange(nb, device=DEV)[None]).clamp(0, 32)
            body = torch.arange(32, device=DEV)[None, None] < (n // 4 * 4)[..., None]
            w = torch.where(body, poly, torch.exp2(x * (1 / (1.442695 * math.log(2.0)))))
            w = torch.where(torch.isinf(sb), torch.zeros_like(w), w) * torch.exp(bm - s.amax(-1)[:, None, None])
            p = w.reshape(S, nb * 32)[:, :T]
            p = p / p.sum(-1, keepdim=True)
        out[h] = p @ kv["v"][h]
    return out.transpose(0, 1).contiguous()


def exact(case, seed):
    k = case["kind"]
    if k == "generate":
        return None
    i = _inputs(case, seed)
    if k == "matmul":
        N, K, gs = case["N"], case["K"], case["gs"]
        a, s = _quantize_rows(i["x"])
        w = (i["codes"].double().view(N, K // gs, gs) * i["scales"].double()[..., None]).view(N, K)
        c = (a.double() @ w.t()) * s.double()
        return c + i["res"].double() if case["add"] else c
    if k == "dense":
        return i["x"].double() @ i["w"].double().t()
    if k == "head":
        return {"logits": (i["x"].double() @ i["w"].double().t()).view(-1), "token": None}
    if k == "attention":
        return _attention64(case, i)
    x, h = i["x"].double(), i["h"].double()
    if case["norm"] == "layer":
        norm = torch.nn.functional.layer_norm(x, (case["width"],), i["w"].double(), i["b"].double(), 1e-5)
    else:
        norm = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * i["w"].double()
    act = {"silu": torch.nn.functional.silu, "gelu_erf": torch.nn.functional.gelu,
           "gelu": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[case["act"]](h)
    return {"norm": norm, "act": act, "sum": x + i["o"].double()}
