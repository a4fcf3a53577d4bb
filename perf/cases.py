"""Performance cases of the quantized matrix path, each one call (or one queue) as a user's program
makes it through the public entry points (opentars_amd.ops, opentars_amd.queue).

Kinds:
  step       one descriptor queue through queue.Machine.run_queue: a whole decoder pass of `rows` tokens
             at position t0 (attention over the KV caches, MLP, head on the last row). rows = 1 is a
             decode step, rows = 4 the exports' prefill chunk. Returns the logits and the KV caches.
  group      ops.quant_gemm_rowcol: one per-token quantization feeding several matrices (q/k/v, gate/up).
  linear     ops.gemm_rowcol: W8A8 on prompt rows, with the epilogue's options.
  ksplit     ops.gemm_rowcol_ksplit: a linear whose K is cut in blocks (Gemma-3's down projection).
  w4         ops.gemm_w4: W4A16 group-128, fp32 or bf16 activations, one row (decode) to a prompt.
  attention  ops.attention: a layer's causal attention, one row (decode) to a whole prompt.
  rows       the row work between a layer's linears on prompt rows: residual add, RMSNorm, quantizer,
             RoPE, gated MLP product, quantizer.

Every result of these entry points is defined bit for bit (exact integer sums, then fp32 steps in a
fixed order), so every tolerance is "exact".
"""
from __future__ import annotations

import numpy as np
import torch

from opentars_amd import contract as C
from opentars_amd import ops
from opentars_amd import queue as Q

_OUT = {"fp32": C.OUT_FP32, "bf16": C.OUT_BF16, "int8": C.OUT_INT8}
_OUT_BYTES = {"fp32": 4, "bf16": 2, "int8": 1}
_ACT = {"none": C.ACT_NONE, "relu": C.ACT_RELU, "gelu": C.ACT_GELU, "silu": C.ACT_SILU}


def listed():
    return [
        # one token's q / k / v of a Qwen3-0.6B layer: the smallest call, latency and host work
        {"name": "decode_qkv", "kind": "group", "M": 1, "K": 1024, "N0": 2048, "N1": 1024, "N2": 1024},
        # one generated token of Qwen3-0.6B at t = 250: 28 layers and the 151936-row head, 1910 descriptors
        {"name": "decode_step", "kind": "step", "rows": 1, "layers": 28, "H": 1024, "heads": 16, "kv_heads": 8,
         "hd": 128, "ff": 3072, "vocab": 151936, "t0": 250},
        # one prefill chunk of four tokens of the same model (the exports' chunk queues)
        {"name": "prompt_chunk", "kind": "step", "rows": 4, "layers": 28, "H": 1024, "heads": 16, "kv_heads": 8,
         "hd": 128, "ff": 3072, "vocab": 151936, "t0": 100},
        # gate / up of Qwen3-0.6B on a 256-token prompt
        {"name": "prompt_linear", "kind": "linear", "M": 256, "K": 1024, "N": 3072, "bias": False, "act": "none",
         "out": "fp32"},
        # a 2048-token prompt through a 4096-wide linear: the largest
        {"name": "prompt_linear_large", "kind": "linear", "M": 2048, "K": 4096, "N": 4096, "bias": False,
         "act": "none", "out": "fp32"},
        # Gemma-3 1B's gate (1152 wide, GELU) on an odd prompt length, bf16 out
        {"name": "prompt_linear_ragged", "kind": "linear", "M": 333, "K": 1152, "N": 6912, "bias": False,
         "act": "gelu", "out": "bf16"},
        # Gemma-3 1B's down projection (6912 = 4096 + 2816) on a 500-token prompt
        {"name": "prompt_ksplit", "kind": "ksplit", "M": 500, "K0": 4096, "K1": 2816, "K2": 0, "N": 1152},
        # Gemma-4 W4A16 gate, one token
        {"name": "w4_decode", "kind": "w4", "M": 1, "K": 1536, "N": 12288, "bf16": False, "out": "fp32"},
        # the same on a 256-token prompt, bf16 activations
        {"name": "w4_prompt", "kind": "w4", "M": 256, "K": 1536, "N": 12288, "bf16": True, "out": "fp32"},
        # one token's attention late in a conversation, binary16 V cache
        {"name": "attention_decode", "kind": "attention", "M": 1, "nk": 2048, "heads": 16, "kv_heads": 8, "hd": 128,
         "v_fp16": True},
        # a 512-token prompt's causal attention
        {"name": "attention_prompt", "kind": "attention", "M": 512, "nk": 512, "heads": 16, "kv_heads": 8, "hd": 128,
         "v_fp16": False},
        # the row work of one Qwen3-0.6B layer on a 512-token prompt
        {"name": "prompt_rows", "kind": "rows", "M": 512, "H": 1024, "heads": 16, "hd": 128, "ff": 3072},
    ]


# ------------------------------------------------------------------------------------------- draws
def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], even over its logarithm."""
    v = lo * (hi / lo) ** rng.random()
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["step", "group", "linear", "linear", "ksplit", "w4", "w4", "attention", "attention", "rows"])
    if kind == "step":
        heads, kv_heads = rng.choice([(4, 1), (8, 2), (8, 8), (16, 8)])
        rows = rng.choice([1, 1, 4, rng.randint(2, 16)])
        return {"kind": kind, "rows": rows, "layers": _log(rng, 1, 8), "H": 128 * rng.randint(2, 9), "heads": heads,
                "kv_heads": kv_heads, "hd": rng.choice([64, 128]), "ff": 256 * rng.randint(2, 14),
                "vocab": _log(rng, 2048, 65536, 64), "t0": _log(rng, 1, 1000)}
    if kind == "group":
        K = _log(rng, 128, 4096, rng.choice([16, 128]))
        n = [_log(rng, 256, 4096, 16) for _ in range(rng.randint(1, 3))] + [0, 0]
        return {"kind": kind, "M": rng.choice([1, 1, rng.randint(2, 16)]), "K": K, "N0": n[0], "N1": n[1], "N2": n[2]}
    if kind == "linear":
        while True:
            c = {"kind": kind, "M": _log(rng, 2, 3000), "K": _log(rng, 256, 8192, rng.choice([16, 128, 256])),
                 "N": _log(rng, 256, 12288, rng.choice([16, 64])), "bias": rng.random() < 0.3,
                 "act": rng.choice(["none", "none", "relu", "gelu", "silu"]), "out": rng.choice(["fp32", "fp32", "bf16", "int8"])}
            if c["M"] * c["K"] * c["N"] <= 2048 * 4096 * 4096 // 2:
                return c
    if kind == "ksplit":
        step = rng.choice([16, 128, 256])
        ks = [_log(rng, 512, 4096, step) for _ in range(rng.randint(2, 3))] + [0]
        return {"kind": kind, "M": _log(rng, 1, 1000), "K0": ks[0], "K1": ks[1], "K2": ks[2], "N": _log(rng, 256, 3072, 16)}
    if kind == "w4":
        while True:
            c = {"kind": kind, "M": rng.choice([1, _log(rng, 2, 1024)]), "K": _log(rng, 256, 8192, 256),
                 "N": _log(rng, 256, 12288, 16), "bf16": rng.random() < 0.5, "out": rng.choice(["fp32", "fp32", "bf16"])}
            if c["M"] * c["K"] * c["N"] <= 256 * 1536 * 12288:
                return c
    if kind == "attention":
        while True:
            heads, kv_heads = rng.choice([(4, 1), (8, 2), (8, 8), (16, 8), (16, 4)])
            M = rng.choice([1, 1, _log(rng, 2, 512)])
            c = {"kind": kind, "M": M, "nk": max((M + 3) // 4 * 4, _log(rng, 16, 4080, 4)), "heads": heads, "kv_heads": kv_heads,
                 "hd": rng.choice([64, 128, 128, 256]), "v_fp16": rng.random() < 0.5}
            if c["M"] * c["nk"] * heads * c["hd"] <= 512 * 512 * 16 * 128:
                return c
    heads = rng.choice([4, 8, 16])
    return {"kind": kind, "M": _log(rng, 1, 2000), "H": _log(rng, 256, 2048, 16), "heads": heads,
            "hd": rng.choice([64, 128, 256]), "ff": _log(rng, 512, 8192, 16)}


# ---------------------------------------------------------------------------------------- work
def work(case):
    k = case["kind"]
    if k == "step":
        H, hq, hk, ff, L, R = case["H"], case["heads"] * case["hd"], case["kv_heads"] * case["hd"], case["ff"], case["layers"], case["rows"]
        lin = L * (H * hq + 2 * H * hk + hq * H + 3 * H * ff)
        keys = case["t0"] + R
        cache = L * 2 * 4 * keys * hk
        return {"bytes": lin + case["vocab"] * H + 4 * (case["vocab"] * 2 + R * H) + cache + L * 2 * 4 * R * hk,
                "flops": 2 * R * lin + 2 * case["vocab"] * H + L * 4 * R * keys * hq}
    if k == "group":
        M, K, N = case["M"], case["K"], case["N0"] + case["N1"] + case["N2"]
        return {"bytes": 4 * M * K + N * K + 4 * N + 4 * M * N, "flops": 2 * M * N * K}
    if k == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": M * K + 4 * M + N * K + 4 * N * (2 if case["bias"] else 1) + _OUT_BYTES[case["out"]] * M * N,
                "flops": 2 * M * N * K}
    if k == "ksplit":
        M, K, N = case["M"], case["K0"] + case["K1"] + case["K2"], case["N"]
        return {"bytes": M * K + 4 * M + N * K + 4 * N + 4 * M * N, "flops": 2 * M * N * K}
    if k == "w4":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": (2 if case["bf16"] else 4) * M * K + N * K // 2 + N * K // 64 + _OUT_BYTES[case["out"]] * M * N,
                "flops": 2 * M * N * K}
    if k == "attention":
        M, nk, hq, hk = case["M"], case["nk"], case["heads"] * case["hd"], case["kv_heads"] * case["hd"]
        pairs = sum(min(nk, nk - M + 1 + m) for m in range(M))  # causal: the (query, key) pairs that count
        return {"bytes": 8 * M * hq + nk * hk * (4 + (2 if case["v_fp16"] else 4)), "flops": 4 * pairs * hq}
    M, H, hq, ff = case["M"], case["H"], case["heads"] * case["hd"], case["ff"]
    # reads: the add's two operands, gamma, q's projection and its table, gate and up; writes: the sum, the
    # norm, q8 and its scales, the rotated rows, the product, its q8 and scales
    return {"bytes": 8 * M * H + 4 * H + 4 * M * (hq + case["hd"]) + 8 * M * ff + 8 * M * H + M * H + 4 * M + 4 * M * hq + 5 * M * ff + 4 * M,
            "flops": M * (6 * H + 3 * hq + 12 * ff)}


# ------------------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _acts(g, m, k):
    """Activation rows: normal values with a few larger channels, as a decoder's hidden states have."""
    x = torch.randn((m, k), device="cuda", generator=g)
    return x * (1 + 8 * (torch.rand(k, device="cuda", generator=g) < 0.01))


def _int8(g, n, k):
    """Per-channel quantized normal weights."""
    return (torch.randn((n, k), device="cuda", generator=g) * 42).round_().clamp_(-127, 127).to(torch.int8)


def _scol(g, n, k):
    return (0.5 + torch.rand(n, device="cuda", generator=g)) / (42 * k ** 0.5)


def _quantized(g, m, k):
    x = _acts(g, m, k)
    s = x.abs().amax(1) / 127
    return torch.round(x / s[:, None]).clamp_(-127, 127).to(torch.int8), s.contiguous()


def _rope_table(positions, rot):
    pos = torch.arange(positions, device="cuda", dtype=torch.float64)[:, None]
    f = pos / 1e6 ** (torch.arange(0, rot, 2, device="cuda", dtype=torch.float64) / rot)
    return torch.cat([f.cos(), f.sin()], 1).float().contiguous()


def prepare(case, seed):
    k, g = case["kind"], _gen(seed)
    st = {"case": case}
    if k == "step":
        return _prepare_step(case, g)
    if k == "group":
        st["x"] = _acts(g, case["M"], case["K"])
        st["mats"] = [(_int8(g, n, case["K"]), _scol(g, n, case["K"])) for n in (case["N0"], case["N1"], case["N2"]) if n]
    elif k == "linear":
        st["q"], st["s"] = _quantized(g, case["M"], case["K"])
        st["W"], st["scol"] = _int8(g, case["N"], case["K"]), _scol(g, case["N"], case["K"])
        st["bias"] = torch.randn(case["N"], device="cuda", generator=g) * 0.1 if case["bias"] else None
    elif k == "ksplit":
        ks = [case[f"K{i}"] for i in range(3) if case[f"K{i}"]]
        st["q"], st["s"] = _quantized(g, case["M"], sum(ks))
        st["W"] = [_int8(g, case["N"], kk) for kk in ks]
        st["scol"] = _scol(g, case["N"], sum(ks))
    elif k == "w4":
        x = _acts(g, case["M"], case["K"])
        st["x"] = x.bfloat16() if case["bf16"] else x
        st["Wp"] = torch.randint(0, 256, (case["N"], case["K"] // 2), dtype=torch.uint8, device="cuda", generator=g)
        st["ws"] = ((0.5 + torch.rand((case["N"], case["K"] // 128), device="cuda", generator=g)) / (4.6 * case["K"] ** 0.5)).half()
    elif k == "attention":
        st["q"] = torch.randn((case["M"], case["heads"] * case["hd"]), device="cuda", generator=g) * 2 / case["hd"] ** 0.5
        st["kc"] = torch.randn((case["nk"], case["kv_heads"] * case["hd"]), device="cuda", generator=g)
        v = torch.randn((case["nk"], case["kv_heads"] * case["hd"]), device="cuda", generator=g)
        st["vc"] = v.half() if case["v_fp16"] else v
    else:
        M, H, hd, ff = case["M"], case["H"], case["hd"], case["ff"]
        st["x"], st["o"] = _acts(g, M, H), torch.randn((M, H), device="cuda", generator=g) * 0.3
        st["gamma"] = 1 + 0.1 * torch.randn(H, device="cuda", generator=g)
        st["qp"] = torch.randn((M * case["heads"], hd), device="cuda", generator=g)
        st["tab"] = _rope_table(M, hd)
        st["gate"] = torch.randn((M, ff), device="cuda", generator=g)
        st["up"] = torch.randn((M, ff), device="cuda", generator=g)
    return st


# ----------------------------------------------------------------------------------------- runs
def run(st):
    case = st["case"]
    k = case["kind"]
    if k == "step":
        status = st["machine"].run_queue(st["qaddr"], st["n"], descs=st["queue"])
        if not status.done:
            raise RuntimeError(f"queue stopped: {status}")
        return {"logits": st["logits"], "caches": st["caches"]}
    if k == "group":
        return ops.quant_gemm_rowcol(st["x"], st["mats"])
    if k == "linear":
        return ops.gemm_rowcol(st["q"], st["s"], st["W"], st["scol"], bias=st["bias"], act=_ACT[case["act"]],
                               out=_OUT[case["out"]], out_scale=50.0 if case["out"] == "int8" else None)
    if k == "ksplit":
        return ops.gemm_rowcol_ksplit(st["q"], st["s"], st["W"], st["scol"])
    if k == "w4":
        return ops.gemm_w4(st["x"], st["Wp"], st["ws"], out=_OUT[case["out"]])
    if k == "attention":
        # the last query row sees every key, row m of the M rows nk - M + 1 + m of them
        return ops.attention(st["q"], st["kc"], st["vc"], case["heads"], case["kv_heads"],
                             causal_k=case["nk"] - case["M"] + 1, v_fp16=case["v_fp16"])
    x1 = ops.elt(ops.ELT_ADD, st["x"], st["o"])
    h = ops.rmsnorm_rows(x1, st["gamma"], None, 1e-6)
    q, s = ops.quant_rows(h)
    qr = ops.rope_rows(st["qp"], st["tab"], case["heads"], case["hd"])
    p = ops.elt(ops.ELT_MUL, st["gate"], st["up"], act=C.ACT_SILU)
    q2, s2 = ops.quant_rows(p)
    return {"sum": x1, "norm": h, "q": q, "s": s, "rope": qr, "prod": p, "q2": q2, "s2": s2}


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------------------ 64-bit references
def _silu64(x):
    return x / (1 + torch.exp(-x))


def _act64(x, act):
    if act == "relu":
        return x.clamp(min=0)
    if act == "gelu":
        return 0.5 * x * (1 + torch.tanh(0.79788456080286536 * (x + 0.044715 * x ** 3)))
    return _silu64(x) if act == "silu" else x


def _quant64(x):
    s = x.abs().amax(1) / 127
    return torch.round(x / s[:, None]).clamp(-127, 127), s


def _rms64(x, gamma):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-6) * gamma


def _rope64(x, tab, per):
    h = x.shape[1] // 2
    t = tab.double().repeat_interleave(per, 0)[:x.shape[0]]
    a, b, c, s = x[:, :h], x[:, h:], t[:, :h], t[:, h:]
    return torch.cat([a * c - b * s, b * c + a * s], 1)


def _attention64(q, kc, vc, heads, kv_heads, causal_k):
    M, nk = q.shape[0], kc.shape[0]
    hd, grp = q.shape[1] // heads, heads // kv_heads
    ok = torch.arange(nk, device="cuda")[None, :] < causal_k + torch.arange(M, device="cuda")[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        kv = slice((h // grp) * hd, (h // grp + 1) * hd)
        sc = q[:, h * hd:(h + 1) * hd].contiguous() @ kc[:, kv].t().contiguous()
        out[:, h * hd:(h + 1) * hd] = torch.softmax(sc.masked_fill(~ok, float("-inf")), 1) @ vc[:, kv].contiguous()
    return out


def exact(case, seed):
    st, k = prepare(case, seed), case["kind"]
    if k == "step":
        return _exact_step(case, st)
    if k == "group":
        q, s = _quant64(st["x"].double())
        return [q @ W.double().t().contiguous() * s[:, None] * sc.double()[None, :] for W, sc in st["mats"]]
    if k == "linear":
        y = st["q"].double() @ st["W"].double().t().contiguous() * st["s"].double()[:, None] * st["scol"].double()[None, :]
        y = _act64(y + (st["bias"].double()[None, :] if case["bias"] else 0), case["act"])
        return torch.round(y * 50.0).clamp(-127, 127) if case["out"] == "int8" else y
    if k == "ksplit":
        W = torch.cat([w.double() for w in st["W"]], 1)
        return st["q"].double() @ W.t().contiguous() * st["s"].double()[:, None] * st["scol"].double()[None, :]
    if k == "w4":
        w = torch.stack([st["Wp"] & 15, st["Wp"] >> 4], 2).reshape(case["N"], case["K"]).to(torch.int8)
        w = torch.where(w > 7, w - 16, w).double() * st["ws"].double().repeat_interleave(128, 1)
        return st["x"].double() @ w.t().contiguous()
    if k == "attention":
        return _attention64(st["q"].double(), st["kc"].double(), st["vc"].double(), case["heads"], case["kv_heads"],
                            case["nk"] - case["M"] + 1)
    x1 = st["x"].double() + st["o"].double()
    h = _rms64(x1, st["gamma"].double())
    q, s = _quant64(h)
    p = _silu64(st["gate"].double()) * st["up"].double()
    q2, s2 = _quant64(p)
    return {"sum": x1, "norm": h, "q": q, "s": s, "rope": _rope64(st["qp"].double(), st["tab"], case["heads"]),
            "prod": p, "q2": q2, "s2": s2}


# --------------------------------------------------------------------------------- whole passes
class _Image:
    """A decoder pass as a descriptor queue in one device image, as the reference's lowering emits it
    (tars_mini/llm.py:705-767, 614-640, 582-593): per layer RMSNorm, quantizer, q / k / v (v straight into
    its cache rows), per-head norms and RoPE (k into its cache rows), per-head scores / causal softmax /
    P V, quantizer, o, residual, RMSNorm, quantizer, gate (SiLU) / up, product in place, quantizer, down,
    residual; then the last row's RMSNorm, quantizer and head in up to 4 row blocks. Row scales are
    addressed in 16-byte units below 2^28, so weights lie last."""

    def __init__(self, case):
        c, R = case, case["rows"]
        H, heads, kv, hd, ff, t0 = c["H"], c["heads"], c["kv_heads"], c["hd"], c["ff"], c["t0"]
        self.descs, self.fills, self.top, self.big = [], [], 0, 0
        self.nk = nk = (t0 + R + 15) // 16 * 16
        hq, hk, kd = heads * hd, kv * hd, 4 * kv * hd // 16
        self.caches = self.take(4 * 2 * c["layers"] * nk * hk)
        self.tab = self.take(4 * hd * (t0 + R))
        x = self.x = self.take(4 * R * H)
        self.layers = []
        for l in range(c["layers"]):
            kc = self.caches + 4 * (2 * l) * nk * hk
            vc = kc + 4 * nk * hk
            w = {}
            n1, w["n1"] = self.norm(x, H, R)
            q1, s1 = self.quant(n1, H, R)
            qp, w["q"] = self.gemm(q1, s1, H, hq, R)
            kp, w["k"] = self.gemm(q1, s1, H, hk, R)
            _, w["v"] = self.gemm(q1, s1, H, hk, R, y=vc + 4 * t0 * hk)
            qn, w["qn"] = self.norm(qp, hd, R * heads, hd ** -0.5)  # the scores' scale, in the q norm's gamma
            qr = self.take(4 * R * hq)
            self.add(OPCODE=C.OP_ROPE, EPI=C.epi(), A_OFF=qn, W_OFF=self.tab + 4 * hd * t0, Y_OFF=qr, M=R * heads, N=hd,
                     K=hd, GROUP_SIZE=heads)
            kn, w["kn"] = self.norm(kp, hd, R * kv)
            self.add(OPCODE=C.OP_ROPE, EPI=C.epi(), A_OFF=kn, W_OFF=self.tab + 4 * hd * t0, Y_OFF=kc + 4 * t0 * hk,
                     M=R * kv, N=hd, K=hd, GROUP_SIZE=kv)
            sc, pr, att = self.take(4 * R * nk), self.take(4 * R * nk), self.take(4 * R * hq)
            wide = 4 * hq // 16 if R > 1 else 0  # one row: no stride
            for h in range(heads):
                j = h // (heads // kv)
                self.add(OPCODE=C.OP_FDOT, EPI=C.epi(), A_OFF=qr + 4 * h * hd, W_OFF=kc + 4 * j * hd, Y_OFF=sc, M=R,
                         N=nk, K=hd, LDA16=wide, GROUP_SIZE=kd)
                self.add(OPCODE=C.OP_ROW, CTRL=C.ROW_SOFTMAX, EPI=C.epi(), A_OFF=sc, Y_OFF=pr, M=R, N=nk, K=t0 + 1)
                self.add(OPCODE=C.OP_FDOT, CTRL=C.FDOT_NN, EPI=C.epi(), A_OFF=pr, W_OFF=vc + 4 * j * hd,
                         Y_OFF=att + 4 * h * hd, M=R, N=hd, K=nk, LDY16=wide, GROUP_SIZE=kd)
            qa, sa = self.quant(att, hq, R)
            o, w["o"] = self.gemm(qa, sa, hq, H, R)
            x1 = self.elt(C.ELT_ADD, x, o, R, H)
            n2, w["n2"] = self.norm(x1, H, R)
            q2, s2 = self.quant(n2, H, R)
            g, w["gate"] = self.gemm(q2, s2, H, ff, R, act=C.ACT_SILU)
            u, w["up"] = self.gemm(q2, s2, H, ff, R)
            self.elt(C.ELT_MUL, g, u, R, ff, y=g)
            q3, s3 = self.quant(g, ff, R)
            d, w["down"] = self.gemm(q3, s3, ff, H, R)
            x = self.elt(C.ELT_ADD, x1, d, R, H)
            self.layers.append(w)
        nf, self.nf = self.norm(x + 4 * (R - 1) * H, H, 1)
        qf, sf = self.quant(nf, H, 1)
        V = c["vocab"]
        self.head = (self.take_big(V * H), self.take(4 * V), V, H)
        self.fills.append(("w",) + self.head)
        self.logits = self.take(4 * V)
        blocks = 4 if V % 64 == 0 else 1
        for b in range(blocks):
            n, at = V // blocks, b * (V // blocks)
            self.add(OPCODE=C.OP_GEMM, CTRL=C.ctrl(C.QM_ROWCOL), EPI=C.epi(), A_OFF=qf, W_OFF=self.head[0] + at * H,
                     SCALE_OFF=self.head[1] + 4 * at, Y_OFF=self.logits + 4 * at, HDR_RSV=sf // 16, M=1, N=n, K=H)
        self.qaddr = self.take(64 * len(self.descs))
        self.base = (self.top + 4095) // 4096 * 4096
        self.size = self.base + self.big

    def take(self, n):
        at = (self.top + 255) // 256 * 256
        self.top = at + n
        return at

    def take_big(self, n):
        at = (self.big + 255) // 256 * 256
        self.big = at + n
        return at

    def add(self, **f):
        self.descs.append(dict(MAGIC=C.MAGIC, VERSION=C.VERSION, VALID=1, **f))

    def norm(self, x, n, rows, scale=1.0):
        g, y = self.take(4 * n), self.take(4 * n * rows)
        self.fills.append(("g", g, n, scale))
        self.add(OPCODE=C.OP_ROW, CTRL=C.ROW_RMSNORM, EPI=C.epi(), A_OFF=x, SCALE_OFF=g,
                 W_OFF=int(np.float32(1e-6).view(np.uint32)), Y_OFF=y, M=rows, N=n)
        return y, (g, n)

    def quant(self, x, k, rows):
        q, s = self.take(k * rows), self.take(max(16, 4 * rows))
        self.add(OPCODE=C.OP_ROW, CTRL=C.ROW_QUANT, EPI=C.epi(out=C.OUT_INT8), A_OFF=x, Y_OFF=q, SCALE_OFF=s, M=rows, N=k)
        return q, s

    def gemm(self, q, s, k, n, rows, act=0, y=None):
        m = (self.take_big(n * k), self.take(4 * n), n, k)
        self.fills.append(("w",) + m)
        y = self.take(4 * n * rows) if y is None else y
        self.add(OPCODE=C.OP_GEMM, CTRL=C.ctrl(C.QM_ROWCOL, fusion=int(act != 0)), EPI=C.epi(act), A_OFF=q, W_OFF=m[0],
                 SCALE_OFF=m[1], Y_OFF=y, HDR_RSV=s // 16, M=rows, N=n, K=k)
        return y, m

    def elt(self, op, a, b, rows, n, y=None):
        y = self.take(4 * rows * n) if y is None else y
        self.add(OPCODE=C.OP_ELT, CTRL=op, EPI=C.epi(), A_OFF=a, W_OFF=b, Y_OFF=y, M=rows, N=n)
        return y

    def queue(self):
        return b"".join(Q.encode_descriptor(dict(d, W_OFF=d["W_OFF"] + self.base) if d["OPCODE"] == C.OP_GEMM else d)
                        for d in self.descs)


def _prepare_step(case, g):
    im = _Image(case)
    image = torch.zeros(im.size, dtype=torch.uint8, device="cuda")
    f32 = lambda at, n: image[at:at + 4 * n].view(torch.float32)
    hk, nk, L = case["kv_heads"] * case["hd"], im.nk, case["layers"]
    caches = f32(im.caches, 2 * L * nk * hk).view(L, 2, nk, hk)
    caches[:, :, :case["t0"]] = torch.randn((L, 2, case["t0"], hk), device="cuda", generator=g)
    f32(im.tab, case["hd"] * (case["t0"] + case["rows"])).copy_(_rope_table(case["t0"] + case["rows"], case["hd"]).view(-1))
    f32(im.x, case["rows"] * case["H"]).copy_(_acts(g, case["rows"], case["H"]).view(-1))
    for f in im.fills:
        if f[0] == "g":
            f32(f[1], f[2]).copy_((1 + 0.1 * torch.randn(f[2], device="cuda", generator=g)) * f[3])
        else:
            _, w, s, n, k = f
            image[im.base + w:im.base + w + n * k].view(torch.int8).view(n, k).copy_(_int8(g, n, k))
            f32(s, n).copy_(_scol(g, n, k))
    raw = im.queue()
    image[im.qaddr:im.qaddr + len(raw)].copy_(torch.frombuffer(bytearray(raw), dtype=torch.uint8))
    return {"case": case, "image": im, "machine": Q.Machine(image), "qaddr": im.qaddr, "n": len(im.descs), "queue": raw,
            "logits": f32(im.logits, case["vocab"]), "caches": caches}


def _exact_step(case, st):
    im, image = st["image"], st["machine"].image
    f64 = lambda at, n: image[at:at + 4 * n].view(torch.float32).double()
    R, H, hd, t0 = case["rows"], case["H"], case["hd"], case["t0"]
    heads, kv = case["heads"], case["kv_heads"]

    def lin(x, m):
        w, s, n, k = m
        q, sr = _quant64(x)
        W = image[im.base + w:im.base + w + n * k].view(torch.int8).view(n, k).double()
        return (q @ W.t().contiguous()) * sr[:, None] * f64(s, n)[None, :]

    norm = lambda x, m: _rms64(x, f64(*m))
    tab = f64(im.tab, hd * (t0 + R)).view(t0 + R, hd)[t0:]
    caches = st["caches"].double()
    x = f64(im.x, R * H).view(R, H)
    for l, w in enumerate(im.layers):
        h = norm(x, w["n1"])
        q = _rope64(norm(lin(h, w["q"]).reshape(R * heads, hd), w["qn"]), tab, heads).reshape(R, heads * hd)
        caches[l, 0, t0:t0 + R] = _rope64(norm(lin(h, w["k"]).reshape(R * kv, hd), w["kn"]), tab, kv).reshape(R, kv * hd)
        caches[l, 1, t0:t0 + R] = lin(h, w["v"])
        x = x + lin(_attention64(q, caches[l, 0], caches[l, 1], heads, kv, t0 + 1), w["o"])
        h = norm(x, w["n2"])
        x = x + lin(_silu64(lin(h, w["gate"])) * lin(h, w["up"]), w["down"])
    return {"logits": lin(norm(x[R - 1:], im.nf), im.head).view(-1), "caches": caches}
