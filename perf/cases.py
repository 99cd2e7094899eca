"""The work this library is measured on: one call, or one transformer block's
projections, through the public operators, over the sizes a program uses them at.

A case is a dict of plain values whose "op" names the family:

  quant   the four weight-only projections of one transformer block (qkv, o,
          gate + up, down) on M tokens, int4 (groups of 128) or int8 weights:
          M = 1 decoding, tens of rows batched decoding, hundreds and up prefill
  linear  nn.Linear with dense 16-bit weights and an optional bias
  matmul  C = A @ B row-major: fp16, bf16, fp32 and FP8 inputs
  dot     the general tl.dot: transposed operands, batches, epilogues
  flash   attention forward (prefill), causal or not, any head dim and length
  decode  one query token per sequence over a contiguous or paged KV cache
  kda     Kimi Delta Attention, chunked (prefill)
  kdastep Kimi Delta Attention, one token per sequence with its state in place
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "triton-metal_amd"))

import triton_metal_amd as tm  # noqa: E402

DT = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32,
      "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
SIZE = {"fp16": 2, "bf16": 2, "fp32": 4, "e4m3": 1, "e5m2": 1}
GROUP = 128
DEV = "cuda"


def listed():
    return [
        # one token of an 8B model's block (32 query / 8 KV heads, FFN 14336), int4
        # with fp16 zero-points: decoding, the path this library puts first
        {"name": "int4_block_decode", "op": "quant", "bits": 4, "M": 1, "hidden": 4096,
         "kv": 1024, "ffn": 14336, "dtype": "fp16", "zeros": "act"},
        # a 7B model's block (FFN 11008) on a 1000-token prompt, GPTQ zero-points
        {"name": "int4_block_prefill", "op": "quant", "bits": 4, "M": 1000, "hidden": 4096,
         "kv": 4096, "ffn": 11008, "dtype": "fp16", "zeros": "u8"},
        # the same block in int8 for 16 sequences decoding together, bf16
        {"name": "int8_block_batch", "op": "quant", "bits": 8, "M": 16, "hidden": 4096,
         "kv": 4096, "ffn": 11008, "dtype": "bf16", "zeros": "none"},
        # an unquantised up projection on 2000 tokens
        {"name": "linear_prefill", "op": "linear", "M": 2000, "N": 11008, "K": 4096,
         "dtype": "bf16", "bias": True},
        # the smallest: 512^3, a call that launch and latency decide
        {"name": "matmul_512", "op": "matmul", "M": 512, "N": 512, "K": 512, "dtype": "fp16"},
        # FP8 activations and weights, fp32 out
        {"name": "matmul_fp8", "op": "matmul", "M": 2048, "N": 4096, "K": 4096,
         "dtype": "e4m3"},
        # a weight gradient added to the accumulated one: dW = X^T dY + dW0
        {"name": "dot_weight_grad", "op": "dot", "batch": 1, "M": 4096, "N": 4096, "K": 2000,
         "dtype": "bf16", "a_cols": True, "b_cols": False, "epilogue": "add-matrix",
         "out": "fp32"},
        # a long causal prefill, four sequences of 32 heads: the largest
        {"name": "flash_causal", "op": "flash", "B": 4, "H": 32, "S": 4096, "D": 128,
         "causal": True, "dtype": "bf16", "rows": "bhsd", "lse": True},
        # an encoder batch of ragged length: no mask, head dim 64, [B, S, H, D] tensors
        {"name": "flash_encoder", "op": "flash", "B": 8, "H": 16, "S": 1500, "D": 64,
         "causal": False, "dtype": "fp16", "rows": "bshd", "lse": False},
        # 16 sequences of mixed length over a paged fp16 cache, grouped-query heads
        {"name": "decode_paged", "op": "decode", "B": 16, "Hq": 32, "Hkv": 8, "D": 128,
         "S": 8192, "page": 16, "dtype": "fp16"},
        # a KDA layer's prefill of 8192 tokens
        {"name": "kda_prefill", "op": "kda", "B": 1, "T": 8192, "H": 16, "state": True},
        # and one token of it for 16 sequences
        {"name": "kda_decode", "op": "kdastep", "B": 16, "T": 1, "H": 16},
    ]


# ---- drawn cases --------------------------------------------------------------
def _log(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, step * round(v / step))))


def draw(rng):
    op = rng.choice(("quant", "quant", "linear", "matmul", "dot", "flash", "decode", "kda",
                     "kdastep"))
    if op == "quant":
        c = {"op": op, "bits": rng.choice((4, 4, 8)), "M": _log(rng, 1, 1000),
             "hidden": _log(rng, 1024, 5120, 256), "dtype": rng.choice(("fp16", "bf16")),
             "zeros": rng.choice(("act", "u8", "none"))}
        c["kv"] = c["hidden"] // rng.choice((1, 2, 4))
        c["ffn"] = 128 * round(c["hidden"] * rng.uniform(2.0, 3.5) / 128)
        if c["bits"] == 8:
            c["zeros"] = "none"
        return c
    if op == "linear":
        # any token count; features are multiples of 8, vocabularies any number
        c = {"op": op, "M": _log(rng, 1, 4096), "K": _log(rng, 512, 8192, 8),
             "N": _log(rng, 512, 16384, rng.choice((1, 8, 64))),
             "dtype": rng.choice(("fp16", "bf16")), "bias": rng.random() < 0.5}
        while c["M"] * c["N"] * c["K"] > 100e9:
            c["M"] = c["M"] // 2 + 1
        return c
    if op == "matmul":
        dt = rng.choice(("fp16", "bf16", "fp32", "e4m3", "e5m2"))
        step = rng.choice((1, 8, 16, 128))
        c = {"op": op, "M": _log(rng, 128, 4096, step), "N": _log(rng, 128, 4096, step),
             "K": _log(rng, 128, 4096, step), "dtype": dt}
        while c["M"] * c["N"] * c["K"] > (16e9 if dt == "fp32" or step == 1 else 70e9):
            c["M"] = step * max(1, c["M"] // 2 // step)
        return c
    if op == "dot":
        epi = rng.choice(("none", "none", "add-matrix", "add-rows", "add-cols", "softmax",
                          "chain-dot"))
        wide = epi in ("softmax", "chain-dot")
        c = {"op": op, "batch": _log(rng, 1, 16), "M": _log(rng, 64, 4096, 8),
             "N": _log(rng, 64, 2048 if wide else 4096, 8),
             "K": _log(rng, 32, 128 if wide else 4096, 8), "dtype": rng.choice(("fp16", "bf16")),
             "a_cols": rng.random() < 0.4, "b_cols": rng.random() < 0.4, "epilogue": epi}
        c["out"] = rng.choice((c["dtype"], "fp32"))
        while c["batch"] * c["M"] * c["N"] * c["K"] > (0.5e9 if wide else 34e9):
            c["batch" if c["batch"] > 1 else "M"] //= 2
        return c
    if op == "flash":
        c = {"op": op, "B": _log(rng, 1, 8), "H": rng.choice((8, 12, 16, 32)),
             "S": _log(rng, 128, 8192), "D": rng.choice((64, 64, 80, 96, 128, 128, 128)),
             "causal": rng.random() < 0.6, "dtype": rng.choice(("fp16", "bf16")),
             "rows": rng.choice(("bhsd", "bshd")), "lse": rng.random() < 0.5}
        while c["B"] * c["H"] * c["S"] ** 2 * c["D"] > 1.3e11:
            c["B" if c["B"] > 1 else "S"] //= 2
        return c
    if op == "decode":
        c = {"op": op, "B": _log(rng, 1, 64), "Hkv": rng.choice((4, 8, 16)),
             "D": rng.choice((64, 80, 96, 128, 128, 128)), "S": _log(rng, 256, 32768),
             "page": rng.choice((0, 16, 16, 64)), "dtype": rng.choice(("fp16", "bf16"))}
        c["Hq"] = c["Hkv"] * rng.choice((1, 4, 8))
        while c["B"] * c["Hkv"] * c["D"] * c["S"] > 150e6:
            c["B" if c["B"] > 1 else "S"] //= 2
        return c
    if op == "kda":
        c = {"op": op, "B": _log(rng, 1, 4), "T": _log(rng, 64, 8192), "H": _log(rng, 4, 32),
             "state": rng.random() < 0.5}
        while c["B"] * c["T"] * c["H"] > 140000:
            c["T"] //= 2
        return c
    return {"op": op, "B": _log(rng, 1, 64), "T": rng.choice((1, 1, 1, 2, 4)),
            "H": rng.choice((8, 16, 32))}


# ---- inputs -------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, device=DEV, generator=g).to(dtype)


def _projections(c):
    """(name, out features, in features) of the block's four projections."""
    h, f = c["hidden"], c["ffn"]
    return [("qkv", h + 2 * c["kv"], h), ("o", h, h), ("gate_up", 2 * f, h), ("down", h, f)]


def _quant_inputs(c, seed):
    g, M, dt = _gen(seed), c["M"], DT[c["dtype"]]
    out = []
    for name, N, K in _projections(c):
        x = _randn(g, M, K, dtype=dt)
        cols = K // GROUP if c["bits"] == 4 else 1
        # weights of standard deviation about 1 / sqrt(K), as trained layers have
        if c["bits"] == 4:
            w = torch.randint(0, 256, (N, K // 2), device=DEV, dtype=torch.uint8, generator=g)
            unit = 1 / (4.6 * math.sqrt(K))
        else:
            w = torch.randint(-127, 128, (N, K), device=DEV, dtype=torch.int8, generator=g)
            unit = 1 / (73 * math.sqrt(K))
        s = ((0.5 + torch.rand(N, cols, device=DEV, generator=g)) * unit).to(dt)
        z = None
        if c["zeros"] != "none":
            z = torch.randint(5, 11, (N, cols), device=DEV, generator=g)
            z = z.to(torch.uint8 if c["zeros"] == "u8" else dt)
        if c["bits"] == 8:
            s = s.reshape(N)
        out.append((name, N, K, x, w, s, z))
    return out


def _dot_inputs(c, seed):
    g, dt = _gen(seed), DT[c["dtype"]]
    b, M, N, K = c["batch"], c["M"], c["N"], c["K"]
    lead = (b,) if b > 1 else ()

    def operand(rows, cols, by_cols):
        if by_cols:  # column-major: stored [cols, rows]
            return _randn(g, *lead, cols, rows, dtype=dt).transpose(-1, -2)
        return _randn(g, *lead, rows, cols, dtype=dt)

    A, B = operand(M, K, c["a_cols"]), operand(K, N, c["b_cols"])
    if c["epilogue"] == "softmax":
        A = A * (K ** -0.5)  # scores of unit variance
    z = w = None
    if c["epilogue"].startswith("add-"):
        shape = {"add-matrix": (M, N), "add-rows": (M, 1), "add-cols": (1, N)}[c["epilogue"]]
        z = _randn(g, *lead, *shape, dtype=DT[c["out"]])
    if c["epilogue"] == "chain-dot":
        w = _randn(g, N, K, dtype=dt)
    cols = K if c["epilogue"] == "chain-dot" else N
    return A, B, z, w, lead + (M, cols)


def _qkv_inputs(c, seed):
    g, dt = _gen(seed), DT[c["dtype"]]
    B, H, S, D = c["B"], c["H"], c["S"], c["D"]
    if c["rows"] == "bshd":
        return [_randn(g, B, S, H, D, dtype=dt).transpose(1, 2) for _ in range(3)]
    return [_randn(g, B, H, S, D, dtype=dt) for _ in range(3)]


def _lengths(c):
    """Positions per sequence: from a quarter of the capacity to all of it."""
    B, S = c["B"], c["S"]
    return [max(1, S // 4 + (S - S // 4) * (i + 1) // B) for i in range(B)]


def _cache_inputs(c, seed):
    g, dt = _gen(seed), DT[c["dtype"]]
    B, Hq, Hkv, D, S, page = (c[k] for k in ("B", "Hq", "Hkv", "D", "S", "page"))
    q = _randn(g, B, Hq, D, dtype=dt)
    lens = torch.tensor(_lengths(c), device=DEV, dtype=torch.int32)
    lens = lens[torch.randperm(B, device=DEV, generator=g)].contiguous()
    if not page:
        return q, _randn(g, B, Hkv, S, D, dtype=dt), _randn(g, B, Hkv, S, D, dtype=dt), lens, None
    per = -(-S // page)
    kc, vc = (_randn(g, B * per, page, Hkv, D, dtype=dt) for _ in range(2))
    table = torch.randperm(B * per, device=DEV, generator=g).int().reshape(B, per)
    return q, kc, vc, lens, table


def _kda_inputs(c, seed):
    g = _gen(seed)
    B, T, H, D = c["B"], c["T"], c["H"], 128
    q, k = (torch.nn.functional.normalize(_randn(g, B, T, H, D), dim=-1).bfloat16()
            for _ in range(2))
    v = _randn(g, B, T, H, D, dtype=torch.bfloat16)
    beta = torch.sigmoid(_randn(g, B, T, H))
    gate = -torch.nn.functional.softplus(_randn(g, B, T, H, D))
    state = 0.1 * _randn(g, B, H, D, D) if c.get("state", True) else None
    return q, k, v, gate, beta, state


def _matmul_inputs(c, seed):
    g, dt = _gen(seed), DT[c["dtype"]]
    return _randn(g, c["M"], c["K"]).to(dt), _randn(g, c["K"], c["N"]).to(dt)


def _linear_inputs(c, seed):
    g, dt = _gen(seed), DT[c["dtype"]]
    x = _randn(g, c["M"], c["K"], dtype=dt)
    w = (_randn(g, c["N"], c["K"]) * c["K"] ** -0.5).to(dt)
    return x, w, _randn(g, c["N"], dtype=dt) if c["bias"] else None


def _out_dtype(c):
    """FP8 products are written in fp32, the others in their inputs' dtype."""
    return torch.float32 if SIZE[c["dtype"]] == 1 else DT[c["dtype"]]


def prepare(case, seed):
    c, op = case, case["op"]
    if op == "quant":
        launches, outs, keep = [], {}, []
        for name, N, K, x, w, s, z in _quant_inputs(c, seed):
            y = torch.empty(c["M"], N, device=DEV, dtype=x.dtype)
            if c["bits"] == 4:
                launches.append(tm.plan_int4_matmul(x, w, y, s, z, c["M"], N, K, GROUP))
            else:
                launches.append(tm.plan_int8_matmul(x, w, y, s, z, c["M"], N, K))
            outs[name] = y
            keep += [x, w, s, z]
        return {"op": op, "launches": launches, "out": outs, "keep": keep}
    if op == "linear":
        x, w, b = _linear_inputs(c, seed)
        y = torch.empty(c["M"], c["N"], device=DEV, dtype=x.dtype)
        return {"op": op, "args": (x, w, y, b, c["M"], c["N"], c["K"])}
    if op == "matmul":
        A, B = _matmul_inputs(c, seed)
        C = torch.empty(c["M"], c["N"], device=DEV, dtype=_out_dtype(c))
        return {"op": op, "launches": [tm.plan_matmul(A, B, C, c["M"], c["N"], c["K"])],
                "out": C, "keep": (A, B)}
    if op == "dot":
        A, B, z, w, shape = _dot_inputs(c, seed)
        C = torch.empty(shape, device=DEV, dtype=DT[c["out"]])
        return {"op": op, "launches": [tm.plan_dot(A, B, C, c["epilogue"], z=z, w=w)],
                "out": C, "keep": (A, B, z, w)}
    if op == "flash":
        q, k, v = _qkv_inputs(c, seed)
        o = torch.empty_like(q)
        lse = (torch.empty(c["B"], c["H"], c["S"], device=DEV) if c["lse"] else None)
        plan = tm.plan_flash_attention(q, k, v, o, lse, causal=c["causal"])
        return {"op": op, "launches": [plan], "out": (o, lse) if c["lse"] else o,
                "keep": (q, k, v)}
    if op == "decode":
        q, kc, vc, lens, table = _cache_inputs(c, seed)
        o = torch.empty_like(q)
        plan = tm.plan_decode_attention(q, kc, vc, o, seq_lens=lens, seq_len=c["S"],
                                        page_table=table)
        return {"op": op, "launches": [plan], "out": o, "keep": (q, kc, vc, lens, table)}
    q, k, v, gate, beta, state = _kda_inputs(c, seed)
    o = torch.empty_like(v)
    if op == "kda":
        final = torch.empty(c["B"], c["H"], 128, 128, device=DEV)
        plan = tm.plan_chunk_kda(q, k, v, gate, beta, o, initial_state=state, final_state=final)
        keep = (q, k, v, gate, beta, state)
    else:  # the state is updated in place, as a decoding loop does
        final = state
        plan = tm.plan_fused_recurrent_kda(q, k, v, gate, beta, o, initial_state=state,
                                           final_state=state)
        keep = (q, k, v, gate, beta)
    return {"op": op, "launches": [plan], "out": (o, final), "keep": keep}


def run(state):
    if state["op"] == "linear":
        return tm.fused_linear(*state["args"])
    for launch in state["launches"]:
        launch()
    return state["out"]


# ---- work and tolerance ---------------------------------------------------------
def work(case):
    c, op = case, case["op"]
    if op == "quant":
        nbytes = flops = 0
        zb = {"act": 2, "u8": 1, "none": 0}[c["zeros"]]
        for _, N, K in _projections(c):
            groups = K // GROUP if c["bits"] == 4 else 1
            nbytes += N * K * c["bits"] // 8 + (2 + zb) * N * groups + 2 * c["M"] * (K + N)
            flops += 2 * c["M"] * N * K
        return {"bytes": nbytes, "flops": flops}
    if op in ("linear", "matmul"):
        M, N, K, e = c["M"], c["N"], c["K"], SIZE[c["dtype"]]
        o = 4 if e == 1 else e
        return {"bytes": e * (M * K + K * N) + o * M * N + (e * N if c.get("bias") else 0),
                "flops": 2 * M * N * K}
    if op == "dot":
        b, M, N, K, e, o = c["batch"], c["M"], c["N"], c["K"], SIZE[c["dtype"]], SIZE[c["out"]]
        cols = K if c["epilogue"] == "chain-dot" else N
        nbytes = b * (e * (M * K + K * N) + o * M * cols)
        nbytes += {"add-matrix": o * b * M * N, "add-rows": o * b * M, "add-cols": o * b * N,
                   "chain-dot": e * N * K}.get(c["epilogue"], 0)
        return {"bytes": nbytes,
                "flops": 2 * b * M * N * K * (2 if c["epilogue"] == "chain-dot" else 1)}
    if op == "flash":
        B, H, S, D = c["B"], c["H"], c["S"], c["D"]
        return {"bytes": 8 * B * H * S * D + (4 * B * H * S if c["lse"] else 0),
                "flops": 4 * B * H * D * (S * (S + 1) // 2 if c["causal"] else S * S)}
    if op == "decode":
        n = sum(_lengths(c))
        return {"bytes": 4 * n * c["Hkv"] * c["D"] + 4 * c["B"] * c["Hq"] * c["D"],
                "flops": 4 * n * c["Hq"] * c["D"]}
    B, T, H, D = c["B"], c["T"], c["H"], 128
    nbytes = B * T * H * (8 * D + 4 * D + 4) + 4 * B * H * D * D
    if c.get("state", True):
        nbytes += 4 * B * H * D * D
    return {"bytes": nbytes, "flops": 6 * B * T * H * D * D}


def tolerance(case):
    """About four times the distance from the 64-bit result: half a unit in the
    last place of the output (relative, root mean square: 2e-4 in fp16, 1.7e-3 in
    bf16), with the operands that the path itself rounds to 16 bits on top (the
    dequantised weights of wide int4 products, attention's probabilities, KDA's
    per-chunk matrices); sums in fp32 where the output is fp32."""
    c, op = case, case["op"]
    if op in ("kda", "kdastep"):
        return {"rel": 0.02, "max": 0.6} if op == "kda" else {"rel": 0.008, "max": 0.05}
    if op in ("flash", "decode"):
        return {"rel": 0.012 if c["dtype"] == "bf16" else 0.0016, "max": 0.4}
    if op == "dot" and c["epilogue"] == "softmax":
        return {"rel": 1e-5 if c["out"] == "fp32" else 0.008 if c["out"] == "bf16" else 0.001}
    out = c["out"] if op == "dot" else "fp32" if SIZE[c["dtype"]] == 1 else c["dtype"]
    if out == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    if op == "quant" and c["dtype"] == "fp16":
        return {"rel": 0.0016, "max": 0.02}
    return {"rel": 0.008 if out == "bf16" else 0.001, "max": 0.02}


# ---- the same in 64 bits ----------------------------------------------------------
def _exact_kda(q, k, v, gate, beta, state, scale):
    B, T, H, D = q.shape
    q, k, v, beta, decay = (t.double() for t in (q, k, v, beta, gate.double().exp()))
    S = torch.zeros(B, H, D, D, device=DEV, dtype=torch.float64)
    if state is not None:
        S += state.double()
    o = torch.empty(B, T, H, D, device=DEV, dtype=torch.float64)
    for t in range(T):
        S *= decay[:, t].unsqueeze(-1)
        kt = k[:, t].unsqueeze(-1)
        u = (v[:, t] - (S * kt).sum(-2)) * beta[:, t].unsqueeze(-1)
        S += kt * u.unsqueeze(-2)
        o[:, t] = scale * (S * q[:, t].unsqueeze(-1)).sum(-2)
    return o, S


def exact(case, seed):
    c, op = case, case["op"]
    if op == "quant":
        out = {}
        for name, N, K, x, w, s, z in _quant_inputs(c, seed):
            y = torch.empty(c["M"], N, device=DEV, dtype=torch.float64)
            for n in range(0, N, 4096):  # in blocks of output features
                if c["bits"] == 4:
                    wb = w[n:n + 4096]
                    q = torch.stack((wb & 15, wb >> 4), -1).reshape(wb.shape[0], K).double()
                    sb = s[n:n + 4096].double().repeat_interleave(GROUP, 1)
                    if z is not None:
                        q -= z[n:n + 4096].double().repeat_interleave(GROUP, 1)
                else:
                    q = w[n:n + 4096].double()
                    sb = s[n:n + 4096].double().unsqueeze(1)
                y[:, n:n + 4096] = x.double() @ (q * sb).t()
            out[name] = y
        return out
    if op == "linear":
        x, w, b = _linear_inputs(c, seed)
        y = x.double() @ w.double().t()
        return y if b is None else y + b.double()
    if op == "matmul":
        A, B = _matmul_inputs(c, seed)
        return A.double() @ B.double()
    if op == "dot":
        A, B, z, w, _ = _dot_inputs(c, seed)
        P = A.double().contiguous() @ B.double().contiguous()
        if z is not None:
            P = P + z.double()
        if c["epilogue"] == "softmax":
            return torch.softmax(P, -1)
        return P @ w.double() if w is not None else P
    if op == "flash":
        q, k, v = _qkv_inputs(c, seed)
        B, H, S, D = q.shape
        o = torch.empty(B, H, S, D, device=DEV, dtype=torch.float64)
        lse = torch.empty(B, H, S, device=DEV, dtype=torch.float64)
        future = torch.ones(S, S, device=DEV, dtype=torch.bool).triu(1) if c["causal"] else None
        for b in range(B):
            for h in range(H):
                p = (q[b, h].double() @ k[b, h].double().t().contiguous()) * D ** -0.5
                if future is not None:
                    p.masked_fill_(future, -math.inf)
                lse[b, h] = torch.logsumexp(p, -1)
                o[b, h] = torch.exp(p - lse[b, h].unsqueeze(-1)) @ v[b, h].double()
        return (o, lse) if c["lse"] else o
    if op == "decode":
        q, kc, vc, lens, table = _cache_inputs(c, seed)
        rep = c["Hq"] // c["Hkv"]
        o = torch.empty(q.shape, device=DEV, dtype=torch.float64)
        for b, n in enumerate(lens.tolist()):
            if table is None:
                k, v = kc[b, :, :n].double(), vc[b, :, :n].double()
            else:
                k, v = (t[table[b].long()].reshape(-1, c["Hkv"], c["D"])[:n].transpose(0, 1)
                        .double() for t in (kc, vc))
            qb = q[b].double().reshape(c["Hkv"], rep, c["D"])
            p = torch.softmax((qb.unsqueeze(2) * k.unsqueeze(1)).sum(-1) * c["D"] ** -0.5, -1)
            o[b] = (p @ v.contiguous()).reshape(c["Hq"], c["D"])
        return o
    q, k, v, gate, beta, state = _kda_inputs(c, seed)
    return _exact_kda(q, k, v, gate, beta, state, 128 ** -0.5)
