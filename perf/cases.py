"""The work whose speed is measured: the quantized linear layers as a program that serves a model calls them.

listed() names twelve cases, draw() gives more of the same ranges. A case's "path" says which operations a pass makes:

  linear     one weight matrix in GGML blocks times 1 to 16 tokens (vecq_fused for one token; quantize_q8_1, then vecq)
  ffn        a gated feed-forward layer in GGML blocks: gate and up with their GLU, then down, 1 to 16 tokens
  moe        a routed-expert feed-forward layer (moe_token for one token of Q4_K experts, else moe_ffn)
  mxfp8      a prompt chunk's activations quantized to MXFP8, then the block-scaled product
  exl3       an EXL3 trellis-coded linear: packed up to 144 rows, reconstructed above, its weights transformed from 1,024
  attention  a decode step over a quantized KV cache: the new K rows (rotated) and V rows stored, then attended
  stored     a weight in its stored encoding times F32 rows: decode_vector up to 16 rows, decode_matrix above
"""
import math

import torch

from llmp_amd import ops

TYPES = {"q8_0": ops.TYPE_Q8_0, "q4_k": ops.TYPE_Q4_K, "q5_k": ops.TYPE_Q5_K, "q6_k": ops.TYPE_Q6_K, "q4_0": ops.TYPE_Q4_0}
GLUS = {"swiglu": ops.GLU_SWIGLU, "geglu": ops.GLU_GEGLU}
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
CODEBOOKS = {"3inst": ops.EXL3_3INST, "mcg": ops.EXL3_MCG, "mul1": ops.EXL3_MUL1}
# A value's codes and scales, in bytes.
STORED_BYTES = {"bf16.dense": 2.0, "q8_0.blocks": 34.0 / 32.0, "nvfp4.split": 0.5 + 1.0 / 16.0, "mxfp8.split": 1.0 + 1.0 / 32.0,
                "mxfp4.split": 0.5 + 1.0 / 32.0}


def listed():
    return [
        # The smallest call: one token through an attention projection, where the launch and its latency are what counts.
        {"name": "q8_0_linear_1_token", "path": "linear", "type": "q8_0", "k": 4096, "n": 4096, "tokens": 1, "dtype": "f32"},
        # A decode step's feed-forward layer at batch 1 (hidden 3840, GeGLU): what a reply spends most of its time in.
        {"name": "q4_k_ffn_1_token", "path": "ffn", "type": "q4_k", "hidden": 3840, "ffn": 15360, "glu": "geglu", "tokens": 1, "dtype": "bf16"},
        # The same layer with six tokens: a few requests together, or drafted tokens being verified.
        {"name": "q4_k_ffn_6_tokens", "path": "ffn", "type": "q4_k", "hidden": 3840, "ffn": 15360, "glu": "geglu", "tokens": 6, "dtype": "f32"},
        # A prompt chunk of 2048 tokens against MXFP8 weights, activations quantized on the way: the largest dense product.
        {"name": "mxfp8_prefill_2048", "path": "mxfp8", "m": 2048, "k": 4096, "n": 12288, "dtype": "bf16"},
        # A routed-expert layer (128 experts, eight a token) at batch 1, at a small batch, and over a prompt chunk.
        {"name": "moe_q4_k_1_token", "path": "moe", "type": "q4_k", "hidden": 2048, "ffn": 768, "experts": 128, "used": 8, "tokens": 1},
        {"name": "moe_q4_k_16_tokens", "path": "moe", "type": "q4_k", "hidden": 2048, "ffn": 768, "experts": 128, "used": 8, "tokens": 16},
        {"name": "moe_q4_k_512_tokens", "path": "moe", "type": "q4_k", "hidden": 2048, "ffn": 768, "experts": 128, "used": 8, "tokens": 512},
        # An EXL3 linear at batch 1, over a short prompt of no round length, and over a prompt chunk.
        {"name": "exl3_linear_1_row", "path": "exl3", "k": 4096, "n": 14336, "bits": 4, "codebook": "3inst", "m": 1, "out": "f32"},
        {"name": "exl3_linear_77_rows", "path": "exl3", "k": 4096, "n": 14336, "bits": 4, "codebook": "3inst", "m": 77, "out": "f32"},
        {"name": "exl3_linear_2048_rows", "path": "exl3", "k": 4096, "n": 14336, "bits": 4, "codebook": "3inst", "m": 2048, "out": "f16"},
        # One token's attention over a Q8_0 cache of 8192 cells, its K and V rows stored first.
        {"name": "attention_q8_0_8192_cells", "path": "attention", "type": "q8_0", "head_dim": 256, "heads": 16, "kv_heads": 8, "rows": 1,
         "cells": 8192},
        # A prompt of no round length against NVFP4 weights as they are stored, on the matrix cores.
        {"name": "nvfp4_matrix_300_rows", "path": "stored", "decoder": "nvfp4.split", "k": 4096, "n": 14336, "rows": 300},
    ]


def _log(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _steps(rng, low, high, step):
    return _log(rng, low // step, high // step) * step


def draw(rng):
    path = rng.choice(["linear", "ffn", "moe", "mxfp8", "exl3", "attention", "stored"])
    if path == "linear":
        tokens = rng.choice([1, _log(rng, 2, 16)])
        return {"path": path, "type": rng.choice(["q8_0", "q4_k", "q5_k", "q6_k", "q4_0"]), "k": _steps(rng, 1024, 15360, 256),
                "n": _steps(rng, 512, 15360, 8), "tokens": tokens, "dtype": rng.choice(["f32", "bf16"]) if tokens == 1 else "f32"}
    if path == "ffn":
        tokens = rng.choice([1, _log(rng, 2, 16)])
        return {"path": path, "type": rng.choice(["q8_0", "q4_k", "q5_k", "q6_k", "q4_0"]), "hidden": _steps(rng, 1024, 4096, 256),
                "ffn": _steps(rng, 2048, 15360, 256), "glu": rng.choice(["swiglu", "geglu"]), "tokens": tokens,
                "dtype": rng.choice(["f32", "bf16"]) if tokens == 1 else "f32"}
    if path == "moe":
        return {"path": path, "type": rng.choice(["q4_k", "q8_0"]), "hidden": rng.choice([1024, 1536, 2048]), "ffn": rng.choice([512, 768]),
                "experts": rng.choice([32, 64, 128]), "used": rng.choice([4, 6, 8]), "tokens": rng.choice([1, _log(rng, 2, 512)])}
    if path == "mxfp8":
        return {"path": path, "m": _log(rng, 17, 2048), "k": _steps(rng, 1024, 4096, 128), "n": _steps(rng, 1024, 12288, 32),
                "dtype": rng.choice(["f32", "bf16"])}
    if path == "exl3":
        return {"path": path, "k": _steps(rng, 1024, 4096, 128), "n": _steps(rng, 1024, 14336, 128), "bits": rng.choice([2, 3, 4, 5, 6]),
                "codebook": rng.choice(["3inst", "mcg", "mul1"]), "m": rng.choice([_log(rng, 1, 144), _log(rng, 145, 2048)]),
                "out": rng.choice(["f32", "f16"])}
    if path == "attention":
        head_dim = rng.choice([64, 256])
        return {"path": path, "type": rng.choice(["q8_0", "q4_0"]), "head_dim": head_dim, "heads": 16, "kv_heads": rng.choice([2, 4, 8]),
                "rows": rng.choice([1, _log(rng, 2, 8)]), "cells": _steps(rng, 256, 32768, 256)}
    return {"path": path, "decoder": rng.choice(list(STORED_BYTES)), "k": _steps(rng, 1024, 4096, 256), "n": _steps(rng, 1024, 14336, 8),
            "rows": rng.choice([_log(rng, 1, 16), _log(rng, 17, 1024)])}


# ---------------------------------------------------------------- inputs


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=g)


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(shape, dtype=torch.float32, device="cuda", generator=g).to(dtype)


def _halves(values):
    """F16 values as the byte pairs they are stored as."""
    return values.to(torch.float16).contiguous().view(torch.uint8).view(*values.shape, 2)


def _blocks(t, n, k, g):
    """[n, a row's bytes] of blocks of type t: codes (and sub-block scales) uniform, scales such that the values have the
    range of weights drawn from N(0, 0.02)."""
    qk, size = ops.BLOCK_ELEMENTS[t], ops.BLOCK_BYTES[t]
    out = _bytes(g, n, k // qk, size)
    spread = torch.rand((n, k // qk, 2), device="cuda", generator=g) * 0.2 + 0.9
    peak = 0.02 * (5.6 if qk == 256 else 2.1)
    if t == ops.TYPE_Q6_K:
        out[:, :, 208:210] = _halves(spread[..., 0] * (peak / (127.0 * 32.0)))
    elif t in (ops.TYPE_Q4_K, ops.TYPE_Q5_K):
        levels = 15.0 if t == ops.TYPE_Q4_K else 31.0
        out[:, :, 0:2] = _halves(spread[..., 0] * (peak / (63.0 * levels)))
        out[:, :, 2:4] = _halves(spread[..., 1] * (0.5 * peak / 63.0))
    else:
        out[:, :, 0:2] = _halves(spread[..., 0] * (peak / (127.0 if t == ops.TYPE_Q8_0 else 8.0)))
    return out.view(n, -1)


def _stored(decoder, n, k, g):
    w = {"k": k}
    if decoder == "bf16.dense":
        w["data"] = _normal(g, n, k, dtype=torch.bfloat16).mul_(0.05).view(torch.uint8)
    elif decoder == "q8_0.blocks":
        w["data"] = _blocks(ops.TYPE_Q8_0, n, k, g)
    elif decoder == "nvfp4.split":
        w["data"] = _bytes(g, n, k // 2)
        w["scales"] = torch.randint(0x20, 0x48, (n * (k // 16),), dtype=torch.uint8, device="cuda", generator=g)
    elif decoder == "mxfp8.split":
        codes = _bytes(g, n, k)
        codes[(codes & 0x7F) == 0x7F] = 0x38  # no NaN codes
        w["data"] = codes
    else:
        w["data"] = _bytes(g, n, k // 2)
    if decoder in ("mxfp8.split", "mxfp4.split"):
        w["scales"] = torch.randint(118, 126, (n * (k // 32),), dtype=torch.uint8, device="cuda", generator=g)
    return w


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = dict(case)
    path = case["path"]
    if path == "linear":
        s["t"] = t = TYPES[case["type"]]
        s["w"] = _blocks(t, case["n"], case["k"], g)
        s["x"] = _normal(g, case["tokens"], case["k"], dtype=DTYPES[case["dtype"]])
    elif path == "ffn":
        s["t"] = t = TYPES[case["type"]]
        s["gate"], s["up"] = (_blocks(t, case["ffn"], case["hidden"], g) for _ in range(2))
        s["down"] = _blocks(t, case["hidden"], case["ffn"], g)
        s["x"] = _normal(g, case["tokens"], case["hidden"], dtype=DTYPES[case["dtype"]])
    elif path == "moe":
        s["t"] = t = TYPES[case["type"]]
        experts, hidden, ffn = case["experts"], case["hidden"], case["ffn"]
        s["gate_up"] = _blocks(t, experts * 2 * ffn, hidden, g).view(experts, -1)
        s["w_down"] = _blocks(t, experts * hidden, ffn, g).view(experts, -1)
        s["logits"] = _normal(g, case["tokens"], experts)
        s["x"] = _normal(g, case["tokens"], hidden)
        if case["tokens"] == 1 and t == ops.TYPE_Q4_K:
            s["token"] = ops.MoeTokenState(case["used"], ffn, s["x"].device)
    elif path == "mxfp8":
        s["w"] = ops.mxfp8_quantize(_normal(g, case["n"], case["k"]) * 0.02)
        s["x"] = _normal(g, case["m"], case["k"], dtype=DTYPES[case["dtype"]])
    elif path == "exl3":
        k, n = case["k"], case["n"]
        trellis = _bytes(g, (k // 16) * (n // 16) * 32 * case["bits"])
        suh = (torch.randint(0, 2, (k,), device="cuda", generator=g) * 2 - 1).to(torch.float16)
        signs = torch.randint(0, 2, (n,), device="cuda", generator=g) * 2 - 1
        svh = (signs * (1.0 + 0.1 * torch.randn((n,), device="cuda", generator=g)).abs()).to(torch.float16)
        s["linear"] = (trellis, suh, svh, k, n, case["bits"], CODEBOOKS[case["codebook"]])
        s["x"] = _normal(g, case["m"], k, dtype=torch.float16)
        if case["m"] > 144:  # the weights' scratch, kept from call to call: a slice of the columns at most
            s["scratch"] = torch.empty(2 * k * n, dtype=torch.uint8, device="cuda")
    elif path == "attention":
        s["t"] = t = TYPES[case["type"]]
        rows, cells, heads, kv, d = case["rows"], case["cells"], case["heads"], case["kv_heads"], case["head_dim"]
        row_bytes = kv * d // 32 * ops.BLOCK_BYTES[t]
        everywhere = torch.arange(cells, dtype=torch.int64, device="cuda")
        for name in ("k_cache", "v_cache"):
            s[name] = torch.empty((cells, row_bytes), dtype=torch.uint8, device="cuda")
            for at in range(0, cells, 8192):
                ids = everywhere[at:at + 8192].contiguous()
                ops.set_rows_quant(t, _normal(g, ids.numel(), kv * d), ids, s[name])
        filled = cells - 37  # the tokens so far, this pass's rows the last of them
        s["q"], s["k_new"], s["v_new"] = _normal(g, heads, rows, d), _normal(g, rows, kv, d), _normal(g, rows, kv * d)
        s["pos"] = torch.arange(filled - rows, filled, dtype=torch.int32, device="cuda")
        s["ids"] = s["pos"].to(torch.int64)
        s["mask"] = torch.zeros((rows, cells), dtype=torch.float16, device="cuda")
        s["mask"][everywhere.view(1, -1) > s["ids"].view(-1, 1)] = -math.inf
        s["theta_scale"] = 10000.0 ** (-2.0 / d)
    else:
        s["id"] = ops.DECODERS.index(case["decoder"])
        s["w"] = _stored(case["decoder"], case["n"], case["k"], g)
        s["x"] = _normal(g, case["rows"], case["k"])
    return s


# ---------------------------------------------------------------- a pass


def run(s):
    path = s["path"]
    if path == "linear":
        if s["tokens"] == 1:
            return ops.vecq_fused(s["t"], s["w"], s["x"], s["k"], s["n"])
        q8 = ops.quantize_q8_1(s["x"])
        return ops.vecq(s["t"], s["w"], q8, s["k"], s["n"], tokens=s["tokens"])
    if path == "ffn":
        t, hidden, ffn, tokens, glu = s["t"], s["hidden"], s["ffn"], s["tokens"], GLUS[s["glu"]]
        if tokens == 1:
            h = ops.vecq_fused(t, s["up"], s["x"], hidden, ffn, gate=s["gate"], glu=glu)
            return ops.vecq_fused(t, s["down"], h, ffn, hidden)
        h = ops.vecq(t, s["up"], ops.quantize_q8_1(s["x"]), hidden, ffn, gate=s["gate"], tokens=tokens, glu=glu)
        return ops.vecq(t, s["down"], ops.quantize_q8_1(h.view(tokens, ffn)), ffn, hidden, tokens=tokens)
    if path == "moe":
        sizes = (s["hidden"], s["ffn"], s["experts"], s["used"])
        if "token" in s:
            y = ops.moe_token(s["t"], s["logits"].view(-1), s["x"].view(-1), s["gate_up"], s["w_down"], *sizes, s["token"])
            return y, s["token"].ids, s["token"].weights
        return ops.moe_ffn(s["t"], s["logits"], s["x"], s["gate_up"], s["w_down"], *sizes)
    if path == "mxfp8":
        codes, scales = ops.mxfp8_quantize(s["x"])
        return ops.mxfp8_gemm(codes, scales, *s["w"])
    if path == "exl3":
        f32 = s["out"] == "f32"
        if s["m"] <= 144:
            return ops.exl3_linear(*s["linear"], s["x"], f32=f32)
        return ops.exl3_linear_reconstructed(*s["linear"], s["x"], f32=f32, fused=s["m"] >= 1024, w=s["scratch"])
    if path == "attention":
        t, d = s["t"], s["head_dim"]
        ops.rope_set_rows_quant(t, s["k_new"], s["pos"], s["ids"], s["k_cache"], d, s["theta_scale"])
        ops.set_rows_quant(t, s["v_new"], s["ids"], s["v_cache"])
        y = ops.attn_vec_quant(t, s["q"], s["k_cache"], s["v_cache"], s["mask"], d, s["heads"], s["kv_heads"], s["cells"], d ** -0.5)
        return y, s["k_cache"], s["v_cache"]
    if s["rows"] <= 16:
        return ops.decode_vector(s["id"], s["w"], s["x"])
    return ops.decode_matrix(s["id"], s["w"], s["x"])


# ---------------------------------------------------------------- what a pass cannot do without


def _weight_bytes(case, n, k):
    t = TYPES[case["type"]]
    return n * k * ops.BLOCK_BYTES[t] / ops.BLOCK_ELEMENTS[t]


def work(case):
    path = case["path"]
    if path == "linear":
        m, n, k = case["tokens"], case["n"], case["k"]
        return {"bytes": _weight_bytes(case, n, k) + m * (k * DTYPES[case["dtype"]].itemsize + n * 4), "flops": 2.0 * m * n * k}
    if path == "ffn":
        m, hidden, ffn = case["tokens"], case["hidden"], case["ffn"]
        return {"bytes": 3 * _weight_bytes(case, ffn, hidden) + m * hidden * (DTYPES[case["dtype"]].itemsize + 4),
                "flops": 6.0 * m * hidden * ffn}
    if path == "moe":
        m, hidden, ffn, experts, used = (case[name] for name in ("tokens", "hidden", "ffn", "experts", "used"))
        touched = experts * (1.0 - (1.0 - used / experts) ** m)  # the experts that m tokens' picks name, expected
        return {"bytes": touched * 3 * _weight_bytes(case, ffn, hidden) + m * (hidden * 8 + experts * 4 + used * 8),
                "flops": 6.0 * m * used * hidden * ffn}
    if path == "mxfp8":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k * 33.0 / 32.0 + m * (k * DTYPES[case["dtype"]].itemsize + n * 2), "flops": 2.0 * m * n * k}
    if path == "exl3":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k * case["bits"] / 8.0 + 2 * (n + k) + m * (k * 2 + n * DTYPES[case["out"]].itemsize), "flops": 2.0 * m * n * k}
    if path == "attention":
        rows, cells, heads, kv, d = case["rows"], case["cells"], case["heads"], case["kv_heads"], case["head_dim"]
        return {"bytes": 2 * _weight_bytes(case, cells, kv * d) + rows * (heads * d * 8 + cells * 2 + 2 * kv * d * 4),
                "flops": 4.0 * rows * cells * heads * d}
    m, n, k = case["rows"], case["n"], case["k"]
    return {"bytes": n * k * STORED_BYTES[case["decoder"]] + m * (k + n) * 4, "flops": 2.0 * m * n * k}


def tolerance(case):
    """About four times what was seen on the device: against F64 sums of the same decoded values, and where a stage's result is
    rounded on the way to the next (to Q8_1, F16 or bf16), with that result disturbed by the last bits of an F32 sum."""
    path = case["path"]
    if path == "linear":
        return {"rel": 1e-6}  # exact integer sums, F32 sums of their products with the scales: 1.7e-7
    if path == "ffn":
        return {"rel": 8e-4, "max": 1e-2}  # a code of h's that turns by one: 1.8e-4, one value 1.6e-3
    if path == "moe":
        return {"rel": 5e-4, "max": 2e-2}  # the same over shorter sums: 1.3e-4, one value 5.1e-3
    if path == "mxfp8":
        return {"rel": 1e-3, "max": 3e-2}  # the bf16 results' last bit: 2.3e-4, one value 7.8e-3
    if path == "exl3":
        # The transformed inputs' last F16 bit: 2.1e-4; reconstructed, the weights' in place of the inputs': 4.5e-4.
        return {"rel": 8e-4, "max": 5e-3} if case["m"] <= 144 else {"rel": 1.8e-3, "max": 1e-2}
    if path == "attention":
        return {"rel": 4e-6, "max": 2e-5}  # F32 sums of exact integer scores and decoded values: 1.0e-6, one value 3.3e-6
    return {"rel": 2e-6}  # F32 sums of exactly decoded (a matrix form's: rounded) values: 4.1e-7
