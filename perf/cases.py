"""The calls a user of this package makes most, as cases that can be timed and checked.

A case names one public entry point with its sizes, storage types and options. The sizes are the
ones the package is configured, tested and benchmarked with: the linears and attention of a
0.5B decoder (hidden 896, intermediate 4864, 14 q / 2 kv heads of 64), of a 1B decoder (hidden
2048, intermediate 8192, 32 q / 8 kv heads of 64) and of an 8B decoder (hidden 4096, intermediate
14336, 32 q / 8 kv heads of 128). `listed` holds twelve of them; `draw` takes others from the same
ranges.

Inputs are torch tensors on the GPU, made from the seed; the entry points get their addresses, as
they get any device pointer. Activations are normal, weights are normal with the standard deviation
0.02 that random-init decoders use (int8 rows quantized to +-127 with one fp16 scale per row, as the
package stores them), K and V rows are normal.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import l0llm_amd as l0

DTYPES = {"f32": (l0.F32, torch.float32, 4), "f16": (l0.F16, torch.float16, 2), "bf16": (l0.BF16, torch.bfloat16, 2),
          "i8": (l0.I8PC, torch.int8, 1)}
PRECISIONS = {"f32": l0.PRECISION_FLOAT32, "f16": l0.PRECISION_FLOAT16, "bf16": l0.PRECISION_BFLOAT16,
              "i8": l0.PRECISION_INT8}
# hidden, intermediate, layers, q heads, kv heads, head dim, vocab, q/k/v bias, RoPE theta
MODELS = {"0.5B": (896, 4864, 24, 14, 2, 64, 151936, True, 1e6),
          "1B": (2048, 8192, 16, 32, 8, 64, 128256, False, 5e5),
          "8B": (4096, 14336, 32, 32, 8, 128, 128256, False, 5e5)}
HEADS = [(32, 8, 128), (14, 2, 64), (32, 8, 64)]

_device = None


def _dev():
    global _device
    if _device is None:
        _device = l0.Device(0)
    return _device


def listed():
    return [
        # Decode, one token, the 0.5B MLP's up projection with 16-bit activations: the smallest call,
        # where the launch counts for more than the 4 MB it reads.
        dict(name="gemv_i8_896x4864", op="gemv", w="i8", rows=1, n=4864, k=896, x="f16", y="f16"),
        # Decode through the reference's own operator and layout (W as [K, N], fp32 activations):
        # the 0.5B down projection of an fp16 matrix.
        dict(name="kn_f16_4864x896", op="kn", w="f16", rows=1, n=896, k=4864),
        # A 14-token chat prompt: 13 rows with fp32 activations through an int8 8B projection.
        dict(name="rows13_i8_4096x14336", op="gemv", w="i8", rows=13, n=14336, k=4096, x="f32", y="f32"),
        # A question of some 40 tokens: its rows through the fp16 gate|up matrix of the 0.5B model.
        dict(name="rows40_f16_896x9728", op="gemv", w="f16", rows=40, n=9728, k=896, x="f32", y="f32"),
        # Prefill of 512 tokens, bf16 gate|up of the 1B model.
        dict(name="gemm_bf16_512x2048x16384", op="gemm", w="bf16", m=512, n=16384, k=2048, y="bf16"),
        # Prefill of a ragged 1000 tokens, int8 down projection of the 8B model.
        dict(name="gemm_i8_1000x14336x4096", op="gemm", w="i8", m=1000, n=4096, k=14336, y="f32"),
        # Batched decode: eight sequences of 4096 positions, 8B heads, fp16 cache.
        dict(name="attn_f16_b8_4096", op="attn", cache="f16", batch=8, heads=32, kv=8, dim=128, seq=4096, cap=4096, q="f16"),
        # Decode of one sequence with the reference's fp32 cache, 0.5B heads, a ragged length.
        dict(name="attn_f32_1000", op="attn", cache="f32", batch=1, heads=14, kv=2, dim=64, seq=1000, cap=2048, q="f32"),
        # Prefill attention of 2047 tokens, 8B heads, fp16 cache.
        dict(name="prefill_attn_f16_2047", op="prefill_attn", cache="f16", heads=32, kv=8, dim=128, pos=0, tokens=2047),
        # A second turn of 500 tokens behind 37 cached ones, 0.5B heads, the reference's fp32 cache.
        dict(name="prefill_attn_f32_37_500", op="prefill_attn", cache="f32", heads=14, kv=2, dim=64, pos=37, tokens=500),
        # A whole decode step of the 8B model behind a 2048-token prompt, int8 weights, fp16 cache.
        dict(name="decode_8b_i8_2048", op="decode", model="8B", w="i8", pos=2048),
        # A whole prefill of a 14-token chat prompt, 0.5B model, int8 weights, fp16 cache.
        dict(name="prefill_05b_i8_14", op="prefill", model="0.5B", w="i8", tokens=14),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of step between lo and hi, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng: random.Random):
    op = rng.choice(["gemv", "rows", "rows", "kn", "gemm", "gemm", "attn", "prefill_attn", "decode", "prefill"])
    if op == "gemv":  # decode linears: one row, any width of the models above
        w = rng.choice(["i8", "i8", "f16", "bf16"])
        x = rng.choice(["f32", "f16"])
        return dict(op="gemv", w=w, rows=1, n=_log(rng, 256, 40000, 4), k=_log(rng, 512, 14336, 32), x=x,
                    y=rng.choice(["f32", x]))
    if op == "rows":  # short prompts, several rows at once
        return dict(op="gemv", w=rng.choice(["i8", "i8", "f16", "bf16"]), rows=_log(rng, 2, 63), n=_log(rng, 512, 28672, 4),
                    k=_log(rng, 512, 14336, 32), x="f32", y="f32")
    if op == "kn":
        w = rng.choice(["f16", "f16", "f32"])
        return dict(op="kn", w=w, rows=_log(rng, 1, 8), n=_log(rng, 512, 16384, 8), k=_log(rng, 512, 8192))
    if op == "gemm":
        w = rng.choice(["bf16", "f16", "i8"])
        return dict(op="gemm", w=w, m=_log(rng, 64, 2048), n=_log(rng, 512, 16384, 4), k=_log(rng, 512, 14336, 32),
                    y=rng.choice(["f32", "f32", "f16" if w == "i8" else w]))
    if op == "attn":
        h, kv, d = rng.choice(HEADS)
        seq = _log(rng, 64, 16384)
        return dict(op="attn", cache=rng.choice(["f16", "f16", "f32"]), batch=rng.choice([1, 1, 2, 4, 8]), heads=h, kv=kv, dim=d,
                    seq=seq, cap=seq + rng.choice([0, 64, 1000]), q=rng.choice(["f32", "f16"]))
    if op == "prefill_attn":
        h, kv, d = rng.choice(HEADS)
        return dict(op="prefill_attn", cache=rng.choice(["f16", "f32"]), heads=h, kv=kv, dim=d, pos=rng.choice([0, _log(rng, 1, 1024)]),
                    tokens=_log(rng, 8, 2048))
    model, w = rng.choice(["0.5B", "1B"]), rng.choice(["i8", "i8", "f16", "bf16"])
    if op == "decode":
        return dict(op="decode", model=model, w=w, pos=_log(rng, 16, 2048))
    return dict(op="prefill", model=model, w=w, tokens=_log(rng, 2, 512))


# ------------------------------------------------------------------------------------ inputs --
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)


def _weights(g, kind, shape):
    """Weights as the package stores them, and their fp16 row scales where they are int8."""
    if kind != "i8":
        return _normal(g, shape, DTYPES[kind][1], 0.02), None
    w = _normal(g, shape, scale=0.02)
    s = (w.abs().amax(dim=1) / 127).half()
    return torch.clamp(torch.round(w / s.float()[:, None]), -127, 127).to(torch.int8), s


def _tensors(case, seed):
    """The input tensors of a single-operator case, by name."""
    g, op = _gen(seed), case["op"]
    if op in ("gemv", "kn", "gemm"):
        n, k = case["n"], case["k"]
        m = case["m"] if op == "gemm" else case["rows"]
        x = "f32" if op == "kn" else case["x"] if op == "gemv" else "f16" if case["w"] == "i8" else case["w"]
        w, s = _weights(g, case["w"], (k, n) if op == "kn" else (n, k))
        return dict(x=_normal(g, (m, k), DTYPES[x][1]), w=w, s=s)
    row = case["kv"] * case["dim"]
    kv = DTYPES[case["cache"]][1]
    if op == "attn":
        b, cap = case["batch"], case["cap"]
        return dict(q=_normal(g, (b, case["heads"] * case["dim"]), DTYPES[case["q"]][1]), k=_normal(g, (b, cap, row), kv),
                    v=_normal(g, (b, cap, row), kv))
    cap = case["pos"] + case["tokens"]
    return dict(q=_normal(g, (case["tokens"], case["heads"] * case["dim"])), k=_normal(g, (cap, row), kv), v=_normal(g, (cap, row), kv))


class _Model:
    """A model, the prompt behind it and the token to decode."""

    def __init__(self, case, seed):
        h, i, layers, nh, nkv, hd, vocab, bias, theta = MODELS[case["model"]]
        n = case["pos"] if case["op"] == "decode" else case["tokens"]
        self.ids = np.random.default_rng(seed).integers(0, vocab, n + 1, dtype=np.int32)
        cfg = l0.HfConfig(hidden_size=h, intermediate_size=i, num_layers=layers, num_attention_heads=nh, num_key_value_heads=nkv,
                          head_dim=hd, vocab_size=vocab, max_position_embeddings=32768, rms_norm_eps=1e-5, rope_theta=theta,
                          attention_bias=bias)
        self.model = l0.LlmModel(_dev(), cfg, precision=PRECISIONS[case["w"]], cache_dtype=l0.F16, max_seq_len=n + 128)
        self.model.init_random(int(seed), 0.02)
        if case["op"] == "decode":
            self.model.prefill(self.ids[:n])

    def __del__(self):
        if getattr(self, "model", None) is not None:
            self.model.dispose()


def prepare(case, seed):
    if case["op"] in ("decode", "prefill"):
        return dict(case=case, m=_Model(case, seed))
    st = dict(case=case, suite=l0.LlmKernelSuite(_dev()), **_tensors(case, seed))
    op = case["op"]
    if op in ("gemv", "kn", "gemm"):
        y = "f32" if op == "kn" else case["y"]
        st["out"] = torch.empty((st["x"].shape[0], case["n"]), dtype=DTYPES[y][1], device="cuda")
    else:
        st["out"] = torch.empty(st["q"].shape, dtype=st["q"].dtype, device="cuda")
    torch.cuda.synchronize()  # the inputs are made on torch's stream, the calls run on the device's own
    return st


def run(st):
    c = st["case"]
    op = c["op"]
    if op == "decode":
        return st["m"].model.compute_logits(int(st["m"].ids[-1]), c["pos"])
    if op == "prefill":
        return st["m"].model.prefill(st["m"].ids[: c["tokens"]])
    su, out = st["suite"], st["out"]
    o = out.data_ptr()
    if op == "attn":
        qd = DTYPES[c["q"]][0]
        if c["batch"] == 1 and c["q"] == "f32":  # the reference's Attention.Execute
            su.attention_execute(st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(), o, c["dim"], c["heads"], c["kv"], c["seq"],
                                 c["cap"], cache_dtype=DTYPES[c["cache"]][0])
        else:
            su.attention_decode(st["q"].data_ptr(), qd, st["k"].data_ptr(), st["v"].data_ptr(), DTYPES[c["cache"]][0], o, qd, c["batch"],
                                c["dim"], c["heads"], c["kv"], c["seq"], c["cap"])
        return out
    if op == "prefill_attn":
        su.attention_execute_prefill(st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(), o, c["dim"], c["heads"], c["kv"],
                                     c["pos"], c["tokens"], c["pos"] + c["tokens"], cache_dtype=DTYPES[c["cache"]][0])
        return out
    x, w = st["x"].data_ptr(), st["w"].data_ptr()
    if op == "kn":
        su.gemv_execute_rows(c["rows"], c["n"], c["k"], x, w, o, w_dtype=DTYPES[c["w"]][0])
    elif op == "gemv":
        s = None if st["s"] is None else st["s"].data_ptr()
        if c["w"] == "i8" and c["x"] == "f32" and c["y"] == "f32":  # the reference's GemvQ8.Execute / ExecuteRows
            su.gemv_q8_execute_rows(c["rows"], c["n"], c["k"], x, w, s, o)
        else:
            su.gemv_nk(DTYPES[c["w"]][0], c["rows"], c["n"], c["k"], x, DTYPES[c["x"]][0], w, s, o, DTYPES[c["y"]][0])
    elif c["w"] == "i8":
        su.gemm_nk_i8pc(c["m"], c["n"], c["k"], x, w, st["s"].data_ptr(), o, DTYPES[c["y"]][0])
    else:
        su.gemm_nk(DTYPES[c["w"]][0], c["m"], c["n"], c["k"], x, w, o, DTYPES[c["y"]][0])
    return out


# -------------------------------------------------------------------------------------- work --
def _model_work(case):
    """Every weight of the layers and the head once, the cache rows read and written, the logits."""
    h, i, layers, nh, nkv, hd, vocab, _, _ = MODELS[case["model"]]
    size = DTYPES[case["w"]][2]
    qd, kvd = nh * hd, nkv * hd
    rows_n = [qd + 2 * kvd, h, 2 * i, h]
    per_layer = (qd + 2 * kvd) * h + h * qd + 3 * h * i
    scales = 2 * sum(rows_n) if case["w"] == "i8" else 0
    head = vocab * h * size + (2 * vocab if case["w"] == "i8" else 0)
    if case["op"] == "decode":
        tokens, ctx = 1, case["pos"] + 1
        seen = ctx
    else:
        tokens = case["tokens"]
        ctx, seen = tokens, tokens * (tokens + 1) // 2
    cache = 2 * ctx * kvd * 2
    flops = layers * (2 * per_layer * tokens + 4 * seen * qd) + 2 * vocab * h
    return dict(bytes=layers * (per_layer * size + scales + cache) + head + 4 * vocab + 4 * h * tokens, flops=flops)


def work(case):
    op = case["op"]
    if op in ("decode", "prefill"):
        return _model_work(case)
    if op in ("gemv", "kn", "gemm"):
        n, k = case["n"], case["k"]
        m = case["m"] if op == "gemm" else case["rows"]
        xs = 4 if op == "kn" else DTYPES[case["x"]][2] if op == "gemv" else 2
        ys = 4 if op == "kn" else DTYPES[case["y"]][2]
        return dict(bytes=n * k * DTYPES[case["w"]][2] + (2 * n if case["w"] == "i8" else 0) + m * k * xs + m * n * ys, flops=2 * m * n * k)
    qd, kvd, cs = case["heads"] * case["dim"], case["kv"] * case["dim"], DTYPES[case["cache"]][2]
    if op == "attn":
        b = case["batch"]
        return dict(bytes=b * (2 * case["seq"] * kvd * cs + 2 * qd * DTYPES[case["q"]][2]), flops=4 * b * case["seq"] * qd)
    t, p = case["tokens"], case["pos"]
    return dict(bytes=2 * (p + t) * kvd * cs + 8 * t * qd, flops=4 * qd * (t * p + t * (t + 1) // 2))


def tolerance(case):
    """About four times what a correct computation in another order of the same precision shows."""
    op = case["op"]
    if op in ("decode", "prefill"):
        # 16 to 32 layers that hand a different rounding on: int8 and fp16 storage of the activations
        # between them moved the logits by 0.0003-0.0012 (0.0019 over the 8B model's 32), bf16 by 0.0034
        return {"rel": 1.4e-2 if case["w"] == "bf16" else 8e-3 if case["model"] == "8B" else 5e-3}
    out = case.get("y") if op in ("gemv", "gemm") else case["q"] if op == "attn" else "f32"
    if out == "bf16":
        return {"rel": 8e-3}
    if out == "f16":
        return {"rel": 1e-3}
    if op == "prefill_attn" and case["cache"] == "f16":
        return {"rel": 1e-3}  # the probabilities and the scaled q are 16-bit operands of the products
    return {"rel": 1e-5}


# ------------------------------------------------------------------------------------- exact --
def _attend(q, k, v, limit):
    """q [t, heads, d] over k, v [positions, kv, d] in 64 bits; query i sees positions 0 .. limit[i] - 1."""
    t, heads, d = q.shape
    group = heads // k.shape[1]
    out = torch.empty_like(q)
    at = torch.arange(k.shape[0], device=q.device)
    for h in range(heads):
        kh, vh = k[:, h // group].contiguous(), v[:, h // group].contiguous()
        s = q[:, h].contiguous() @ kh.t().contiguous() / math.sqrt(d)
        s = s.masked_fill(at[None, :] >= limit[:, None], -math.inf)
        out[:, h] = torch.softmax(s, dim=1) @ vh
    return out


def exact(case, seed):
    op = case["op"]
    if op in ("decode", "prefill"):
        return None  # the package's own generator makes the weights
    t = {n: None if v is None else v.double() for n, v in _tensors(case, seed).items()}
    if op in ("gemv", "gemm", "kn"):
        w = t["w"] if op == "kn" else t["w"].t().contiguous()
        y = t["x"] @ w
        return y if t["s"] is None else y * t["s"][None, :]
    h, kv, d = case["heads"], case["kv"], case["dim"]
    if op == "attn":
        seq, b = case["seq"], case["batch"]
        one = torch.full((1,), seq, device="cuda")
        out = [_attend(t["q"][i].view(1, h, d), t["k"][i, :seq].view(seq, kv, d), t["v"][i, :seq].view(seq, kv, d), one) for i in range(b)]
        return torch.stack(out).view(b, h * d)
    n, cap = case["tokens"], case["pos"] + case["tokens"]
    limit = torch.arange(n, device="cuda") + case["pos"] + 1
    return _attend(t["q"].view(n, h, d), t["k"].view(cap, kv, d), t["v"].view(cap, kv, d), limit).view(n, h * d)
