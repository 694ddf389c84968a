"""The work a user of this backend has it do, as cases to be timed and compared.

Every case goes through the public entry points of `yule_amd.backend`
(`HipBackend`, `HipRunner`).  `listed()` names the cases, `draw(rng)` gives
another one of the same ranges, `prepare(case, seed)` makes what a program has
in hand before the call (weights laid out on the device, activations, caches,
a runner), `run(state)` is one pass, `exact(case, seed)` the same result in 64
bits from plain torch.

Kinds of work:
  matvec       one quantized_matmul (decode, batch 1)
  projections  the four projection launches of a decoder layer (Q/K/V, O,
               gate/up, down), every one a quantized_matmul(_multi)
  head         lm_head matvec and the greedy pick over its logits
  attention    gqa_decode_attn of one token over a KV cache
  heads        the same attention as the trait has it, head by head:
               attn_score, softmax, attn_value
  block        one decoder layer of a decode step, op by op through the trait
  gemm         a prompt's projection: quantized_gemm, _f32 or _noalloc
  prefill      HipRunner.prefill_batched of a prompt (in one or more pieces)
  decode       HipRunner.generate_greedy from a prompt, then one decode_step
"""
from __future__ import annotations

import math

import numpy as np
import torch

from yule_amd import DType, GEOMETRY, matrix_bytes, row_bytes, synth
from yule_amd.backend import HipBackend, HipRunner
from yule_amd.model import LAYER_KEYS, LlamaConfig, SyntheticModel

# model shapes (layers, dim, query heads, KV heads, FFN width, vocabulary)
SHAPES = {
    "tinyllama": (22, 2048, 32, 4, 5632, 32000),
    "llama3-8b": (2, 4096, 32, 8, 14336, 32000),   # its layers, two of them
}
CONTEXT = 2048   # positions a runner is created for
FORMATS = ("Q4_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K", "Q8_K")


def listed():
    return [
        # the smallest projection of a decode step (TinyLlama's K or V): launch latency
        {"name": "matvec_small", "kind": "matvec", "dtype": "Q4_K", "rows": 256, "cols": 2048},
        # an ordinary matrix of another format with an odd row count and a width that fills no team evenly
        {"name": "matvec_odd", "kind": "matvec", "dtype": "Q5_K", "rows": 4099, "cols": 5120},
        # a decoder layer's projections at the 8B width in 4 bits, the bulk of a decode step
        {"name": "layer_projections", "kind": "projections", "dtype": "Q4_K", "dim": 4096, "kv": 1024, "ff": 14336},
        # the largest matrix of an 8B model: logits of the whole vocabulary and the greedy pick
        {"name": "lm_head", "kind": "head", "dtype": "Q6_K", "vocab": 128256, "dim": 4096},
        # one token's attention over a long context
        {"name": "attention_long", "kind": "attention", "heads": 32, "kv_heads": 8, "head_dim": 128, "seq": 15001},
        # a program written against the reference's trait: attention head by head
        {"name": "attention_heads", "kind": "heads", "heads": 32, "kv_heads": 4, "head_dim": 64, "seq": 777},
        # the same program's whole decoder layer, op by op
        {"name": "layer_by_ops", "kind": "block", "shape": "tinyllama", "dtype": "Q4_K", "pos": 300},
        # a short prompt through a byte-quantized matrix, f32 activations
        {"name": "gemm_short", "kind": "gemm", "dtype": "Q8_0", "x": "f32", "m": 13, "rows": 4096, "cols": 4096},
        # an ordinary prompt with a ragged length through a down projection
        {"name": "gemm_ragged", "kind": "gemm", "dtype": "Q6_K", "x": "bf16", "m": 333, "rows": 4096, "cols": 14336},
        # a long prompt through the widest projection: matrix-core rate
        {"name": "gemm_long", "kind": "gemm", "dtype": "Q4_K", "x": "bf16", "m": 2048, "rows": 14336, "cols": 4096},
        # a whole model over a long prompt
        {"name": "prefill_long", "kind": "prefill", "shape": "tinyllama", "prompt": 1531, "pieces": 1},
        # a whole model answering a short prompt
        {"name": "generate", "kind": "decode", "shape": "tinyllama", "prompt": 128, "steps": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("matvec", "projections", "head", "attention", "heads", "block", "gemm", "gemm", "prefill",
                       "decode"))
    if kind == "matvec":
        dtype = rng.choice(FORMATS)
        cols = _log_int(rng, 256, 14336) // GEOMETRY[DType[dtype]][0] * GEOMETRY[DType[dtype]][0]
        return {"kind": kind, "dtype": dtype, "rows": _log_int(rng, 200, min(128256, 4e8 // cols)), "cols": cols}
    if kind == "projections":
        dim = 256 * rng.randint(4, 16)
        return {"kind": kind, "dtype": rng.choice(FORMATS), "dim": dim, "kv": dim // rng.choice((1, 4, 8)),
                "ff": 256 * rng.randint(dim // 100, dim * 7 // 512)}
    if kind == "head":
        return {"kind": kind, "dtype": rng.choice(("Q4_K", "Q6_K", "Q8_0")), "vocab": _log_int(rng, 4096, 100000),
                "dim": 256 * rng.randint(4, 16)}
    if kind == "attention":
        heads, kv = rng.choice(((32, 4), (32, 8), (12, 2), (16, 16)))
        return {"kind": kind, "heads": heads, "kv_heads": kv, "head_dim": rng.choice((64, 80, 128)),
                "seq": _log_int(rng, 1, 15000 * 8 // kv)}
    if kind == "heads":
        heads, kv = rng.choice(((32, 4), (32, 8), (12, 2)))
        return {"kind": kind, "heads": heads, "kv_heads": kv, "head_dim": rng.choice((64, 128)),
                "seq": _log_int(rng, 1, 2000)}
    if kind == "block":
        return {"kind": kind, "shape": rng.choice(list(SHAPES)), "dtype": rng.choice(("Q4_0", "Q8_0", "Q4_K", "Q6_K")),
                "pos": _log_int(rng, 1, 2000) - 1}
    if kind == "gemm":
        cols, x = 256 * rng.randint(4, 56), rng.choice(("bf16", "f32", "bf16 noalloc"))
        # (the allocation-free entry serves what fits its static workspace)
        return {"kind": kind, "dtype": rng.choice(FORMATS), "x": x, "m": _log_int(rng, 1, 64 if "noalloc" in x else 1000),
                "rows": _log_int(rng, 512, 14336 * 4096 // cols), "cols": cols}
    if kind == "prefill":
        return {"kind": kind, "shape": rng.choice(list(SHAPES)), "prompt": _log_int(rng, 4, 1500),
                "pieces": rng.choice((1, 1, 2, 3))}
    return {"kind": kind, "shape": rng.choice(list(SHAPES)), "prompt": _log_int(rng, 2, 800),
            "steps": rng.randint(1, 60)}


# ---------------------------------------------------------------- inputs (host)
def _activations(seed, shape):
    """N(0, 1) with a few channels of larger magnitude, as a residual stream has after its norm."""
    x = synth.gauss(seed, shape)
    loud = np.random.default_rng(seed).permutation(shape[-1])[:max(1, shape[-1] // 256)]
    x[..., loud] *= 8.0
    return x


def _bf16(x):
    """(u16 bit patterns, their values in f32), rounded to nearest even."""
    t = torch.from_numpy(x).to(torch.bfloat16)
    return t.view(torch.int16).numpy().view(np.uint16), t.float().numpy()


def _model(case, seed):
    layers, dim, heads, kv, ff, vocab = SHAPES[case["shape"]]
    cfg = LlamaConfig(layers, dim, heads, kv, ff, vocab, CONTEXT)
    return SyntheticModel.generate(cfg, seed=seed % 100003, scheme="Q4_K_M")


def _prompt(case, seed):
    return synth.uniform_tokens(seed * 7 + 5, case["prompt"], SHAPES[case["shape"]][5])


def _pieces(case):
    """Lengths of the pieces that a prompt arrives in."""
    n, k = case["prompt"], min(case["pieces"], case["prompt"])
    return [n // k + (1 if i < n % k else 0) for i in range(k)]


def _block_matrices(case):
    _, dim, heads, kv, ff, vocab = SHAPES[case["shape"]]
    kvd = dim // heads * kv
    return {"embd": (vocab, dim), "q": (dim, dim), "k": (kvd, dim), "v": (kvd, dim), "o": (dim, dim),
            "gate": (ff, dim), "up": (ff, dim), "down": (dim, ff)}


def _inputs(case, seed):
    """Host arrays of a case, from its seed alone."""
    s, kind = seed * 64, case["kind"]
    if kind == "matvec":
        dt = DType[case["dtype"]]
        return {"w": synth.gen_quant(dt, s, case["rows"], case["cols"]), "x": _activations(s + 1, (case["cols"],))}
    if kind == "projections":
        dt, d, kv, ff = DType[case["dtype"]], case["dim"], case["kv"], case["ff"]
        mats = {"q": (d, d), "k": (kv, d), "v": (kv, d), "o": (d, d), "gate": (ff, d), "up": (ff, d), "down": (d, ff)}
        got = {n: synth.gen_quant(dt, s + i, r, c) for i, (n, (r, c)) in enumerate(mats.items())}
        got |= {"x": _activations(s + 20, (d,)), "attn": synth.gauss(s + 21, (d,)),
                "act": synth.gauss(s + 22, (ff,), 0.5)}
        return got
    if kind == "head":
        return {"w": synth.gen_quant(DType[case["dtype"]], s, case["vocab"], case["dim"]),
                "x": _activations(s + 1, (case["dim"],))}
    if kind in ("attention", "heads"):
        kvd = case["kv_heads"] * case["head_dim"]
        return {"q": synth.gauss(s, (case["heads"] * case["head_dim"],)), "k": synth.gauss(s + 1, (case["seq"], kvd)),
                "v": synth.gauss(s + 2, (case["seq"], kvd))}
    if kind == "block":
        _, dim, heads, kv, _, vocab = SHAPES[case["shape"]]
        kvd = dim // heads * kv
        dt = DType[case["dtype"]]
        got = {n: synth.gen_quant(dt, s + i, r, c) for i, (n, (r, c)) in enumerate(_block_matrices(case).items())}
        got |= {"norm1": 1.0 + synth.gauss(s + 20, (dim,), 0.02), "norm2": 1.0 + synth.gauss(s + 21, (dim,), 0.02),
                "kc": synth.gauss(s + 22, (case["pos"] + 1, kvd)), "vc": synth.gauss(s + 23, (case["pos"] + 1, kvd)),
                "token": int(synth.uniform_tokens(s + 24, 1, vocab)[0])}
        return got
    if kind == "gemm":
        x = _activations(s + 1, (case["m"], case["cols"]))
        got = {"w": synth.gen_quant(DType[case["dtype"]], s, case["rows"], case["cols"]), "x": x}
        if case["x"] != "f32":
            got["bits"], got["x"] = _bf16(x)
        return got
    return {"model": _model(case, seed), "prompt": _prompt(case, seed)}


# ---------------------------------------------------------------- state and one pass
_backend = None


def _hip():
    """The program's backend: one per process, as its stream and buffers are."""
    global _backend
    if _backend is None:
        _backend = HipBackend(0)
    return _backend


class Memory:
    """Device buffers by name, freed with the last holder (a state, or a result that is still looked at)."""

    def __init__(self):
        self.hip, self.h = _hip(), {}

    def __del__(self):
        for h in self.h.values():
            self.hip.free(h)


class Buffers(dict):
    """Named output buffers of a state.  The backend's buffers are opaque
    handles and a program leaves its results on the device between calls, so a
    pass returns the buffers and a value is copied out when it is looked at."""

    def __init__(self, memory, shapes):
        super().__init__(shapes)
        self.memory = memory

    def __getitem__(self, name):
        return self.memory.hip.download(self.memory.h[name], super().__getitem__(name),
                                        np.uint32 if name == "token" else np.float32)


class State:
    def __init__(self, case):
        self.hip, self.case, self.memory, self.runner = _hip(), case, Memory(), None
        self.h = self.memory.h

    def upload(self, **arrays):
        for name, a in arrays.items():
            self.h[name] = self.hip.upload(a)

    def out(self, **sizes):
        for name, n in sizes.items():
            self.h[name] = self.hip.allocate(4 * n)

    def outputs(self, **shapes):
        return Buffers(self.memory, shapes)

    def __del__(self):
        if self.runner is not None:
            self.runner.close()


def prepare(case, seed):
    st, kind = State(case), case["kind"]
    a = _inputs(case, seed)
    if kind in ("prefill", "decode"):
        st.runner, st.prompt = HipRunner(st.hip, a["model"]), a["prompt"]
        if kind == "prefill":
            cuts = np.cumsum(_pieces(case))[:-1]
            st.parts = np.split(st.prompt, cuts)
        return st
    if kind == "block":
        st.token = a.pop("token")
    if kind == "gemm" and case["x"] != "f32":
        a["x"] = a.pop("bits")
    st.upload(**a)
    if kind == "matvec":
        st.out(y=case["rows"])
        st.result = st.outputs(y=case["rows"])
    elif kind == "projections":
        d, kv, ff = case["dim"], case["kv"], case["ff"]
        shapes = dict(yq=d, yk=kv, yv=kv, yo=d, ygate=ff, yup=ff, ydown=d)
        st.out(**shapes)
        st.result = st.outputs(**shapes)
    elif kind == "head":
        st.out(logits=case["vocab"], token=1)
        st.result = st.outputs(logits=case["vocab"], token=1)
    elif kind == "attention":
        n = case["heads"] * case["head_dim"]
        st.out(out=n)
        st.result = st.outputs(out=n)
    elif kind == "heads":
        n = case["heads"] * case["head_dim"]
        st.out(scores=case["seq"], probs=case["seq"], out=n)
        st.result = st.outputs(out=n)
    elif kind == "block":
        _, dim, heads, kv, ff, _ = SHAPES[case["shape"]]
        kvd = dim // heads * kv
        st.out(x=dim, n1=dim, yq=dim, yk=kvd, yv=kvd, attn=dim, yo=dim, h1=dim, n2=dim, ygate=ff, yup=ff, act=ff,
               ydown=dim, h2=dim)
        st.result = st.outputs(h2=dim, kc=(case["pos"] + 1, kvd), vc=(case["pos"] + 1, kvd))
    else:
        st.out(y=case["m"] * case["rows"])
        st.result = st.outputs(y=(case["m"], case["rows"]))
    return st


def _run_block(st):
    hip, h, case = st.hip, st.h, st.case
    dt, pos = DType[case["dtype"]], case["pos"]
    _, dim, heads, kv, ff, _ = SHAPES[case["shape"]]
    hd = dim // heads
    kvd = hd * kv
    hip.dequantize(h["embd"], st.token * row_bytes(dt, dim), h["x"], dim // GEOMETRY[dt][0], dt)
    hip.rms_norm(h["x"], h["norm1"], h["n1"], dim, 1e-5)
    hip.quantized_matmul(h["q"], h["n1"], h["yq"], dim, dim, dt)
    hip.quantized_matmul(h["k"], h["n1"], h["yk"], kvd, dim, dt)
    hip.quantized_matmul(h["v"], h["n1"], h["yv"], kvd, dim, dt)
    hip.rope(h["yq"], h["yk"], pos, hd, 10000.0, heads, kv)
    hip.copy_buffer_offset(h["yk"], h["kc"], 0, 4 * pos * kvd, 4 * kvd)
    hip.copy_buffer_offset(h["yv"], h["vc"], 0, 4 * pos * kvd, 4 * kvd)
    hip.gqa_decode_attn(h["yq"], h["kc"], h["vc"], h["attn"], heads, kv, hd, pos + 1)
    hip.quantized_matmul(h["o"], h["attn"], h["yo"], dim, dim, dt)
    hip.add(h["x"], h["yo"], h["h1"], dim)
    hip.rms_norm(h["h1"], h["norm2"], h["n2"], dim, 1e-5)
    hip.quantized_matmul(h["gate"], h["n2"], h["ygate"], ff, dim, dt)
    hip.quantized_matmul(h["up"], h["n2"], h["yup"], ff, dim, dt)
    hip.silu_mul(h["ygate"], h["yup"], h["act"], ff)
    hip.quantized_matmul(h["down"], h["act"], h["ydown"], dim, ff, dt)
    hip.add(h["h1"], h["ydown"], h["h2"], dim)


def run(st):
    hip, h, case = st.hip, st.h, st.case
    kind = case["kind"]
    if kind == "matvec":
        hip.quantized_matmul(h["w"], h["x"], h["y"], case["rows"], case["cols"], DType[case["dtype"]])
    elif kind == "projections":
        dt, d, kv, ff = DType[case["dtype"]], case["dim"], case["kv"], case["ff"]
        hip.quantized_matmul_multi([h["q"], h["k"], h["v"]], h["x"], [h["yq"], h["yk"], h["yv"]], [d, kv, kv], d, dt)
        hip.quantized_matmul(h["o"], h["attn"], h["yo"], d, d, dt)
        hip.quantized_matmul_multi([h["gate"], h["up"]], h["x"], [h["ygate"], h["yup"]], [ff, ff], d, dt)
        hip.quantized_matmul(h["down"], h["act"], h["ydown"], d, ff, dt)
    elif kind == "head":
        hip.quantized_matmul(h["w"], h["x"], h["logits"], case["vocab"], case["dim"], DType[case["dtype"]])
        hip.argmax(h["logits"], case["vocab"], h["token"])
    elif kind == "attention":
        hip.gqa_decode_attn(h["q"], h["k"], h["v"], h["out"], case["heads"], case["kv_heads"], case["head_dim"],
                            case["seq"])
    elif kind == "heads":
        hd, group, stride = case["head_dim"], case["heads"] // case["kv_heads"], case["kv_heads"] * case["head_dim"]
        for i in range(case["heads"]):
            kv = i // group * hd
            hip.attn_score(h["q"], h["k"], h["scores"], hd, case["seq"], i * hd, kv, stride)
            hip.softmax(h["scores"], h["probs"], case["seq"])
            hip.attn_value(h["probs"], h["v"], h["out"], hd, case["seq"], kv, stride, i * hd)
    elif kind == "block":
        _run_block(st)
    elif kind == "gemm":
        entry = {"bf16": hip.quantized_gemm, "f32": hip.quantized_gemm_f32,
                 "bf16 noalloc": hip.quantized_gemm_noalloc}[case["x"]]
        entry(h["w"], h["x"], h["y"], case["m"], case["rows"], case["cols"], DType[case["dtype"]])
    elif kind == "prefill":
        st.runner.reset()
        for part in st.parts:
            logits = st.runner.prefill_batched(part)
        return {"logits": logits}
    else:
        st.runner.reset()
        tokens, _ = st.runner.generate_greedy(st.prompt, case["steps"])
        return {"tokens": tokens.astype(np.int64), "logits": st.runner.decode_step(int(tokens[-1]))}
    return st.result


# ---------------------------------------------------------------- what a pass cannot do without
def _model_work(case):
    """(bytes of the layers and the head, floats of a layer's weights, floats of the head) and the shape."""
    layers, dim, heads, kv, ff, vocab = SHAPES[case["shape"]]
    kvd = dim // heads * kv
    q4 = 2 * dim * dim + 2 * kvd * dim + 2 * ff * dim
    weights = layers * (matrix_bytes(DType.Q4_K, q4 // 256, 256) + matrix_bytes(DType.Q6_K, dim, ff))
    return weights + matrix_bytes(DType.Q6_K, vocab, dim), q4 + dim * ff, vocab * dim


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        r, c = case["rows"], case["cols"]
        return {"bytes": matrix_bytes(DType[case["dtype"]], r, c) + 4 * (r + c), "flops": 2 * r * c}
    if kind == "projections":
        d, kv, ff, dt = case["dim"], case["kv"], case["ff"], DType[case["dtype"]]
        mats = [(d, d), (kv, d), (kv, d), (d, d), (ff, d), (ff, d), (d, ff)]
        return {"bytes": sum(matrix_bytes(dt, r, c) + 4 * r for r, c in mats) + 4 * (2 * d + ff),
                "flops": sum(2 * r * c for r, c in mats)}
    if kind == "head":
        r, c = case["vocab"], case["dim"]
        return {"bytes": matrix_bytes(DType[case["dtype"]], r, c) + 4 * (r + c + 1), "flops": 2 * r * c}
    if kind in ("attention", "heads"):
        n = case["heads"] * case["head_dim"]
        return {"bytes": 8 * case["seq"] * case["kv_heads"] * case["head_dim"] + 8 * n, "flops": 4 * n * case["seq"]}
    if kind == "block":
        _, dim, heads, kv, ff, _ = SHAPES[case["shape"]]
        dt, kvd, mats = DType[case["dtype"]], dim // heads * kv, _block_matrices(case)
        mats.pop("embd")
        return {"bytes": sum(matrix_bytes(dt, r, c) for r, c in mats.values()) + row_bytes(dt, dim) + 12 * dim
                + 8 * (case["pos"] + 1) * kvd,
                "flops": sum(2 * r * c for r, c in mats.values()) + 4 * dim * (case["pos"] + 1)}
    if kind == "gemm":
        m, r, c = case["m"], case["rows"], case["cols"]
        return {"bytes": matrix_bytes(DType[case["dtype"]], r, c) + m * (c * (4 if case["x"] == "f32" else 2) + 4 * r),
                "flops": 2 * m * r * c}
    layers, dim, heads, kv, _, _ = SHAPES[case["shape"]]
    weights, layer, head = _model_work(case)
    kvd, n = dim // heads * kv, case["prompt"]
    prompt_flops = layers * (2 * n * layer + 2 * dim * n * (n + 1)) + 2 * head
    if kind == "prefill":
        return {"bytes": weights + 16 * layers * n * kvd, "flops": prompt_flops}
    steps = case["steps"] + 1
    seen = sum(n + i + 1 for i in range(steps))
    return {"bytes": (steps + 1) * weights + 8 * layers * kvd * (2 * n + seen),
            "flops": prompt_flops + steps * (2 * layers * layer + 2 * head) + 4 * layers * dim * seen}


# About four times the largest error against 64 bits seen over the listed cases and some 70 drawn ones (f32 sums; a
# whole model amplifies the rounding of its first layers).
_REL = {"matvec": 2.7e-6, "projections": 2.7e-6, "head": 2.7e-6, "attention": 1.3e-6, "heads": 2.7e-6, "block": 9e-6,
        "gemm": 4e-6, "prefill": 8e-5, "decode": 2.2e-5}
# Q6_K against bf16 activations: the products of scales and quants above 2048 are rounded to f16 (2^-11)
_REL_Q6K_BF16 = 6.6e-4


def tolerance(case):
    rel = _REL[case["kind"]]
    if case["kind"] == "gemm" and case["dtype"] == "Q6_K" and case["x"] != "f32":
        rel = _REL_Q6K_BF16
    return {"rel": rel, "max": 20 * rel}


# ---------------------------------------------------------------- the same in 64 bits
_DEV = "cuda"


def _f16(b):
    """f16 values (as f64) of byte pairs [..., 2]."""
    return b.contiguous().view(torch.float16).squeeze(-1).double()


def _scales_mins(q):
    """The eight 6-bit scales and mins of a Q4_K / Q5_K header's 12 bytes."""
    q = q.to(torch.int32)
    sc = torch.cat([q[:, 0:4] & 63, (q[:, 8:12] & 15) | ((q[:, 0:4] >> 6) << 4)], 1)
    mn = torch.cat([q[:, 4:8] & 63, (q[:, 8:12] >> 4) | ((q[:, 4:8] >> 6) << 4)], 1)
    return sc.double(), mn.double()


def _dequant(dtype, raw, rows, cols):
    """[rows, cols] f64 weights of raw GGUF blocks."""
    bs, bb = GEOMETRY[dtype]
    b = torch.from_numpy(np.ascontiguousarray(raw).view(np.uint8).reshape(-1)[: rows * cols // bs * bb]).to(_DEV)
    b = b.view(-1, bb)
    n = b.shape[0]
    if dtype == DType.Q8_0:
        w = b[:, 2:].view(torch.int8).double() * _f16(b[:, 0:2])[:, None]
    elif dtype == DType.Q8_K:
        w = b[:, 4:260].view(torch.int8).double() * b[:, 0:4].contiguous().view(torch.float32).double()
    elif dtype == DType.Q4_0:
        # byte i holds weights 2i (low half) and 2i + 1
        q = torch.stack([b[:, 2:] & 15, b[:, 2:] >> 4], 2).reshape(n, 32)
        w = (q.double() - 8.0) * _f16(b[:, 0:2])[:, None]
    elif dtype in (DType.Q4_K, DType.Q5_K):
        sc, mn = _scales_mins(b[:, 4:16])
        qs = b[:, 16:144] if dtype == DType.Q4_K else b[:, 48:176]
        qs = qs.reshape(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32).to(torch.int32)
        if dtype == DType.Q5_K:
            bit = torch.arange(8, device=b.device, dtype=torch.int32).view(1, 8, 1)
            q = q + (((b[:, 16:48].to(torch.int32).view(n, 1, 32) >> bit) & 1) << 4)
        d, dmin = _f16(b[:, 0:2])[:, None], _f16(b[:, 2:4])[:, None]
        w = q.double() * (d * sc)[:, :, None] - (dmin * mn)[:, :, None]
    else:   # Q6_K
        ql, qh = b[:, 0:128].reshape(n, 2, 2, 32).to(torch.int32), b[:, 128:192].reshape(n, 2, 32).to(torch.int32)
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | (((qh >> 6) & 3) << 4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()[:, :, None]
        w = (q.reshape(n, 16, 16).double() - 32.0) * sc * _f16(b[:, 208:210])[:, None, None]
    return w.reshape(rows, cols)


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_DEV).double()


def _norm(x, w, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _silu(x):
    return x * torch.sigmoid(x)


def _angles(positions, hd, base=10000.0):
    """cos and sin [position, pair] of the f32 angles that the model defines."""
    i = np.arange(hd // 2, dtype=np.float32)
    freq = np.float32(1.0) / np.power(np.float32(base), np.float32(2.0) * i / np.float32(hd), dtype=np.float32)
    theta = _t(np.asarray(positions, np.float32)[:, None] * freq[None, :])
    return torch.cos(theta), torch.sin(theta)


def _rope(x, cos, sin):
    """x [n, heads, hd] with interleaved pairs rotated by the n positions' angles."""
    a, b = x[..., 0::2], x[..., 1::2]
    c, s = cos[:, None, :], sin[:, None, :]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _attend(q, k, v, pos0):
    """Causal GQA: q [n, heads, hd] at positions pos0.., k and v [seq, kv_heads, hd]."""
    n, heads, hd = q.shape
    seq, kv, _ = k.shape
    out = torch.empty_like(q)
    hidden = (torch.arange(seq, device=q.device)[None, :] > pos0 + torch.arange(n, device=q.device)[:, None]
              if n > 1 else None)
    for i in range(heads):
        j = i // (heads // kv)
        s = q[:, i] @ k[:, j].T.contiguous() / math.sqrt(hd)
        if hidden is not None:
            s = s.masked_fill(hidden, -math.inf)
        out[:, i] = torch.softmax(s, -1) @ v[:, j].contiguous()
    return out


class _Model64:
    """A dense Llama forward over rows of tokens, weights and KV cache in f64."""

    def __init__(self, model):
        self.cfg, self.k, self.v = model.cfg, [], []
        c = self.cfg

        def mat(t):
            return _dequant(t.dtype, t.data, t.shape[1], t.shape[0])

        self.embd, self.out_norm, self.out = (model["token_embd.weight"], _t(model["output_norm.weight"].data),
                                              mat(model["output.weight"]))
        self.layers = []
        for i in range(c.n_layers):
            t = model.layer(i)
            self.layers.append({k: _t(t[k].data) if k.endswith("norm") else mat(t[k]) for k in LAYER_KEYS})
            self.k.append(torch.zeros(0, c.n_kv_heads, c.head_dim, dtype=torch.float64, device=_DEV))
            self.v.append(torch.zeros(0, c.n_kv_heads, c.head_dim, dtype=torch.float64, device=_DEV))

    def forward(self, tokens):
        """Logits after the last of `tokens`."""
        c, pos0 = self.cfg, self.k[0].shape[0]
        n, hd = len(tokens), c.head_dim
        per = row_bytes(self.embd.dtype, c.dim)
        rows = np.stack([self.embd.data.reshape(-1)[int(t) * per:(int(t) + 1) * per] for t in tokens])
        x = _dequant(self.embd.dtype, rows, n, c.dim)
        cos, sin = _angles(np.arange(pos0, pos0 + n), hd)
        for i, w in enumerate(self.layers):
            h = _norm(x, w["attn_norm"], c.norm_eps)
            q = _rope((h @ w["attn_q"].T).view(n, c.n_heads, hd), cos, sin)
            k = _rope((h @ w["attn_k"].T).view(n, c.n_kv_heads, hd), cos, sin)
            self.k[i] = torch.cat([self.k[i], k])
            self.v[i] = torch.cat([self.v[i], (h @ w["attn_v"].T).view(n, c.n_kv_heads, hd)])
            x = x + _attend(q, self.k[i], self.v[i], pos0).reshape(n, -1) @ w["attn_output"].T
            h = _norm(x, w["ffn_norm"], c.norm_eps)
            x = x + (_silu(h @ w["ffn_gate"].T) * (h @ w["ffn_up"].T)) @ w["ffn_down"].T
        return self.out @ _norm(x[-1], self.out_norm, c.norm_eps)


def _exact_block(case, a):
    _, dim, heads, kv, ff, _ = SHAPES[case["shape"]]
    hd, pos, dt = dim // heads, case["pos"], DType[case["dtype"]]
    per = row_bytes(dt, dim)
    x = _dequant(dt, a["embd"].reshape(-1)[a["token"] * per:(a["token"] + 1) * per], 1, dim)[0]
    w = {n: _dequant(dt, a[n], r, c) for n, (r, c) in _block_matrices(case).items() if n != "embd"}
    n1 = _norm(x, _t(a["norm1"]))
    cos, sin = _angles([pos], hd)
    q = _rope((w["q"] @ n1).view(1, heads, hd), cos, sin)
    kc, vc = _t(a["kc"]), _t(a["vc"])
    kc[pos] = _rope((w["k"] @ n1).view(1, kv, hd), cos, sin).reshape(-1)
    vc[pos] = w["v"] @ n1
    attn = _attend(q, kc.view(-1, kv, hd), vc.view(-1, kv, hd), pos).reshape(-1)
    h1 = x + w["o"] @ attn
    n2 = _norm(h1, _t(a["norm2"]))
    return {"h2": h1 + w["down"] @ (_silu(w["gate"] @ n2) * (w["up"] @ n2)), "kc": kc, "vc": vc}


def exact(case, seed):
    kind, a = case["kind"], _inputs(case, seed)
    if kind == "matvec":
        return {"y": _dequant(DType[case["dtype"]], a["w"], case["rows"], case["cols"]) @ _t(a["x"])}
    if kind == "projections":
        dt, d, kv, ff = DType[case["dtype"]], case["dim"], case["kv"], case["ff"]
        x, attn, act = _t(a["x"]), _t(a["attn"]), _t(a["act"])
        shapes = {"q": (d, d, x), "k": (kv, d, x), "v": (kv, d, x), "o": (d, d, attn), "gate": (ff, d, x),
                  "up": (ff, d, x), "down": (d, ff, act)}
        return {"y" + n: _dequant(dt, a[n], r, c) @ v for n, (r, c, v) in shapes.items()}
    if kind == "head":
        logits = _dequant(DType[case["dtype"]], a["w"], case["vocab"], case["dim"]) @ _t(a["x"])
        return {"logits": logits, "token": None}
    if kind in ("attention", "heads"):
        hd = case["head_dim"]
        return {"out": _attend(_t(a["q"]).view(1, -1, hd), _t(a["k"]).view(case["seq"], -1, hd),
                               _t(a["v"]).view(case["seq"], -1, hd), case["seq"] - 1).reshape(-1)}
    if kind == "block":
        return _exact_block(case, a)
    if kind == "gemm":
        return {"y": _t(a["x"]) @ _dequant(DType[case["dtype"]], a["w"], case["rows"], case["cols"]).T.contiguous()}
    m = _Model64(a["model"])
    logits = m.forward(a["prompt"])
    if kind == "prefill":
        return {"logits": logits}
    for _ in range(case["steps"] + 1):
        logits = m.forward([int(torch.argmax(logits))])
    return {"tokens": None, "logits": logits}
