"""The calls that stand for this framework's work when its speed is measured.

Every case goes through the C entry points of include/nimbleml_hip.h on device buffers,
as a host program of the library calls them: the layers one by one (the FFN sublayer, the
attention layer, a whole block, a cached decode step's attention, the sampler, the tied
head's loss), the training step, and a request (prefill, then cached decode steps).
Weights are the repository's N(0, 0.02) model, activations unit normal.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from nimbleml_amd import _native as N

EPS = 1e-5
DTYPES = {"float16": torch.float16, "float32": torch.float32}
CODES = {"float16": N.F16, "float32": N.F32}
GRAD_SCALE = {"float16": 16384.0, "float32": 1.0}


def listed():
    return [
        # The FFN sublayer of one decode step of 8 rows (RMSNorm, W1 + GELU, W2 + residual):
        # three launches, 16 MB of weights.
        {"name": "ffn_decode_f16", "op": "ffn", "rows": 8, "d": 1024, "dtype": "float16"},
        # The same sublayer at the default dtype for a batch of 48 rows: more rows than a
        # GEMV takes, fewer than a GEMM tile.
        {"name": "ffn_rows48_f32", "op": "ffn", "rows": 48, "d": 1024, "dtype": "float32"},
        # One layer's attention of a batched decode step over rows of ragged length.
        {"name": "decode_attn_f16", "op": "decode_attn", "batch": 32, "heads": 16, "dk": 64,
         "max_seq": 2048, "lo": 128, "hi": 1280, "dtype": "float16"},
        # Choosing the next token of 32 rows with generate()'s defaults (T 0.8, top-p 0.9).
        {"name": "sample_topp_f16", "op": "sample", "batch": 32, "vocab": 32000, "top_k": 0,
         "top_p": 0.9, "penalty": 1.0, "dtype": "float16"},
        # Training the Small configuration (head dim 32) at the default dtype.
        {"name": "train_small_f32", "op": "train", "batch": 8, "seq": 256, "d": 256, "heads": 8,
         "layers": 6, "vocab": 4096, "dtype": "float32"},
        # MultiHeadAttention as the module runs it by default: every key attended.
        {"name": "mha_full_f16", "op": "mha", "batch": 4, "seq": 1024, "d": 1024, "heads": 16,
         "mode": "full", "dtype": "float16"},
        # One block of the 4 x 4096 prefill at d 2048.
        {"name": "block_prefill_f16", "op": "block", "batch": 4, "seq": 4096, "d": 2048,
         "heads": 16, "mode": "causal", "dtype": "float16"},
        # A training step's loss and gradients at d 1024 (two of the model's 24 equal layers),
        # in both dtypes.
        {"name": "train_f16", "op": "train", "batch": 4, "seq": 1024, "d": 1024, "heads": 16,
         "layers": 2, "vocab": 32000, "dtype": "float16"},
        {"name": "train_f32", "op": "train", "batch": 4, "seq": 1024, "d": 1024, "heads": 16,
         "layers": 2, "vocab": 32000, "dtype": "float32"},
        # Evaluating the loss: the tied head and its cross-entropy over 4096 positions.
        {"name": "head_loss_f32", "op": "head_loss", "rows": 4096, "d": 1024, "vocab": 32000,
         "dtype": "float32"},
        # One request: a 512-token prompt, then 32 cached decode steps at batch 1.
        {"name": "request_b1_f16", "op": "request", "batch": 1, "lo": 512, "hi": 512, "steps": 32,
         "d": 1024, "heads": 16, "layers": 24, "vocab": 32000, "max_seq": 2048,
         "dtype": "float16"},
        # A batch of requests of ragged length, prefilled in one pass, then decoded together.
        {"name": "request_b32_f16", "op": "request", "batch": 32, "lo": 128, "hi": 1024,
         "steps": 16, "d": 1024, "heads": 16, "layers": 24, "vocab": 32000, "max_seq": 2048,
         "dtype": "float16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges: odd row counts, ragged and short lengths, every head
    dim the kernels treat apart, both dtypes, causal / full / masked attention."""
    while True:
        c = _draw(rng)
        w = work(c)
        # what a case costs, in fp16 matrix operations: fp32 ones are about ten times as dear
        cost = w["flops"] * (10 if c["dtype"] == "float32" else 1) + 50 * w["bytes"]
        limit = 1.5e12 if c["op"] in ("train", "head_loss") else 4e11
        if cost <= limit:
            return c


def _draw(rng):
    op = rng.choice(["ffn", "ffn", "decode_attn", "sample", "train", "mha", "mha", "block",
                     "head_loss", "request"])
    dtype = rng.choice(["float16", "float32"])
    dk = rng.choice([16, 32, 32, 64, 64, 64, 96, 128, 128])
    heads = rng.choice([4, 8, 12, 16])
    c = {"op": op, "dtype": dtype}
    if op == "ffn":
        return {**c, "rows": _log_int(rng, 1, 16384), "d": 64 * rng.randint(2, 32)}
    if op == "decode_attn":
        hi = _log_int(rng, 64, 2048)
        return {**c, "batch": _log_int(rng, 1, 48), "heads": heads, "dk": dk, "max_seq": 2048,
                "lo": max(1, hi // 8), "hi": hi}
    if op == "sample":
        top_k, top_p = rng.choice([(0, 0.9), (50, 1.0), (0, 1.0), (40, 0.95)])
        return {**c, "batch": _log_int(rng, 1, 64), "vocab": _log_int(rng, 1000, 50304),
                "top_k": top_k, "top_p": top_p, "penalty": rng.choice([1.0, 1.0, 1.2])}
    if op == "mha":
        return {**c, "batch": _log_int(rng, 1, 16), "seq": _log_int(rng, 16, 2048), "d": heads * dk,
                "heads": heads, "mode": rng.choice(["full", "causal", "window", "bias"])}
    if op == "block":
        return {**c, "batch": _log_int(rng, 1, 16), "seq": _log_int(rng, 16, 4096), "d": heads * dk,
                "heads": heads, "mode": rng.choice(["causal", "causal", "full"])}
    if op == "train":
        return {**c, "batch": _log_int(rng, 1, 8), "seq": _log_int(rng, 16, 1024), "d": heads * dk,
                "heads": heads, "layers": rng.randint(1, 4),
                "vocab": 8 * _log_int(rng, 32, 4000)}  # the backward takes multiples of 4
    if op == "head_loss":
        return {**c, "rows": _log_int(rng, 16, 4096), "d": 64 * rng.randint(2, 32),
                "vocab": _log_int(rng, 256, 50304)}
    hi = _log_int(rng, 16, 768)
    return {**c, "batch": _log_int(rng, 1, 32), "lo": rng.choice([hi, max(1, hi // 4)]), "hi": hi,
            "steps": rng.randint(4, 24), "d": heads * dk, "heads": heads,
            "layers": rng.randint(2, 8), "vocab": _log_int(rng, 1000, 32000), "max_seq": 1024}


# ------------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _normal(g, shape, dtype, std=1.0, mean=0.0):
    t = torch.empty(shape, device="cuda", dtype=torch.float32)
    t.normal_(mean, std, generator=g)
    return t.to(dtype)


def _ids(g, shape, vocab):
    return torch.randint(0, vocab, shape, device="cuda", dtype=torch.int64, generator=g)


def _lengths(case, seed):
    r = np.random.RandomState((int(seed) * 31 + 5) % (1 << 31))
    return r.randint(case["lo"], case["hi"] + 1, size=case["batch"]).astype(np.int32)


def _params(case, g):
    """{(kind, layer): tensor} of a model in the device layout ((out, in) weights)."""
    d, f, dt = case["d"], 4 * case["d"], DTYPES[case["dtype"]]
    p = {}
    if "vocab" in case:
        p[(N.P_TOKEN_EMB, 0)] = _normal(g, (case["vocab"], d), dt, 0.02)
        p[(N.P_POS_EMB, 0)] = _normal(g, (_positions(case), d), dt, 0.02)
        p[(N.P_LN_F, 0)] = _normal(g, (d,), dt, 0.1, 1.0)
    for i in range(case.get("layers", 1)):
        p[(N.P_LN1, i)] = _normal(g, (d,), dt, 0.1, 1.0)
        p[(N.P_WQKV, i)] = _normal(g, (3 * d, d), dt, 0.02)
        p[(N.P_BQKV, i)] = _normal(g, (3 * d,), dt, 0.02)
        p[(N.P_WO, i)] = _normal(g, (d, d), dt, 0.02)
        p[(N.P_BO, i)] = _normal(g, (d,), dt, 0.02)
        p[(N.P_LN2, i)] = _normal(g, (d,), dt, 0.1, 1.0)
        p[(N.P_W1, i)] = _normal(g, (f, d), dt, 0.02)
        p[(N.P_B1, i)] = _normal(g, (f,), dt, 0.02)
        p[(N.P_W2, i)] = _normal(g, (d, f), dt, 0.02)
        p[(N.P_B2, i)] = _normal(g, (d,), dt, 0.02)
    return p


def _positions(case):
    return case.get("max_seq", case.get("seq"))


def _mask(case, dtype):
    """The additive mask of a masked call: a causal window of seq / 4 keys, or a bias that
    falls off with distance over every key. None: the call takes no mask."""
    s, mode = case["seq"], case["mode"]
    if mode in ("full", "causal"):
        return None
    i = torch.arange(s, device="cuda")
    dist = i[:, None] - i[None, :]
    if mode == "bias":
        return (dist.abs() * (-4.0 / s)).to(dtype)
    keep = (dist >= 0) & (dist < max(1, s // 4))
    return torch.zeros((s, s), device="cuda").masked_fill(~keep, -math.inf).to(dtype)


class _Foreign:
    """A device buffer of the library as torch sees it."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr,
                                         "data": (int(ptr), False), "version": 3}


class _Model:
    """A device model of the library with the given parameters."""

    def __init__(self, case, params):
        h = C.c_void_p()
        N.check(N.lib.nml_model_create(case.get("vocab", 64), case["d"], case["heads"],
                                       case.get("layers", 1), _positions(case), 4 * case["d"],
                                       CODES[case["dtype"]], C.byref(h)))
        self.h = h
        self.shapes = {k: tuple(t.shape) for k, t in params.items()}
        torch.cuda.synchronize()
        for (kind, layer), t in params.items():
            p = C.c_void_p()
            N.check(N.lib.nml_model_param_ptr(h, kind, layer, C.byref(p)))
            N.check(N.lib.nml_memcpy_d2d(p, t.data_ptr(), t.numel() * t.element_size()))
        N.check(N.lib.nml_synchronize())

    def grads(self):
        """The float32 gradient of every parameter, the library's own buffers."""
        N.check(N.lib.nml_model_zero_grad(self.h))
        out = []
        for (kind, layer), shape in self.shapes.items():
            p = C.c_void_p()
            N.check(N.lib.nml_model_grad_ptr(self.h, kind, layer, C.byref(p)))
            out.append(torch.as_tensor(_Foreign(p.value, shape, "<f4", self), device="cuda"))
        return out

    def __del__(self):
        if getattr(self, "h", None):
            N.lib.nml_model_destroy(self.h)
            self.h = None


def _inputs(case, seed):
    """The tensors of one call, from the seed alone (prepare and exact both start here)."""
    g = _gen(seed)
    dt, op = DTYPES[case["dtype"]], case["op"]
    if op == "ffn":
        d, f = case["d"], 4 * case["d"]
        return {"x": _normal(g, (case["rows"], d), dt), "g": _normal(g, (d,), dt, 0.1, 1.0),
                "w1": _normal(g, (f, d), dt, 0.02), "b1": _normal(g, (f,), dt, 0.02),
                "w2": _normal(g, (d, f), dt, 0.02), "b2": _normal(g, (d,), dt, 0.02)}
    if op == "decode_attn":
        kv = (case["batch"], case["heads"], case["max_seq"], case["dk"])
        return {"q": _normal(g, kv[:2] + kv[3:], dt), "k": _normal(g, kv, dt),
                "v": _normal(g, kv, dt), "lens": torch.from_numpy(_lengths(case, seed)).cuda()}
    if op == "sample":
        b, v = case["batch"], case["vocab"]
        return {"logits": _normal(g, (b, v), dt, 2.5),
                "u": torch.rand((b,), device="cuda", dtype=torch.float64, generator=g),
                "hist": _ids(g, (b, 256), v),
                "hist_len": torch.full((b,), 256, device="cuda", dtype=torch.int32)}
    if op == "head_loss":
        return {"h": _normal(g, (case["rows"], case["d"]), dt),
                "w": _normal(g, (case["vocab"], case["d"]), dt, 0.02),
                "labels": _ids(g, (case["rows"],), case["vocab"])}
    s = {"params": _params(case, g)}
    if op in ("mha", "block"):
        s["x"] = _normal(g, (case["batch"], case["seq"], case["d"]), dt)
        s["mask"] = _mask(case, dt)
    elif op == "train":
        shape = (case["batch"], case["seq"])
        s["ids"], s["labels"] = _ids(g, shape, case["vocab"]), _ids(g, shape, case["vocab"])
    else:
        s["plen"] = _lengths(case, seed)
        s["prompts"] = _ids(g, (case["batch"], int(s["plen"].max())), case["vocab"])
        s["fed"] = _ids(g, (case["steps"], case["batch"]), case["vocab"])
    return s


def prepare(case, seed):
    N.ensure_init()
    s = _inputs(case, seed)
    op, dt = case["op"], DTYPES[case["dtype"]]
    if op == "ffn":
        s["n"] = torch.empty_like(s["x"])
        s["h"] = torch.empty((case["rows"], 4 * case["d"]), device="cuda", dtype=dt)
        s["out"] = torch.empty_like(s["x"])
    elif op == "decode_attn":
        s["out"] = torch.empty((case["batch"], case["heads"] * case["dk"]), device="cuda", dtype=dt)
    elif op == "sample":
        s["out"] = torch.empty((case["batch"],), device="cuda", dtype=torch.int64)
    elif op != "head_loss":
        s["model"] = _Model(case, s.pop("params"))
        if op in ("mha", "block"):
            s["out"] = torch.empty_like(s["x"])
        elif op == "train":
            s["grads"] = s["model"].grads()
        else:
            s["out"] = torch.empty((case["steps"] + 1, case["batch"], case["vocab"]), device="cuda",
                                   dtype=dt)
    s["case"] = dict(case)
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------------- runs

def run(state):
    return _RUN[state["case"]["op"]](state, state["case"])


def _ptr(t):
    return None if t is None else t.data_ptr()


def _run_ffn(s, c):
    r, d, code = c["rows"], c["d"], CODES[c["dtype"]]
    N.check(N.lib.nml_rmsnorm_forward_device(_ptr(s["x"]), _ptr(s["g"]), _ptr(s["n"]), None, None,
                                             r, d, EPS, code))
    N.check(N.lib.nml_linear_device(_ptr(s["n"]), d, _ptr(s["w1"]), _ptr(s["b1"]), None,
                                    _ptr(s["h"]), r, d, 4 * d, 2, code))
    N.check(N.lib.nml_linear_device(_ptr(s["h"]), 4 * d, _ptr(s["w2"]), _ptr(s["b2"]), _ptr(s["x"]),
                                    _ptr(s["out"]), r, 4 * d, d, 3, code))
    return s["out"]


def _run_decode_attn(s, c):
    N.check(N.lib.nml_decode_attention_device(
        _ptr(s["q"]), _ptr(s["k"]), _ptr(s["v"]), _ptr(s["lens"]), _ptr(s["out"]), c["batch"],
        c["heads"], c["max_seq"], c["dk"], math.sqrt(c["dk"]), None, CODES[c["dtype"]]))
    return s["out"]


def _run_sample(s, c):
    penalised = c["penalty"] != 1.0
    N.check(N.lib.nml_sample_device(
        _ptr(s["logits"]), c["batch"], c["vocab"], 0.8, c["top_k"], c["top_p"], c["penalty"],
        _ptr(s["u"]), _ptr(s["hist"]) if penalised else None, 256 if penalised else 0,
        _ptr(s["hist_len"]) if penalised else None, _ptr(s["out"]), CODES[c["dtype"]]))
    return s["out"]


def _run_mha(s, c):
    N.check(N.lib.nml_model_mha_forward(s["model"].h, 0, _ptr(s["x"]), _ptr(s["out"]), c["batch"],
                                        c["seq"], int(c["mode"] == "causal"), _ptr(s["mask"])))
    return s["out"]


def _run_block(s, c):
    N.check(N.lib.nml_model_blocks_forward(s["model"].h, _ptr(s["x"]), _ptr(s["out"]), c["batch"],
                                           c["seq"], 0, int(c["mode"] == "causal"),
                                           _ptr(s["mask"])))
    return s["out"]


def _run_train(s, c):
    h, loss = s["model"].h, C.c_double()
    N.check(N.lib.nml_model_zero_grad(h))
    N.check(N.lib.nml_model_loss_train(h, _ptr(s["ids"]), _ptr(s["labels"]), c["batch"], c["seq"],
                                       0, 0, C.byref(loss)))
    N.check(N.lib.nml_model_backward(h, GRAD_SCALE[c["dtype"]]))
    return {"loss": loss.value, "grads": s["grads"]}


def _run_head_loss(s, c):
    loss = C.c_double()
    N.check(N.lib.nml_tied_ce_forward_device(_ptr(s["h"]), _ptr(s["w"]), _ptr(s["labels"]),
                                             c["rows"], c["d"], c["vocab"], 0, 0, C.byref(loss),
                                             CODES[c["dtype"]]))
    return loss.value


def _run_request(s, c):
    h, b, cache = s["model"].h, c["batch"], C.c_void_p()
    N.check(N.lib.nml_cache_create(h, b, C.byref(cache)))
    try:
        step = b * c["vocab"] * s["out"].element_size()
        out = _ptr(s["out"])
        N.check(N.lib.nml_model_prefill_ragged(h, cache, _ptr(s["prompts"]),
                                               s["prompts"].shape[1],
                                               s["plen"].ctypes.data_as(N.PI32), b, out))
        for t in range(c["steps"]):
            N.check(N.lib.nml_model_forward_cached(h, cache, _ptr(s["fed"]) + 8 * b * t, b, 1,
                                                   out + (t + 1) * step, 0))
    finally:
        N.lib.nml_cache_destroy(cache)
    return s["out"]


_RUN = {"ffn": _run_ffn, "decode_attn": _run_decode_attn, "sample": _run_sample, "mha": _run_mha,
        "block": _run_block, "train": _run_train, "head_loss": _run_head_loss,
        "request": _run_request}


# --------------------------------------------------------------------------- work

def work(case):
    es = 2 if case["dtype"] == "float16" else 4
    op = case["op"]
    if op == "ffn":
        r, d = case["rows"], case["d"]
        return {"bytes": es * (8 * d * d + 2 * r * d), "flops": 16 * r * d * d}
    if op == "decode_attn":
        keys = case["batch"] * case["heads"] * (case["lo"] + case["hi"]) / 2
        return {"bytes": 2 * es * keys * case["dk"], "flops": 4 * keys * case["dk"]}
    if op == "sample":
        n = case["batch"] * case["vocab"]
        return {"bytes": es * n, "flops": 4 * n}
    if op == "head_loss":
        r, d, v = case["rows"], case["d"], case["vocab"]
        return {"bytes": es * d * (r + v), "flops": 2 * r * d * v}
    d = case["d"]
    if op in ("mha", "block"):
        r, s = case["batch"] * case["seq"], case["seq"]
        pairs = r * s * (1 if case["mode"] in ("full", "bias") else
                         0.5 if case["mode"] == "causal" else 0.25)
        dense = 8 if op == "mha" else 24
        return {"bytes": es * (dense / 2 * d * d + 2 * r * d), "flops": dense * r * d * d + 4 * pairs * d}
    layers, v = case["layers"], case["vocab"]
    weights = 12 * layers * d * d + v * d
    if op == "train":
        r, s = case["batch"] * case["seq"], case["seq"]
        fwd = 2 * r * weights + layers * 2 * r * s * d
        # the weights once, their gradients written once (float32)
        return {"bytes": weights * (es + 4), "flops": 3 * fwd}
    mean = (case["lo"] + case["hi"]) / 2
    r, steps, b = case["batch"] * mean, case["steps"], case["batch"]
    ctx = mean + steps / 2
    flops = 24 * layers * d * d * (r + b * steps) + 2 * layers * r * mean * d + \
        2 * b * (steps + 1) * v * d + 4 * layers * b * steps * ctx * d
    kv = 2 * layers * b * d * es
    return {"bytes": (steps + 1) * (weights + b * v) * es + kv * (steps * ctx + mean), "flops": flops}


# ---------------------------------------------------------------------- tolerances

# Largest relative error (2-norm) that another correct implementation would show: about four
# times what the path differs by from 64-bit arithmetic on the same inputs.
_REL = {
    "ffn": {"float16": 2e-3, "float32": 3e-6},
    "decode_attn": {"float16": 2e-3, "float32": 4e-6},
    "mha": {"float16": 4e-3, "float32": 4e-6},
    "block": {"float16": 4e-3, "float32": 4e-6},
    "train": {"float16": 2e-2, "float32": 2e-5},
    "head_loss": {"float16": 1e-4, "float32": 1e-6},
    "request": {"float16": 1e-2, "float32": 1e-5},
}


def tolerance(case):
    if case["op"] == "sample":
        return "exact"
    return {"rel": _REL[case["op"]][case["dtype"]]}


# --------------------------------------------------------------------------- exact

def _f64(t):
    return None if t is None else t.double()


def _rms64(x, g):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * g


def _gelu64(x):
    return 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _attention64(q, k, v, bias):
    """(..., s, dk) attention with an additive bias, one batch row at a time."""
    out = []
    for b in range(q.shape[0]):
        s = q[b] @ k[b].transpose(-1, -2).contiguous() / math.sqrt(q.shape[-1])
        out.append(torch.softmax(s if bias is None else s + bias, -1) @ v[b])
    return torch.stack(out)


def _causal64(s):
    return torch.full((s, s), -math.inf, device="cuda", dtype=torch.float64).triu(1)


def _mha64(x, p, i, heads, bias):
    b, s, d = x.shape
    qkv = (x @ p[(N.P_WQKV, i)].t() + p[(N.P_BQKV, i)]).view(b, s, 3, heads, d // heads)
    q, k, v = (qkv[:, :, j].transpose(1, 2).contiguous() for j in range(3))
    a = _attention64(q, k, v, bias).transpose(1, 2).reshape(b, s, d)
    return a @ p[(N.P_WO, i)].t() + p[(N.P_BO, i)]


def _block64(x, p, i, heads, bias):
    x = x + _mha64(_rms64(x, p[(N.P_LN1, i)]), p, i, heads, bias)
    h = _gelu64(_rms64(x, p[(N.P_LN2, i)]) @ p[(N.P_W1, i)].t() + p[(N.P_B1, i)])
    return x + (h @ p[(N.P_W2, i)].t() + p[(N.P_B2, i)])


def _hidden64(ids, p, case):
    s = ids.shape[1]
    x = p[(N.P_TOKEN_EMB, 0)][ids] + p[(N.P_POS_EMB, 0)][:s]
    bias = _causal64(s)
    for i in range(case["layers"]):
        x = _block64(x, p, i, case["heads"], bias)
    return _rms64(x, p[(N.P_LN_F, 0)])


def _nll64(h, w, labels, rows=4096):
    total = 0.0
    for r in range(0, h.shape[0], rows):
        total = total + torch.nn.functional.cross_entropy(h[r:r + rows] @ w.t(), labels[r:r + rows],
                                                          reduction="sum")
    return total / h.shape[0]


def exact(case, seed):
    op = case["op"]
    if op == "sample":
        return None
    s = _inputs(case, seed)
    if op == "ffn":
        x = s["x"].double()
        h = _gelu64(_rms64(x, s["g"].double()) @ s["w1"].double().t() + s["b1"].double())
        return x + (h @ s["w2"].double().t() + s["b2"].double())
    if op == "decode_attn":
        out = []
        for b, n in enumerate(s["lens"].tolist()):
            q, k, v = s["q"][b].double(), s["k"][b, :, :n].double(), s["v"][b, :, :n].double()
            w = torch.softmax((k * q[:, None]).sum(-1) / math.sqrt(case["dk"]), -1)
            out.append((w[..., None] * v).sum(1).reshape(-1))
        return torch.stack(out)
    if op == "head_loss":
        return float(_nll64(s["h"].double(), s["w"].double(), s["labels"]))
    p = {k: t.double() for k, t in s["params"].items()}
    if op in ("mha", "block"):
        bias = _causal64(case["seq"]) if case["mode"] == "causal" else _f64(s["mask"])
        f = _mha64 if op == "mha" else _block64
        return f(s["x"].double(), p, 0, case["heads"], bias)
    if op == "train":
        for t in p.values():
            t.requires_grad_(True)
        h = _hidden64(s["ids"], p, case)
        loss = _nll64(h.reshape(-1, case["d"]), p[(N.P_TOKEN_EMB, 0)], s["labels"].reshape(-1))
        (loss * GRAD_SCALE[case["dtype"]]).backward()
        return {"loss": float(loss.detach()), "grads": [t.grad for t in p.values()]}
    out = torch.empty((case["steps"] + 1, case["batch"], case["vocab"]), device="cuda",
                      dtype=torch.float64)
    for b, n in enumerate(s["plen"].tolist()):
        ids = torch.cat([s["prompts"][b, :n], s["fed"][:, b]])[None]
        out[:, b] = _hidden64(ids, p, case)[0, n - 1:] @ p[(N.P_TOKEN_EMB, 0)].t()
    return out
