"""The calls a user of accelep_amd makes, over the sizes and options they are made with.

Every case is a dict of plain values. Its "kind" says which path it takes:

* "q8": one linear layer on a constant int8 weight, C = A @ dequant(W), through
  accel_hip_matmul_quantized_fused: what the execution provider issues for a claimed
  MatMul / Gemm / FusedMatMul on a packed constant weight. One activation row is a decode step,
  up to 16 a decode batch, hundreds to thousands a prompt. "scale" is where the weight's scales
  lie ("col": one per output column, "row": one per input row, "tensor": one), "zero" whether it
  has zero points (asymmetric quantization), "epi" what is fused behind it.
* "q8mlp": a decoder layer's int8 MLP block through the device calls: RMSNorm, gate and up,
  SiLU * up, down with the residual in its store.
* "f32": the same layer on an fp32 weight (accel_hip_matmul_fused).
* "mlp": an fp32 MLP of two fused Gemms (bias + GELU, bias + residual).
* "attn": a decoder layer's attention block, as a program that drives the device calls itself
  writes it: RMSNorm, q/k/v on int8 weights, RoPE, KV append, causal attention over the cache,
  o projection with the residual in its store.
* "llama": a whole generation (accel_llama_generate): prompt in, greedy ids and the last logits
  out, on int8 or fp32 weights of the SmolLM2-135M shape.

Weights are uploaded once, and int8 weights prepared once (accel_hip_prepare_quantized), as a
loader does; inputs and outputs stay in the library's device memory.
"""

import ctypes as C
import math

import numpy as np
import torch

from accelep_amd.capi import F32P, I8P, I32P, Epilogue, LlamaConfig, check, lib
from accelep_amd.device import DeviceArray, quant_plane

SMOL = dict(vocab=49152, hidden=576, layers=30, heads=9, kv_heads=3, intermediate=1536, context=640, eps=1e-5,
            rope_theta=100000.0)
EPS = 1e-5
THETA = 100000.0


def listed():
    return [
        # The smallest work: four sequences' step through a small decoder's MLP (latency, launches).
        {"name": "q8_mlp_step_4x576x1536", "kind": "q8mlp", "m": 4, "hidden": 576, "inter": 1536, "zero": False},
        # One token through a large MLP projection: the decode step of a served model.
        {"name": "q8_decode_1x4096x14336", "kind": "q8", "m": 1, "k": 4096, "n": 14336, "scale": "col",
         "zero": False, "epi": "none"},
        # The same projection for a batch of sixteen sequences.
        {"name": "q8_batch_16x4096x14336", "kind": "q8", "m": 16, "k": 4096, "n": 14336, "scale": "col",
         "zero": False, "epi": "none"},
        # A small decode batch on an asymmetrically quantized weight, bias and ReLU fused.
        {"name": "q8_asym_batch_8x4096x4096", "kind": "q8", "m": 8, "k": 4096, "n": 4096, "scale": "col",
         "zero": True, "epi": "bias_relu"},
        # A long prompt through a large projection with the RMSNorm behind it (the largest product).
        {"name": "q8_prefill_2048x4096x14336", "kind": "q8", "m": 2048, "k": 4096, "n": 14336, "scale": "col",
         "zero": False, "epi": "rms"},
        # A prompt of no round length on an asymmetrically quantized weight, bias and GELU fused.
        {"name": "q8_asym_prefill_333x4096x4096", "kind": "q8", "m": 333, "k": 4096, "n": 4096, "scale": "col",
         "zero": True, "epi": "bias_gelu"},
        # The fp32 MLP of an encoder: 256 rows, 1024 -> 4096 -> 1024.
        {"name": "mlp_f32_256x1024x4096", "kind": "mlp", "m": 256, "d": 1024, "h": 4096},
        # A large fp32 product with a ragged row count.
        {"name": "f32_gemm_1000x4096x4096", "kind": "f32", "m": 1000, "k": 4096, "n": 4096, "epi": "none"},
        # One token through an fp32 projection (an unquantized model's decode step).
        {"name": "f32_decode_1x4096x4096", "kind": "f32", "m": 1, "k": 4096, "n": 4096, "epi": "bias"},
        # A prompt's attention block through the device calls.
        {"name": "attn_prompt_512", "kind": "attn", "seq": 512, "position": 0, "hidden": 576, "heads": 9,
         "kv_heads": 3, "dim": 64},
        # A chat turn: a 512-id prompt and 32 new tokens on int8 weights.
        {"name": "llama_int8_512_32", "kind": "llama", "weights": "int8", "prompt": 512, "new": 32},
        # A short completion on fp32 weights (the checkpoint's own type).
        {"name": "llama_f32_64_16", "kind": "llama", "weights": "f32", "prompt": 64, "new": 16},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _size(rng, low, high):
    """A layer's width: mostly whole blocks of 64 or 8, as models have them, one in four odd."""
    v = _log_int(rng, low, high)
    r = rng.random()
    if r < 0.5:
        return max(64, v // 64 * 64)
    return max(8, v // 8 * 8) if r < 0.75 else v | 1


def draw(rng):
    kind = rng.choice(["q8"] * 5 + ["q8mlp"] * 3 + ["f32"] * 4 + ["mlp"] * 2 + ["attn"] * 4 + ["llama"] * 2)
    if kind == "q8":
        # Decode steps and batches of large projections, and prompts through all of them.
        if rng.random() < 0.5:
            m, k, n = _log_int(rng, 1, 16), _size(rng, 2048, 4096), _size(rng, 8192, 14336)
        else:
            m, k, n = _log_int(rng, 33, 2048), _size(rng, 768, 4096), _size(rng, 1024, 14336)
        return {"kind": "q8", "m": m, "k": k, "n": n, "scale": rng.choice(["col"] * 6 + ["tensor", "row"]),
                "zero": rng.random() < 0.35, "epi": rng.choice(["none", "bias", "bias_relu", "bias_gelu", "residual", "rms"])}
    if kind == "q8mlp":
        h = _size(rng, 256, 2048)
        return {"kind": "q8mlp", "m": _log_int(rng, 1, 1024), "hidden": h, "inter": rng.choice([2, 3, 4]) * h,
                "zero": rng.random() < 0.25}
    if kind == "f32":
        m = _log_int(rng, 1, 16) if rng.random() < 0.5 else _log_int(rng, 17, 2048)
        return {"kind": "f32", "m": m, "k": _size(rng, 512, 4096), "n": _size(rng, 512, 4096),
                "epi": rng.choice(["none", "bias", "bias_gelu", "residual"])}
    if kind == "mlp":
        d = _size(rng, 256, 2048)
        return {"kind": "mlp", "m": _log_int(rng, 1, 1024), "d": d, "h": rng.choice([2, 3, 4]) * d}
    if kind == "attn":
        dim = rng.choice([64, 64, 128])
        kv = rng.choice([1, 2, 3, 4])
        heads = kv * rng.choice([1, 2, 3, 4])
        return {"kind": "attn", "seq": _log_int(rng, 1, 1024), "position": rng.choice([0, 0, rng.randrange(1, 2048)]),
                "hidden": heads * dim, "heads": heads, "kv_heads": kv, "dim": dim}
    return {"kind": "llama", "weights": rng.choice(["int8", "f32"]), "prompt": _log_int(rng, 8, 512),
            "new": rng.randrange(4, 17)}


# ---- inputs, made on the GPU from the seed ---------------------------------------------------

class _Made:
    """Host inputs of one case: `exact` computes from the same arrays that `prepare` uploads."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        return (torch.randn(shape, generator=self.g, device="cuda") * std + mean).cpu().numpy()

    def uniform(self, low, high, *shape):
        return (torch.rand(shape, generator=self.g, device="cuda") * (high - low) + low).cpu().numpy()

    def int8(self, low, high, *shape):
        return torch.randint(low, high, shape, generator=self.g, device="cuda", dtype=torch.int8).cpu().numpy()

    def ids(self, high, count):
        return torch.randint(0, high, (count,), generator=self.g, device="cuda", dtype=torch.int32).cpu().numpy()

    def quantized(self, rows, cols, std=0.02):
        """A matrix ~ N(0, std) quantized symmetrically per row: (int8 [rows, cols], scale [rows])."""
        w = torch.randn((rows, cols), generator=self.g, device="cuda") * std
        s = w.abs().amax(dim=1) / 127
        q = torch.round(w / s[:, None]).clamp(-127, 127).to(torch.int8)
        return q.cpu().numpy(), s.cpu().numpy()


def _q8_inputs(case, seed):
    r, m, k, n = _Made(seed), case["m"], case["k"], case["n"]
    count = {"col": n, "row": k, "tensor": 1}[case["scale"]]
    d = {"x": r.normal(m, k), "q": r.int8(-127, 128, k, n), "scale": r.uniform(1e-3, 1e-2, count),
         "zero": r.int8(-32, 33, count) if case["zero"] else None}
    return _epilogue_inputs(d, case["epi"], r, m, n, 1.0)


def _f32_inputs(case, seed):
    r, m, k, n = _Made(seed), case["m"], case["k"], case["n"]
    return _epilogue_inputs({"x": r.normal(m, k), "w": r.normal(k, n, std=0.02)}, case["epi"], r, m, n, 0.02)


def _epilogue_inputs(d, epi, r, m, n, std):
    if epi.startswith("bias"):
        d["bias"] = r.normal(n, std=std)
    if epi == "residual":
        d["residual"] = r.normal(m, n)
    if epi == "rms":
        d["gamma"] = r.normal(n, std=0.1, mean=1.0)
    return d


def _q8mlp_inputs(case, seed):
    r, m, H, I = _Made(seed), case["m"], case["hidden"], case["inter"]
    d = {"x": r.normal(m, H), "norm": r.normal(H, std=0.1, mean=1.0)}
    for name, rows, cols in (("gate", H, I), ("up", H, I), ("down", I, H)):
        q, d["s_" + name] = r.quantized(cols, rows)  # scales per output column
        d["q_" + name] = np.ascontiguousarray(q.T)
        d["z_" + name] = r.int8(-8, 9, cols) if case["zero"] else None
    return d


def _mlp_inputs(case, seed):
    r, m, d, h = _Made(seed), case["m"], case["d"], case["h"]
    return {"x": r.normal(m, d), "w1": r.normal(d, h, std=0.02), "b1": r.normal(h, std=0.02),
            "w2": r.normal(h, d, std=0.02), "b2": r.normal(d, std=0.02)}


def _attn_inputs(case, seed):
    r, seq, pos, H, dim = _Made(seed), case["seq"], case["position"], case["hidden"], case["dim"]
    qo, ko = case["heads"] * dim, case["kv_heads"] * dim
    d = {"x": r.normal(seq, H), "norm": r.normal(H, std=0.1, mean=1.0), "past_k": r.normal(pos, ko),
         "past_v": r.normal(pos, ko)}
    for name, rows, cols in (("q", H, qo), ("k", H, ko), ("v", H, ko), ("o", qo, H)):
        q, s = r.quantized(cols, rows)  # scales per output column
        d["w" + name], d["s" + name] = np.ascontiguousarray(q.T), s
    inv = THETA ** (-np.arange(0, dim, 2) / dim)
    angle = np.arange(pos + seq)[:, None] * np.concatenate([inv, inv])[None, :]
    d["cos"], d["sin"] = np.cos(angle).astype(np.float32), np.sin(angle).astype(np.float32)
    return d


def _llama_weights(r, int8):
    """(kind, layer, matrix, scale or None) in Hugging Face layout; the LM head is tied."""
    H, I, V = SMOL["hidden"], SMOL["intermediate"], SMOL["vocab"]
    kv = SMOL["kv_heads"] * (H // SMOL["heads"])
    make = (lambda o, i: r.quantized(o, i)) if int8 else (lambda o, i: (r.normal(o, i, std=0.02), None))
    emb = make(V, H)
    yield 1, -1, *emb
    yield 3, -1, *emb
    yield 2, -1, r.normal(H, std=0.1, mean=1.0), None
    for layer in range(SMOL["layers"]):
        for kind in (4, 5):
            yield kind, layer, r.normal(H, std=0.1, mean=1.0), None
        for kind, o, i in ((6, H, H), (7, kv, H), (8, kv, H), (9, H, H), (10, I, H), (11, I, H), (12, H, I)):
            yield kind, layer, *make(o, i)


# ---- what a program holds before the call ----------------------------------------------------

class _View:
    """A torch view of a DeviceArray's memory (the array lives as long as the view)."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": array.dtype.str, "data": (array.ptr, False),
                                         "version": 2}


def _view(array):
    return torch.as_tensor(_View(array), device="cuda")


def _weight(q, scale, zero, mode, hold):
    """An int8 weight [k, n] on the device, prepared; returns its plane."""
    k, n = q.shape
    arrays = [DeviceArray.from_numpy(v) if v is not None else None for v in (q, scale, zero)]
    plane = quant_plane(*arrays, [k, n], {"col": 1, "row": 0, "tensor": -1}[mode])
    check(lib().accel_hip_prepare_quantized(C.byref(plane), k, n, 0, None))
    hold += [*arrays, plane]
    return plane


def _epilogue(d, n, hold, out, act=0):
    e = Epilogue(alpha=1.0, beta=1.0, activation=act)
    if "bias" in d:
        hold.append(DeviceArray.from_numpy(d["bias"]))
        e.bias, e.bias_rank = hold[-1].ptr, 1
        e.bias_shape[0] = n
    if "residual" in d:
        hold.append(DeviceArray.from_numpy(d["residual"]))
        e.residual = hold[-1].ptr
    if "gamma" in d:  # the rows are normalized in place
        hold.append(DeviceArray.from_numpy(d["gamma"]))
        e.rms_weight, e.rms_eps, e.rms_out = hold[-1].ptr, EPS, out.ptr
    hold.append(e)
    return e


ACTS = {"bias_relu": 1, "bias_gelu": 2}


class _Llama:
    def __init__(self, case, seed):
        L, r = lib(), _Made(seed)
        self.destroy = L.accel_llama_destroy
        self.h = L.accel_llama_create(C.byref(LlamaConfig(**SMOL)))
        if not self.h:
            raise RuntimeError(L.accel_llama_last_error().decode())
        for kind, layer, w, s in _llama_weights(r, case["weights"] == "int8"):
            rows, cols = (w.shape[0], 1) if w.ndim == 1 else w.shape
            if s is None:
                self.ok(L.accel_llama_weight(self.h, kind, layer, w.ctypes.data_as(F32P), rows, cols))
            else:
                self.ok(L.accel_llama_weight_q8(self.h, kind, layer, w.ctypes.data_as(I8P), s.ctypes.data_as(F32P),
                                                rows, cols))
        self.prompt = r.ids(SMOL["vocab"], case["prompt"])

    def ok(self, rc):
        if rc != 0:
            raise RuntimeError(lib().accel_llama_last_error().decode())

    def __del__(self):
        if self.h:
            self.destroy(self.h)
            self.h = None


def prepare(case, seed):
    check(lib().accel_hip_init())
    kind, hold = case["kind"], []
    up = DeviceArray.from_numpy
    state = {"kind": kind, "hold": hold}
    if kind == "q8":
        d, m, k, n = _q8_inputs(case, seed), case["m"], case["k"], case["n"]
        plane = _weight(d["q"], d["scale"], d["zero"], case["scale"], hold)
        x, c = up(d["x"]), DeviceArray((m, n))
        e = _epilogue(d, n, hold, c, ACTS.get(case["epi"], 0))
        hold += [x, c]
        state.update(args=(x.ptr, None, None, C.byref(plane), c.ptr, m, k, n, C.byref(e)), out=_view(c))
    elif kind == "q8mlp":
        d, m, H, I = _q8mlp_inputs(case, seed), case["m"], case["hidden"], case["inter"]
        b = {"x": up(d["x"]), "norm": up(d["norm"]), "normed": DeviceArray((m, H)), "gate": DeviceArray((m, I)),
             "up": DeviceArray((m, I)), "y": DeviceArray((m, H))}
        planes = {t: _weight(d["q_" + t], d["s_" + t], d["z_" + t], "col", hold) for t in ("gate", "up", "down")}
        state.update(b=b, planes=planes, epi=Epilogue(alpha=1.0, beta=1.0, residual=b["x"].ptr), sizes=(m, H, I),
                     out={"y": _view(b["y"]), "silu_up": _view(b["gate"])})
    elif kind == "f32":
        d, m, k, n = _f32_inputs(case, seed), case["m"], case["k"], case["n"]
        x, w, c = up(d["x"]), up(d["w"]), DeviceArray((m, n))
        e = _epilogue(d, n, hold, c, ACTS.get(case["epi"], 0))
        hold += [x, w, c]
        state.update(args=(x.ptr, w.ptr, c.ptr, m, k, n, C.byref(e)), out=_view(c))
    elif kind == "mlp":
        d, m, w, h = _mlp_inputs(case, seed), case["m"], case["d"], case["h"]
        x, w1, w2, t, y = up(d["x"]), up(d["w1"]), up(d["w2"]), DeviceArray((m, h)), DeviceArray((m, w))
        e1 = _epilogue({"bias": d["b1"]}, h, hold, t, 2)
        e2 = _epilogue({"bias": d["b2"]}, w, hold, y)
        e2.residual = x.ptr
        hold += [x, w1, w2, t, y]
        state.update(first=(x.ptr, w1.ptr, t.ptr, m, w, h, C.byref(e1)),
                     second=(t.ptr, w2.ptr, y.ptr, m, h, w, C.byref(e2)), out={"hidden": _view(t), "y": _view(y)})
    elif kind == "attn":
        d, seq, pos, H, dim = _attn_inputs(case, seed), case["seq"], case["position"], case["hidden"], case["dim"]
        hq, hk = case["heads"], case["kv_heads"]
        b = {name: up(d[name]) for name in ("x", "norm", "cos", "sin")}
        b.update(normed=DeviceArray((seq, H)), q=DeviceArray((seq, hq * dim)), k=DeviceArray((seq, hk * dim)),
                 v=DeviceArray((seq, hk * dim)), kc=DeviceArray((pos + seq, hk * dim)),
                 vc=DeviceArray((pos + seq, hk * dim)), scores=DeviceArray((pos + seq,)),
                 mixed=DeviceArray((seq, hq * dim)), y=DeviceArray((seq, H)))
        for name in ("k", "v"):
            past = np.zeros((pos + seq, hk * dim), np.float32)
            past[:pos] = d["past_" + name]
            b[name + "c"].upload(past)
        planes = {name: _weight(d["w" + name], d["s" + name], None, "col", hold) for name in "qkvo"}
        e = Epilogue(alpha=1.0, beta=1.0, residual=b["x"].ptr)
        hold += [b, e, planes]
        state.update(b=b, planes=planes, epi=e, sizes=(seq, pos, H, hq, hk, dim),
                     out={"y": _view(b["y"]), "k_cache": _view(b["kc"]), "v_cache": _view(b["vc"])})
    else:
        state.update(model=_Llama(case, seed), new=case["new"])
    return state


# ---- one pass --------------------------------------------------------------------------------

def run(state):
    L, kind = lib(), state["kind"]
    if kind == "q8":
        check(L.accel_hip_matmul_quantized_fused(*state["args"]))
        return state["out"]
    if kind == "f32":
        check(L.accel_hip_matmul_fused(*state["args"]))
        return state["out"]
    if kind == "mlp":
        check(L.accel_hip_matmul_fused(*state["first"]))
        check(L.accel_hip_matmul_fused(*state["second"]))
        return state["out"]
    if kind == "q8mlp":
        return _run_q8mlp(L, state)
    if kind == "attn":
        return _run_attention(L, state)
    return _run_llama(L, state)


def _run_q8mlp(L, state):
    b, planes, (m, H, I) = state["b"], state["planes"], state["sizes"]
    check(L.accel_hip_rms_norm(b["x"].buffer, b["norm"].buffer, b["normed"].buffer, m, H, EPS, 0))
    for name in ("gate", "up"):
        check(L.accel_hip_matmul_quantized(b["normed"].ptr, None, None, C.byref(planes[name]), b[name].ptr, m, H, I))
    check(L.accel_hip_silu_mul(b["gate"].buffer, b["up"].buffer, m * I))
    check(L.accel_hip_matmul_quantized_fused(b["gate"].ptr, None, None, C.byref(planes["down"]), b["y"].ptr, m, I, H,
                                             C.byref(state["epi"])))
    return state["out"]


def _run_attention(L, state):
    b, planes = state["b"], state["planes"]
    seq, pos, H, hq, hk, dim = state["sizes"]
    check(L.accel_hip_rms_norm(b["x"].buffer, b["norm"].buffer, b["normed"].buffer, seq, H, EPS, 0))
    for name, heads in (("q", hq), ("k", hk), ("v", hk)):
        check(L.accel_hip_matmul_quantized(b["normed"].ptr, None, None, C.byref(planes[name]), b[name].ptr, seq, H,
                                           heads * dim))
    check(L.accel_hip_rope(b["q"].buffer, b["cos"].buffer, b["sin"].buffer, seq, hq, dim, pos))
    check(L.accel_hip_rope(b["k"].buffer, b["cos"].buffer, b["sin"].buffer, seq, hk, dim, pos))
    check(L.accel_hip_append_cache(b["k"].buffer, b["kc"].buffer, seq, pos, hk, dim))
    check(L.accel_hip_append_cache(b["v"].buffer, b["vc"].buffer, seq, pos, hk, dim))
    check(L.accel_hip_attention(b["q"].buffer, b["kc"].buffer, b["vc"].buffer, b["scores"].buffer, b["mixed"].buffer,
                                seq, pos, hq, hk, dim))
    check(L.accel_hip_matmul_quantized_fused(b["mixed"].ptr, None, None, C.byref(planes["o"]), b["y"].ptr, seq,
                                             hq * dim, H, C.byref(state["epi"])))
    return state["out"]


def _run_llama(L, state):
    model, new = state["model"], state["new"]
    ids, count = np.zeros(new, np.int32), C.c_int32()
    logits = np.empty(SMOL["vocab"], np.float32)
    model.ok(L.accel_llama_generate(model.h, model.prompt.ctypes.data_as(I32P), model.prompt.size, new, -1, 0.0, 0, 0,
                                    ids.ctypes.data_as(I32P), C.byref(count)))
    model.ok(L.accel_llama_logits(model.h, logits.ctypes.data_as(F32P), logits.size))
    return {"ids": ids[:count.value], "logits": logits}


# ---- the work of a pass, and what its results may differ by ----------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("q8", "f32"):
        m, k, n = case["m"], case["k"], case["n"]
        weight = 4 * k * n
        if kind == "q8":
            weight = k * n + (5 if case["zero"] else 4) * {"col": n, "row": k, "tensor": 1}[case["scale"]]
        extra = {"residual": 4 * m * n, "none": 0}.get(case["epi"], 4 * n)
        return {"bytes": weight + 4 * m * k + 4 * m * n + extra, "flops": 2 * m * k * n}
    if kind == "q8mlp":
        m, H, I = case["m"], case["hidden"], case["inter"]
        return {"bytes": 3 * H * I + (5 if case["zero"] else 4) * (2 * I + H) + 4 * H + 4 * (2 * m * H + m * I),
                "flops": 6 * m * H * I}
    if kind == "mlp":
        m, d, h = case["m"], case["d"], case["h"]
        return {"bytes": 4 * (2 * d * h + d + h + 2 * m * d + m * h), "flops": 4 * m * d * h}
    if kind == "attn":
        seq, pos, H, dim = case["seq"], case["position"], case["hidden"], case["dim"]
        qo, ko = case["heads"] * dim, case["kv_heads"] * dim
        pairs = seq * pos + seq * (seq + 1) // 2
        weights = H * (qo + 2 * ko) + qo * H
        return {"bytes": weights + 4 * (2 * qo + 2 * ko + 2 * H) + 4 * (2 * seq * H + 2 * (pos + seq) * ko + 2 * seq * ko)
                + 8 * seq * dim, "flops": 2 * seq * weights + 4 * pairs * qo}
    H, I, V, layers = SMOL["hidden"], SMOL["intermediate"], SMOL["vocab"], SMOL["layers"]
    dim = H // SMOL["heads"]
    kv = SMOL["kv_heads"] * dim
    weights, size = layers * (2 * H * H + 2 * H * kv + 3 * H * I), 1 if case["weights"] == "int8" else 4
    p, new = case["prompt"], case["new"]
    pairs = sum(range(1, p + new + 1))
    seen = sum(range(p + 1, p + new + 1))  # cache rows the decode steps read
    return {"bytes": (1 + new) * size * (weights + H * V) + layers * 8 * kv * (p + seen),
            "flops": 2 * weights * (p + new) + 2 * H * V * (1 + new) + 4 * layers * pairs * H}


def tolerance(case):
    """fp32 sums in another order: the relative error of a K-long fp32 sum of random terms is a
    few 1e-7, up to 1.2e-6 at K = 4096 (measured against 64 bits), a whole model's logits 3e-7 to
    1e-6; two orders differ by the sum of theirs. `max` is one value's difference over the rms (or
    itself where larger)."""
    if case["kind"] == "llama":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}
    return {"rel": 1e-5, "max": 1e-4}


# ---- 64-bit results --------------------------------------------------------------------------

def _d(v):
    return torch.from_numpy(np.ascontiguousarray(v)).cuda().double()


def _finish(c, d, act):
    if "bias" in d:
        c = c + _d(d["bias"])
    if act == 1:
        c = torch.clamp(c, min=0)
    elif act == 2:
        c = _gelu(c)
    if "residual" in d:
        c = c + _d(d["residual"])
    return _rms(c, _d(d["gamma"])) if "gamma" in d else c


def _gelu(c):
    return 0.5 * c * (1 + torch.erf(c / math.sqrt(2)))


def _rms(x, gamma):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * gamma


def _dequant(q, scale, zero, mode):
    shape = {"col": (1, -1), "row": (-1, 1), "tensor": (1, 1)}[mode]
    w = _d(q)
    if zero is not None:
        w = w - _d(zero).reshape(shape)
    return w * _d(scale).reshape(shape)


def _rope(x, cos, sin):
    """x [seq, heads, dim], rotate-half."""
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * cos[:, None, :] + turned * sin[:, None, :]


def _attend(q, k, v, position):
    """q [seq, heads, dim]; k, v [rows, kv_heads, dim]; causal from `position`."""
    seq, heads, dim = q.shape
    rows, group = k.shape[0], heads // k.shape[1]
    seen = torch.arange(rows, device="cuda")[None, :] <= position + torch.arange(seq, device="cuda")[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        s = q[:, h] @ k[:, h // group].T.contiguous() / math.sqrt(dim)
        p = torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1)
        out[:, h] = p @ v[:, h // group].contiguous()
    return out.reshape(seq, heads * dim)


def exact(case, seed):
    kind = case["kind"]
    if kind == "q8":
        d = _q8_inputs(case, seed)
        return _finish(_d(d["x"]) @ _dequant(d["q"], d["scale"], d["zero"], case["scale"]), d,
                       ACTS.get(case["epi"], 0))
    if kind == "f32":
        d = _f32_inputs(case, seed)
        return _finish(_d(d["x"]) @ _d(d["w"]), d, ACTS.get(case["epi"], 0))
    if kind == "q8mlp":
        d = _q8mlp_inputs(case, seed)
        x = _d(d["x"])
        normed = _rms(x, _d(d["norm"]))
        w = {t: _dequant(d["q_" + t], d["s_" + t], d["z_" + t], "col") for t in ("gate", "up", "down")}
        gate = normed @ w["gate"]
        t = gate * torch.sigmoid(gate) * (normed @ w["up"])
        return {"y": t @ w["down"] + x, "silu_up": t}
    if kind == "mlp":
        d = _mlp_inputs(case, seed)
        t = _gelu(_d(d["x"]) @ _d(d["w1"]) + _d(d["b1"]))
        return {"hidden": t, "y": t @ _d(d["w2"]) + _d(d["b2"]) + _d(d["x"])}
    if kind == "attn":
        return _exact_attention(case, _attn_inputs(case, seed))
    return _exact_llama(case, seed)


def _exact_attention(case, d):
    seq, pos, dim, hq, hk = case["seq"], case["position"], case["dim"], case["heads"], case["kv_heads"]
    x, cos, sin = _d(d["x"]), _d(d["cos"])[pos:], _d(d["sin"])[pos:]
    normed = _rms(x, _d(d["norm"]))
    q, k, v = (normed @ _dequant(d["w" + t], d["s" + t], None, "col") for t in "qkv")
    q, k = _rope(q.reshape(seq, hq, dim), cos, sin), _rope(k.reshape(seq, hk, dim), cos, sin)
    kc = torch.cat([_d(d["past_k"]), k.reshape(seq, hk * dim)])
    vc = torch.cat([_d(d["past_v"]), v])
    mixed = _attend(q, kc.reshape(-1, hk, dim), vc.reshape(-1, hk, dim), pos)
    return {"y": mixed @ _dequant(d["wo"], d["so"], None, "col") + x, "k_cache": kc, "v_cache": vc}


def _exact_llama(case, seed):
    r = _Made(seed)
    w = {}
    for kind, layer, m, s in _llama_weights(r, case["weights"] == "int8"):
        if (kind, layer) != (3, -1):  # the LM head is the embedding
            w[kind, layer] = _d(m) * (_d(s)[:, None] if s is not None else 1)
    prompt = torch.from_numpy(r.ids(SMOL["vocab"], case["prompt"])).cuda().long()
    hq, hk = SMOL["heads"], SMOL["kv_heads"]
    dim = SMOL["hidden"] // hq
    inv = THETA ** (-torch.arange(0, dim, 2, device="cuda").double() / dim)
    angle = torch.arange(SMOL["context"], device="cuda")[:, None].double() * torch.cat([inv, inv])[None, :]
    cos, sin = torch.cos(angle), torch.sin(angle)
    caches = [(torch.empty(0, hk, dim, device="cuda").double(),) * 2 for _ in range(SMOL["layers"])]

    def forward(ids, pos):
        x, seq = w[1, -1][ids], len(ids)
        c, s = cos[pos:pos + seq], sin[pos:pos + seq]
        for layer in range(SMOL["layers"]):
            a = _rms(x, w[4, layer])
            q, k, v = (a @ w[t, layer].T for t in (6, 7, 8))
            k = torch.cat([caches[layer][0], _rope(k.reshape(seq, hk, dim), c, s)])
            v = torch.cat([caches[layer][1], v.reshape(seq, hk, dim)])
            caches[layer] = (k, v)
            x = x + _attend(_rope(q.reshape(seq, hq, dim), c, s), k, v, pos) @ w[9, layer].T
            a = _rms(x, w[5, layer])
            gate = a @ w[10, layer].T
            x = x + (gate * torch.sigmoid(gate) * (a @ w[11, layer].T)) @ w[12, layer].T
        return _rms(x[-1], w[2, -1]) @ w[1, -1].T

    logits = forward(prompt, 0)
    ids = []
    for step in range(case["new"]):
        ids.append(int(logits.argmax()))
        logits = forward(torch.tensor(ids[-1:], device="cuda"), case["prompt"] + step)
    return {"ids": np.array(ids, np.int32), "logits": logits}
