"""The workloads this library is timed on: what a program that serves a Gemma-3-shaped quantized
model has it do, through the public entry points (sapphire_hip.h, kernels.h, quantize.h and
decoder.h) over the sizes of the repository's own configurations.

listed() names the fixed workloads, draw() gives others of the same ranges. prepare() makes what
the program holds before the call (weights in the library's layouts, activations, decoders) from
a seed, run() is one pass, work() its algorithmic bytes and operations, tolerance() what two
correct implementations at the same precision may differ by, and exact() the same outputs in
64-bit arithmetic from plain torch.
"""
from __future__ import annotations

import ctypes as C
import dataclasses
import math

import numpy as np
import torch

from sapphire_amd import load
from sapphire_amd import model as smodel
from sapphire_amd._lib import GemmInput, GemmOutput
from sapphire_amd.engine import Decoder

F32, BF16, Q4_0, Q8_0 = 0, 1, 3, 4
BLOCK_BYTES = {Q4_0: 20, Q8_0: 36}
PACKED, TILED = 1, 2
DTYPES = {"f32": F32, "bf16": BF16, "q4_0": Q4_0, "q8_0": Q8_0}
MODELS = {"gemma3_270m": smodel.GEMMA3_270M, "gemma3_1b": smodel.GEMMA3_1B}
EPS = 1e-6
DEV = "cuda:0"

# Measured against exact() over the listed sizes and draws, each limit about four times the most
# seen: 0.7e-7 to 4.2e-7 for the single layers (32-bit sums in different orders), up to 3.2e-6 for
# the LM head's probabilities (one fp32 normaliser divides them all), 0.8e-7 to 7e-7 for the logits
# of whole decodes.
SUMS32 = {"rel": 1.5e-6, "max": 6e-5}
HEAD32 = {"rel": 1.3e-5, "max": 1e-4}
WHOLE32 = {"rel": 3e-6, "max": 1e-4}


def listed():
    return [
        # One token through one layer's feed-forward block, as a host engine on the device-pointer
        # API issues it (270M shape): the smallest calls, six launches and a copy.
        {"name": "mlp-vector", "kind": "mlp", "dtype": "q4_0", "hidden": 640, "ffn": 2048},
        # One projection through the drop-in host-pointer API (the reference's kernel_gemv).
        {"name": "host-gemv", "kind": "host_gemv", "dtype": "q8_0", "m": 2048, "k": 640},
        # The LM head of the 270M shape with its softmax and greedy token (bench.py's headline).
        {"name": "lm-head-q8", "kind": "lm_head", "dtype": "q8_0", "m": 262144, "k": 640},
        # The LM head of the 1B shape in the smaller block format.
        {"name": "lm-head-q4", "kind": "lm_head", "dtype": "q4_0", "m": 262144, "k": 1152},
        # The weight-tied BF16 LM head over sixteen sequences.
        {"name": "lm-head-bf16-batch", "kind": "gemm_bf16", "m": 262144, "k": 640, "batch": 16},
        # One projection over a prompt of a few hundred tokens (the 1B shape's gate).
        {"name": "projection-prompt", "kind": "gemm_q", "dtype": "q4_0", "m": 6912, "k": 1152, "batch": 300},
        # One layer's feed-forward block of sixteen sequences in lock step (1B shape, fused calls).
        {"name": "mlp-batch", "kind": "mlp_batch", "dtype": "q4_0", "hidden": 1152, "ffn": 6912, "batch": 16},
        # Temperature sampling of one sequence over the whole vocabulary.
        {"name": "sample", "kind": "sample", "n": 262144, "batch": 1, "temperature": 0.8},
        # Quantizing a checkpoint's BF16 embedding rows at load time.
        {"name": "quantize", "kind": "quantize", "src": "bf16", "dtype": "q4_0", "m": 262144, "k": 640},
        # Chat decode of one sequence: greedy tokens, then the logits of the following step.
        {"name": "decode", "kind": "decode", "model": "gemma3_270m", "layers": 18, "vocab": 262144, "dtype": "q4_0",
         "head": "q4_0", "pos": 1024, "steps": 32},
        # Time to first token of a 1000-token prompt.
        {"name": "prompt", "kind": "prompt", "model": "gemma3_270m", "layers": 18, "vocab": 262144, "dtype": "q4_0",
         "head": "q4_0", "pos": 0, "tokens": 1000},
        # Sixteen sequences decoded in lock step: greedy tokens, then the following step's logits.
        {"name": "decode-batch", "kind": "decode_batch", "model": "gemma3_1b", "layers": 26, "vocab": 262144,
         "dtype": "q4_0", "head": "q4_0", "pos": 1024, "steps": 32, "batch": 16},
    ]


def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, int(round(v / multiple)) * multiple)


def draw(rng):
    kind = rng.choice(["mlp", "host_gemv", "lm_head", "gemm_bf16", "gemm_q", "mlp_batch", "sample", "quantize",
                       "decode", "prompt", "decode_batch"])
    quant = rng.choice(["q4_0", "q8_0"])
    c = {"kind": kind}
    if kind == "mlp":
        c.update(dtype=quant, hidden=_log_int(rng, 128, 2560, 32), ffn=_log_int(rng, 256, 8192, 32))
    elif kind == "host_gemv":
        c.update(dtype=rng.choice(["f32", "bf16", "q4_0", "q8_0"]), m=_log_int(rng, 1, 16384), k=_log_int(rng, 32, 4096))
    elif kind == "lm_head":
        c.update(dtype=quant, m=_log_int(rng, 16000, 262144), k=rng.choice([640, 1024, 1152]))
    elif kind == "gemm_bf16":
        c.update(m=_log_int(rng, 512, 262144), k=_log_int(rng, 128, 1152, 8), batch=_log_int(rng, 2, 32))
    elif kind == "gemm_q":
        c.update(dtype=quant, m=_log_int(rng, 128, 16384), k=_log_int(rng, 128, 6912, 128), batch=_log_int(rng, 2, 512))
    elif kind == "mlp_batch":
        c.update(dtype=quant, hidden=128 * rng.randint(1, 9), ffn=_log_int(rng, 256, 8192, 128), batch=rng.randint(1, 16))
    elif kind == "sample":
        c.update(n=_log_int(rng, 2000, 262144), batch=rng.choice([1, 1, 2, 5, 16]), temperature=round(rng.uniform(0.2, 1.5), 2))
    elif kind == "quantize":
        c.update(src=rng.choice(["f32", "bf16"]), dtype=quant, m=_log_int(rng, 256, 262144), k=_log_int(rng, 100, 1152))
    else:
        model = rng.choice(sorted(MODELS))
        c.update(model=model, layers=rng.randint(4, 18), vocab=_log_int(rng, 32000, 262144),
                 dtype=rng.choice(["q4_0", "q4_0", "q8_0"]), head=rng.choice(["q4_0", "q8_0", "bf16"]))
        if kind == "prompt":
            c.update(pos=rng.choice([0, 0, rng.randint(1, 700)]), tokens=_log_int(rng, 5, 1000 if model == "gemma3_270m" else 500))
        else:
            c.update(pos=_log_int(rng, 1, 1900), steps=_log_int(rng, 1, 24))
        if kind == "decode_batch":
            c.update(batch=rng.randint(2, 16))
    return c


# ---- inputs ----

class _Inputs:
    """Tensors on the GPU from one seed, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 1000003 + 17)

    def normal(self, *shape, mean=0.0, std=1.0):
        return torch.randn(*shape, generator=self.g, device=DEV) * std + mean

    def blocks(self, dtype, *rows, k):
        """[*rows, ceil(k / 32), block bytes] uint8: scales |N(0, 0.01)|, uniform quants."""
        nb = (k + 31) // 32
        q = torch.randint(0, 256, (*rows, nb, BLOCK_BYTES[dtype]), generator=self.g, device=DEV, dtype=torch.uint8)
        scale = (torch.randn(*rows, nb, 1, generator=self.g, device=DEV) * 0.01).abs()
        if dtype == Q8_0:
            q.masked_fill_(q == 128, 0)          # quantizers emit -127..127
        q[..., :4] = scale.view(torch.uint8)
        return q

    def matrix(self, dtype, m, k):
        """An [m, k] weight matrix as the framework's callers hold it."""
        if dtype in BLOCK_BYTES:
            return self.blocks(dtype, m, k=k)
        w = self.normal(m, k, std=0.05)
        return w.to(torch.bfloat16) if dtype == BF16 else w


def _dequant(dtype, blocks):
    """float64 weights [..., nb * 32] of a block tensor."""
    scale = blocks[..., :4].contiguous().view(torch.float32).double()
    q = blocks[..., 4:]
    if dtype == Q4_0:
        q = torch.stack([(q & 15).to(torch.int8) - 8, (q >> 4).to(torch.int8) - 8], dim=-1).flatten(-2)
    else:
        q = q.contiguous().view(torch.int8)
    return (q.double() * scale).flatten(-2)


def _weights64(dtype, w, k):
    return _dequant(dtype, w)[..., :k] if dtype in BLOCK_BYTES else w.double()


def _check(rc):
    if rc != 0:
        raise RuntimeError(load().sapphire_last_error().decode(errors="replace"))


def _device_matrix(dtype, blocks, k, layout):
    """A block tensor in one of the library's device layouts."""
    L = load()
    m = blocks.shape[0]
    out = torch.empty(L.sapphire_q_layout_bytes(dtype, layout, m, k), dtype=torch.uint8, device=DEV)
    _check(L.sapphire_q_convert_dev(dtype, blocks.data_ptr(), m, k, layout, out.data_ptr(), None))
    return out


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device=DEV)


# ---- one feed-forward block of one token ----

def _mlp_inputs(c, seed):
    g, dt, h, f = _Inputs(seed), DTYPES[c["dtype"]], c["hidden"], c["ffn"]
    return {"hidden": g.normal(h), "w_pre": g.normal(h, mean=1.0, std=0.1), "w_post": g.normal(h, mean=1.0, std=0.1),
            "gate": g.blocks(dt, f, k=h), "up": g.blocks(dt, f, k=h), "down": g.blocks(dt, h, k=f)}


class _Mlp:
    def prepare(self, c, seed):
        s, dt, h, f = _mlp_inputs(c, seed), DTYPES[c["dtype"]], c["hidden"], c["ffn"]
        s.update(dt=dt, h=h, f=f)
        for n, k in (("gate", h), ("up", h), ("down", f)):
            s[n] = _device_matrix(dt, s[n], k, PACKED)
        s.update(resid=_empty(h), xn=_empty(h), g=_empty(f), u=_empty(f), out=_empty(h))
        s["at"] = {n: x.data_ptr() for n, x in s.items() if torch.is_tensor(x)}
        return s

    def run(self, s):
        L, dt, h, f, p = load(), s["dt"], s["h"], s["f"], s["at"]
        _check(L.sapphire_memcpy_d2d(p["resid"], p["hidden"], 4 * h, None))
        _check(L.sapphire_rmsnorm_delta_dev(p["xn"], p["hidden"], p["w_pre"], EPS, h, 1, None))
        _check(L.sapphire_gemv_q_dev(dt, PACKED, p["gate"], f, h, p["xn"], p["g"], None))
        _check(L.sapphire_gemv_q_dev(dt, PACKED, p["up"], f, h, p["xn"], p["u"], None))
        _check(L.sapphire_gelu_mul_dev(p["g"], p["u"], f, None))
        _check(L.sapphire_gemv_q_dev(dt, PACKED, p["down"], h, f, p["g"], p["out"], None))
        _check(L.sapphire_norm_residual_dev(p["out"], p["resid"], p["w_post"], EPS, h, None))
        return {"hidden": s["out"], "resid": s["resid"], "geglu": s["g"]}

    def work(self, c):
        dt, h, f = DTYPES[c["dtype"]], c["hidden"], c["ffn"]
        return {"bytes": 3 * h * f // 32 * BLOCK_BYTES[dt] + 4 * (3 * h) + 4 * (2 * h + f), "flops": 6 * h * f}

    def tolerance(self, c):
        return SUMS32

    def exact(self, c, seed):
        s, dt = _mlp_inputs(c, seed), DTYPES[c["dtype"]]
        x = _norm64(s["hidden"].double(), s["w_pre"].double())
        g = _gelu64(_dequant(dt, s["gate"]) @ x) * (_dequant(dt, s["up"]) @ x)
        h = s["hidden"].double() + _norm64(_dequant(dt, s["down"]) @ g, s["w_post"].double())
        return {"hidden": h, "resid": h, "geglu": g}


def _norm64(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * (1.0 + w)


def _gelu64(x):
    # the constants are the fp32 ones of the reference's gelu (activations.c:64-76)
    return 0.5 * x * (1.0 + torch.tanh(float(np.float32(0.7978845608)) * (x + float(np.float32(0.044715)) * x ** 3)))


# ---- one GEMV through the host-pointer API ----

class _HostGemv:
    def prepare(self, c, seed):
        L, dt, m, k = load(), DTYPES[c["dtype"]], c["m"], c["k"]
        g = _Inputs(seed)
        w = g.matrix(dt, m, k).cpu().contiguous()
        x = g.normal(k).cpu().numpy()
        ctx = L.kernel_ctx_create(0, 0)
        if not ctx or L.kernel_ctx_init(ctx) != 0:
            raise RuntimeError("kernel_ctx_init")
        t = L.tensor_create_view(dt, 2, (C.c_int * 2)(m, k), w.data_ptr())
        if not t or not L.sapphire_tensor_device_data(t, C.byref(C.c_int()), None):
            raise RuntimeError("tensor_create_view")
        return _HostState(ctx, t, w, x, np.empty(m, np.float32))

    def run(self, s):
        _check(load().kernel_gemv(s.ctx, s.y.ctypes.data, s.t, s.x.ctypes.data))
        return s.y

    def work(self, c):
        return {"bytes": _matrix_bytes(c["dtype"], c["m"], c["k"]) + 4 * (c["m"] + c["k"]), "flops": 2 * c["m"] * c["k"]}

    def tolerance(self, c):
        return SUMS32

    def exact(self, c, seed):
        dt, g = DTYPES[c["dtype"]], _Inputs(seed)
        w = _weights64(dt, g.matrix(dt, c["m"], c["k"]), c["k"])
        return (w @ g.normal(c["k"]).double()).cpu().numpy()


class _HostState:
    def __init__(self, ctx, t, w, x, y):
        self.ctx, self.t, self.w, self.x, self.y = ctx, t, w, x, y

    def __del__(self):
        L = load()
        L.tensor_release(self.t)
        L.kernel_ctx_destroy(self.ctx)


def _matrix_bytes(dtype, m, k):
    dt = DTYPES[dtype]
    return m * ((k + 31) // 32) * BLOCK_BYTES[dt] if dt in BLOCK_BYTES else m * k * (4 if dt == F32 else 2)


# ---- the LM head with its softmax and greedy token ----

class _LmHead:
    def prepare(self, c, seed):
        g, dt = _Inputs(seed), DTYPES[c["dtype"]]
        w = _device_matrix(dt, g.blocks(dt, c["m"], k=c["k"]), c["k"], TILED)
        return {"dt": dt, "m": c["m"], "k": c["k"], "w": w, "x": g.normal(c["k"]), "logits": _empty(c["m"]),
                "probs": _empty(c["m"]), "token": _empty(1, dtype=torch.int32)}

    def run(self, s):
        _check(load().sapphire_gemv_softmax_dev(s["dt"], TILED, s["w"].data_ptr(), s["m"], s["k"], s["x"].data_ptr(),
                                                s["logits"].data_ptr(), s["probs"].data_ptr(), s["token"].data_ptr(), None))
        return {"logits": s["logits"], "probs": s["probs"], "token": s["token"]}

    def work(self, c):
        return {"bytes": _matrix_bytes(c["dtype"], c["m"], c["k"]) + 4 * c["k"] + 8 * c["m"], "flops": 2 * c["m"] * c["k"]}

    def tolerance(self, c):
        return HEAD32

    def exact(self, c, seed):
        g, dt = _Inputs(seed), DTYPES[c["dtype"]]
        w = g.blocks(dt, c["m"], k=c["k"])
        x = g.normal(c["k"]).double()
        y = torch.cat([_dequant(dt, w[i:i + 32768]) @ x for i in range(0, c["m"], 32768)])
        return {"logits": y, "probs": torch.softmax(y, 0), "token": None}


# ---- BF16 rows times a batch ----

class _GemmBf16:
    def prepare(self, c, seed):
        g = _Inputs(seed)
        return {"c": c, "w": g.matrix(BF16, c["m"], c["k"]), "x": g.normal(c["batch"], c["k"]), "y": _empty(c["batch"], c["m"])}

    def run(self, s):
        c = s["c"]
        _check(load().sapphire_gemm_bf16_dev(s["w"].data_ptr(), c["m"], c["k"], s["x"].data_ptr(), c["k"], c["batch"],
                                             s["y"].data_ptr(), c["m"], None))
        return s["y"]

    def work(self, c):
        return {"bytes": 2 * c["m"] * c["k"] + 4 * c["batch"] * (c["m"] + c["k"]), "flops": 2 * c["batch"] * c["m"] * c["k"]}

    def tolerance(self, c):
        return SUMS32

    def exact(self, c, seed):
        g = _Inputs(seed)
        w = g.matrix(BF16, c["m"], c["k"])
        x = g.normal(c["batch"], c["k"]).double()
        return torch.cat([x @ w[i:i + 32768].double().T.contiguous() for i in range(0, c["m"], 32768)], dim=1)


# ---- quantized rows times a batch of tokens ----

class _GemmQ:
    def prepare(self, c, seed):
        L, g, dt = load(), _Inputs(seed), DTYPES[c["dtype"]]
        w = _device_matrix(dt, g.blocks(dt, c["m"], k=c["k"]), c["k"], TILED)
        return {"c": c, "dt": dt, "w": w, "x": g.normal(c["batch"], c["k"]), "y": _empty(c["batch"], c["m"]),
                "ws": _empty(L.sapphire_gemm_workspace_bytes(dt, c["m"], c["k"]), dtype=torch.uint8)}

    def run(self, s):
        c = s["c"]
        _check(load().sapphire_gemm_q_dev(s["dt"], TILED, s["w"].data_ptr(), c["m"], c["k"], s["x"].data_ptr(), c["batch"],
                                          s["y"].data_ptr(), s["ws"].data_ptr(), None))
        return s["y"]

    def work(self, c):
        return {"bytes": _matrix_bytes(c["dtype"], c["m"], c["k"]) + 4 * c["batch"] * (c["m"] + c["k"]),
                "flops": 2 * c["batch"] * c["m"] * c["k"]}

    def tolerance(self, c):
        return SUMS32

    def exact(self, c, seed):
        g, dt = _Inputs(seed), DTYPES[c["dtype"]]
        w = _dequant(dt, g.blocks(dt, c["m"], k=c["k"]))
        return g.normal(c["batch"], c["k"]).double() @ w.T.contiguous()


# ---- one feed-forward block of a batch, fused calls ----

def _mlp_batch_inputs(c, seed):
    g, dt, h, f, b = _Inputs(seed), DTYPES[c["dtype"]], c["hidden"], c["ffn"], c["batch"]
    return {"x": g.normal(b, h), "o": g.normal(b, h), "w_delta": g.normal(h, mean=1.0, std=0.1),
            "w_norm": g.normal(h, mean=1.0, std=0.1), "gate_up": g.blocks(dt, 2 * f, k=h), "down": g.blocks(dt, h, k=f)}


class _MlpBatch:
    def prepare(self, c, seed):
        L, s, dt, h, f, b = load(), _mlp_batch_inputs(c, seed), DTYPES[c["dtype"]], c["hidden"], c["ffn"], c["batch"]
        s["gate_up"] = _device_matrix(dt, s["gate_up"], h, TILED)
        s["down"] = _device_matrix(dt, s["down"], f, TILED)
        need = max(L.sapphire_gemm_workspace_bytes(dt, 2 * f, h), L.sapphire_gemm_workspace_bytes(dt, h, f))
        # the GeGLU output travels in block order: 16 slots, read by the down projection
        s.update(dt=dt, h=h, f=f, b=b, resid=_empty(b, h), g=_empty(16 * f), y=_empty(b, h),
                 ws=_empty(need, dtype=torch.uint8))
        s["calls"] = (
            (GemmInput(x=s["x"].data_ptr(), ldx=h, parts=s["o"].data_ptr(), nparts=1, ldp=h, part_stride=b * h,
                       w_delta=s["w_delta"].data_ptr(), resid_out=s["resid"].data_ptr(), ldr=h,
                       w_norm=s["w_norm"].data_ptr(), eps=EPS, x_blocked=0),
             GemmOutput(y=s["g"].data_ptr(), ldy=0, parts=None, geglu=1, y_blocked=1)),
            (GemmInput(x=s["g"].data_ptr(), ldx=0, parts=None, nparts=0, ldp=0, part_stride=0, w_delta=None,
                       resid_out=None, ldr=0, w_norm=None, eps=EPS, x_blocked=1),
             GemmOutput(y=s["y"].data_ptr(), ldy=h, parts=None, geglu=0, y_blocked=0)))
        return s

    def run(self, s):
        L, dt, h, f, b = load(), s["dt"], s["h"], s["f"], s["b"]
        (i1, o1), (i2, o2) = s["calls"]
        _check(L.sapphire_gemm_q_fused_dev(dt, s["gate_up"].data_ptr(), 2 * f, h, b, C.byref(i1), C.byref(o1),
                                           s["ws"].data_ptr(), None))
        _check(L.sapphire_gemm_q_fused_dev(dt, s["down"].data_ptr(), h, f, b, C.byref(i2), C.byref(o2),
                                           s["ws"].data_ptr(), None))
        return {"resid": s["resid"], "down": s["y"]}

    def work(self, c):
        dt, h, f, b = DTYPES[c["dtype"]], c["hidden"], c["ffn"], c["batch"]
        return {"bytes": 3 * h * f // 32 * BLOCK_BYTES[dt] + 4 * (2 * h + 4 * b * h), "flops": 6 * b * h * f}

    def tolerance(self, c):
        return SUMS32

    def exact(self, c, seed):
        s, dt = _mlp_batch_inputs(c, seed), DTYPES[c["dtype"]]
        h = s["x"].double() + _norm64(s["o"].double(), s["w_delta"].double())
        # gate and up rows interleaved by eight
        gu = _norm64(h, s["w_norm"].double()) @ _dequant(dt, s["gate_up"]).T.contiguous()
        gu = gu.view(c["batch"], -1, 2, 8)
        g = (_gelu64(gu[:, :, 0]) * gu[:, :, 1]).reshape(c["batch"], -1)
        return {"resid": h, "down": g @ _dequant(dt, s["down"]).T.contiguous()}


# ---- temperature sampling ----

class _Sample:
    def inputs(self, c, seed):
        g = _Inputs(seed)
        return g.normal(c["batch"], c["n"], std=2.5), torch.rand(c["batch"], generator=g.g, device=DEV)

    def prepare(self, c, seed):
        logits, draws = self.inputs(c, seed)
        need = load().sapphire_sample_workspace_bytes(c["n"], c["batch"])
        return {"c": c, "logits": logits, "draws": draws, "rows": torch.empty_like(logits),
                "tokens": _empty(c["batch"], dtype=torch.int32), "ws": _empty(need, dtype=torch.uint8)}

    def run(self, s):
        # the draw overwrites its rows: it works on a copy of the logits the program keeps
        L, c = load(), s["c"]
        _check(L.sapphire_memcpy_d2d(s["rows"].data_ptr(), s["logits"].data_ptr(), 4 * c["batch"] * c["n"], None))
        _check(L.sapphire_sample_dev(s["rows"].data_ptr(), c["n"], c["batch"], c["n"], c["temperature"],
                                     s["draws"].data_ptr(), s["tokens"].data_ptr(), s["ws"].data_ptr(), None))
        return {"tokens": s["tokens"], "weights": s["rows"]}

    def work(self, c):
        return {"bytes": 8 * c["batch"] * c["n"] + 8 * c["batch"], "flops": 4 * c["batch"] * c["n"]}

    def tolerance(self, c):
        return "exact"            # the reference's tokens and weights, bit for bit

    def exact(self, c, seed):
        x = self.inputs(c, seed)[0].double() / c["temperature"]
        return {"tokens": None, "weights": torch.exp((x - x.amax(1, keepdim=True)) / c["temperature"])}


# ---- quantizing checkpoint rows ----

class _Quantize:
    def prepare(self, c, seed):
        src, dt = DTYPES[c["src"]], DTYPES[c["dtype"]]
        return {"c": c, "src": src, "dt": dt, "w": _Inputs(seed).matrix(src, c["m"], c["k"]),
                "out": _empty(_matrix_bytes(c["dtype"], c["m"], c["k"]), dtype=torch.uint8)}

    def run(self, s):
        c = s["c"]
        _check(load().sapphire_quantize_dev(s["dt"], s["src"], s["w"].data_ptr(), c["m"], c["k"], s["out"].data_ptr(), None))
        return s["out"]

    def work(self, c):
        return {"bytes": _matrix_bytes(c["src"], c["m"], c["k"]) + _matrix_bytes(c["dtype"], c["m"], c["k"]),
                "flops": 4 * c["m"] * c["k"]}

    def tolerance(self, c):
        return "exact"            # blocks are bytes

    def exact(self, c, seed):
        return None


# ---- whole decodes ----

def _config(c):
    return dataclasses.replace(MODELS[c["model"]], n_layers=c["layers"], vocab=c["vocab"], wdtype=DTYPES[c["dtype"]],
                               lm_dtype=DTYPES[c["head"]])


def _model_inputs(c, seed):
    """The model's tensors on the GPU (weights [layers, rows, blocks, bytes]) and the input stream."""
    cfg, g = _config(c), _Inputs(seed)
    t = {n: g.blocks(cfg.wdtype, cfg.n_layers, smodel.proj_shape(cfg, n)[0], k=smodel.proj_shape(cfg, n)[1])
         for n in smodel.PROJ}
    for n in smodel.NORMS:
        t[n] = g.normal(cfg.n_layers, cfg.hidden, mean=1.0, std=0.1)
    for n in ("q_norm", "k_norm"):
        t[n] = g.normal(cfg.n_layers, cfg.head_dim, mean=1.0, std=0.1)
    t["norm_final"] = g.normal(cfg.hidden, mean=1.0, std=0.1)
    t["embed"] = g.normal(cfg.vocab, cfg.hidden).to(torch.bfloat16)
    t["head"] = t["embed"] if cfg.lm_dtype == BF16 else g.blocks(cfg.lm_dtype, cfg.vocab, k=cfg.hidden)
    return cfg, g, t


def _kv_inputs(cfg, g, batch, n_pos):
    """Filled K and V caches [batch, layers, kv heads, max_ctx, head_dim], N(0, 1) below n_pos."""
    kv = torch.zeros(2, batch, cfg.n_layers, cfg.n_kv_heads, cfg.max_ctx, cfg.head_dim, device=DEV)
    kv[:, :, :, :, :n_pos] = g.normal(2, batch, cfg.n_layers, cfg.n_kv_heads, n_pos, cfg.head_dim)
    return kv


def _tokens(cfg, g, n):
    return torch.randint(0, cfg.vocab, (n,), generator=g.g, device=DEV).cpu().numpy().astype(np.int32)


def _host_model(cfg, t):
    host = lambda x: x.view(torch.uint8 if x.dtype == torch.uint8 else torch.float32).cpu().numpy()  # noqa: E731
    embed = t["embed"].view(torch.int16).cpu().numpy().view(np.uint16)
    return smodel.SyntheticModel(
        cfg=cfg, seed=0, weights={n: host(t[n]) for n in smodel.PROJ},
        norms={n: host(t[n]) for n in (*smodel.NORMS, "q_norm", "k_norm")}, embed_bf16=embed,
        norm_final=host(t["norm_final"]), lm_head=embed if cfg.lm_dtype == BF16 else host(t["head"]))


def _decoder(cfg, t, kv, batch):
    dec = Decoder(_host_model(cfg, t), batch=batch)
    for b in range(batch if kv is not None else 0):
        k, v = kv[:, b].cpu().numpy()
        dec.set_kv_seq(b, k, v)
    return dec


def _model_work(c, tokens, passes, heads):
    """Weights read once per pass, the attended K/V rows, every token's products."""
    cfg = _config(c)
    layer = sum(_matrix_bytes(c["dtype"], *smodel.proj_shape(cfg, n)) for n in smodel.PROJ) * cfg.n_layers
    params = sum(m * k for m, k in (smodel.proj_shape(cfg, n) for n in smodel.PROJ)) * cfg.n_layers
    head = _matrix_bytes(c["head"], cfg.vocab, cfg.hidden)
    rows = {False: 0, True: 0}                   # attended rows of a local / a global layer
    for p in range(c["pos"], c["pos"] + tokens):
        rows[False] += min(p + 1, cfg.sliding_window)
        rows[True] += p + 1
    n_global = sum(cfg.is_global(l) for l in range(cfg.n_layers))
    kv = rows[True] * n_global + rows[False] * (cfg.n_layers - n_global)
    return {"layer": layer * passes, "head": head * heads, "kv_bytes": kv * cfg.nk * 8, "logits": 4 * cfg.vocab,
            "flops": 2 * params * tokens + 2 * cfg.vocab * cfg.hidden * heads + 4 * kv * cfg.nq}


class _Model64:
    """The model in 64-bit arithmetic; the caches [batch, layers, kv, ctx, hd] grow in place."""

    def __init__(self, cfg, t, kv):
        self.cfg, self.t, self.kv, self.w = cfg, t, kv.double(), {}
        self.rope = {g: self._tables(cfg.rope_theta if g else cfg.rope_local_base) for g in (False, True)}

    def _tables(self, base):
        # the tables are fp32 inputs of the path: 32-bit frequencies and angles
        hd = self.cfg.head_dim
        freq = np.array([np.float32(1.0) / np.float32(float(np.float32(base)) ** float(np.float32(2.0 * i) / np.float32(hd)))
                         for i in range(hd // 2)], np.float32)
        ang = (np.arange(self.cfg.max_ctx, dtype=np.float32)[:, None] * freq[None]).astype(np.float64)
        return [torch.from_numpy(f(ang)).to(DEV).repeat(1, 2) for f in (np.cos, np.sin)]

    def weight(self, name, l):
        if (name, l) not in self.w:
            self.w[name, l] = _dequant(self.cfg.wdtype, self.t[name][l]).T.contiguous()
        return self.w[name, l]

    def forward(self, tokens, pos, seqs):
        """Rows of tokens at positions pos (LongTensors [n]) of sequence seqs[0], or one row of each
        sequence seqs[n] -> hidden [n, H]."""
        cfg, t, w = self.cfg, self.t, self.weight
        hd, n = cfg.head_dim, tokens.shape[0]
        h = t["embed"][tokens].double() * math.sqrt(cfg.hidden)
        for l in range(cfg.n_layers):
            cos, sin = (r[pos][:, None] for r in self.rope[cfg.is_global(l)])
            x = _norm64(h, t["norm_attn"][l].double())

            def heads(name, norm):
                q = _norm64((x @ w(name, l)).view(n, -1, hd), t[norm][l].double())
                half = torch.cat([-q[..., hd // 2:], q[..., :hd // 2]], -1)
                return q * cos + half * sin
            q = heads("wq", "q_norm")
            self.kv[0, seqs, l, :, pos] = heads("wk", "k_norm")
            self.kv[1, seqs, l, :, pos] = (x @ w("wv", l)).view(n, -1, hd)
            top = int(pos.max()) + 1
            at, p = torch.arange(top, device=DEV)[None], pos[:, None]
            seen = at <= p
            if not cfg.is_global(l):
                seen &= at > p - cfg.sliding_window
            a = []
            for hh in range(cfg.n_heads):
                k, v = (self.kv[i, seqs, l, hh * cfg.n_kv_heads // cfg.n_heads, :top] for i in (0, 1))   # [seqs, top, hd]
                # a row of each sequence, or every row of the one sequence
                sc = (k @ q[:, hh, :, None])[..., 0] if len(seqs) == n else q[:, hh] @ k[0].T.contiguous()
                pr = torch.softmax((sc / math.sqrt(cfg.query_pre_attn_scalar)).masked_fill(~seen, -math.inf), -1)
                a.append((pr[:, None] @ v)[:, 0] if len(seqs) == n else pr @ v[0])
            a = torch.stack(a, 1)
            h = h + _norm64(a.flatten(1) @ w("wo", l), t["norm_attn_post"][l].double())
            x = _norm64(h, t["norm_ffn"][l].double())
            g = _gelu64(x @ w("wgate", l)) * (x @ w("wup", l))
            h = h + _norm64(g @ w("wdown", l), t["norm_ffn_post"][l].double())
        return h

    def logits(self, h):
        x = _norm64(h, self.t["norm_final"].double())
        head = self.t["head"]
        return torch.cat([x @ _weights64(self.cfg.lm_dtype, head[i:i + 32768], self.cfg.hidden).T.contiguous()
                          for i in range(0, self.cfg.vocab, 32768)], 1)

    def greedy(self, tokens, pos, steps):
        """`steps` greedy steps of every sequence -> (tokens [steps, batch], last logits)."""
        out, seqs = [], torch.arange(tokens.shape[0], device=DEV)
        for s in range(steps):
            y = self.logits(self.forward(tokens, pos + s, seqs))
            tokens = y.argmax(1)
            out.append(tokens)
        return torch.stack(out), y


class _Decode:
    """`steps` greedy tokens, then one more step whose logits the program takes."""

    def batch(self, c):
        return c.get("batch", 1)

    def inputs(self, c, seed):
        cfg, g, t = _model_inputs(c, seed)
        return cfg, t, _kv_inputs(cfg, g, self.batch(c), c["pos"]), _tokens(cfg, g, self.batch(c))

    def prepare(self, c, seed):
        cfg, t, kv, tok = self.inputs(c, seed)
        return {"dec": _decoder(cfg, t, kv, self.batch(c)), "tokens": tok, "pos": c["pos"], "steps": c["steps"]}

    def run(self, s):
        dec, pos, steps = s["dec"], s["pos"], s["steps"]
        toks, _, _ = dec.generate(s["tokens"][0], pos, steps)
        last, logits, _ = dec.generate(toks[-1], pos + steps, 1, keep_logits=True)
        return {"tokens": np.concatenate([toks, last]), "logits": logits}

    def work(self, c):
        n, b = c["steps"] + 1, self.batch(c)
        w = _model_work(c, n, n, n)
        return {"bytes": w["layer"] + w["head"] + b * (w["kv_bytes"] + w["logits"]), "flops": b * w["flops"]}

    def tolerance(self, c):
        return WHOLE32

    def exact(self, c, seed):
        cfg, t, kv, tok = self.inputs(c, seed)
        m = _Model64(cfg, t, kv)
        pos = torch.full((self.batch(c),), c["pos"], device=DEV)
        toks, y = m.greedy(torch.from_numpy(tok).long().to(DEV), pos, c["steps"] + 1)
        return {"tokens": None, "logits": (y if self.batch(c) == 1 else y[None]).cpu().numpy()}


class _DecodeBatch(_Decode):
    def run(self, s):
        dec, steps = s["dec"], s["steps"]
        pos = np.full(dec.batch, s["pos"], np.int32)
        toks, _, _ = dec.generate_batch(s["tokens"], pos, steps)
        last, logits, _ = dec.generate_batch(toks[-1], pos + steps, 1, keep_logits=True)
        return {"tokens": np.concatenate([toks, last]), "logits": logits}


class _Prompt:
    """A prompt behind `pos` cached positions, then the first token with its logits."""

    def inputs(self, c, seed):
        cfg, g, t = _model_inputs(c, seed)
        return cfg, t, _kv_inputs(cfg, g, 1, c["pos"]), _tokens(cfg, g, c["tokens"])

    def prepare(self, c, seed):
        cfg, t, kv, tok = self.inputs(c, seed)
        return {"dec": _decoder(cfg, t, kv if c["pos"] else None, 1), "tokens": tok, "pos": c["pos"]}

    def run(self, s):
        dec, tok, pos = s["dec"], s["tokens"], s["pos"]
        dec.prefill(tok[:-1], pos)
        first, logits, _ = dec.generate(tok[-1], pos + len(tok) - 1, 1, keep_logits=True)
        return {"token": first, "logits": logits}

    def work(self, c):
        w, cfg = _model_work(c, c["tokens"], 1, 1), _config(c)
        rows = (c["pos"] + 2 * c["tokens"]) * cfg.n_layers * cfg.nk * 8     # the cache read, new rows written and read
        return {"bytes": w["layer"] + w["head"] + rows + w["logits"] + 2 * c["tokens"] * cfg.hidden, "flops": w["flops"]}

    def tolerance(self, c):
        return WHOLE32

    def exact(self, c, seed):
        cfg, t, kv, tok = self.inputs(c, seed)
        m = _Model64(cfg, t, kv)
        n = c["tokens"]
        h = m.forward(torch.from_numpy(tok).long().to(DEV), c["pos"] + torch.arange(n, device=DEV),
                      torch.zeros(1, dtype=torch.long, device=DEV))
        return {"token": None, "logits": m.logits(h[-1:]).cpu().numpy()}


_KINDS = {"mlp": _Mlp(), "host_gemv": _HostGemv(), "lm_head": _LmHead(), "gemm_bf16": _GemmBf16(), "gemm_q": _GemmQ(),
          "mlp_batch": _MlpBatch(), "sample": _Sample(), "quantize": _Quantize(), "decode": _Decode(), "prompt": _Prompt(),
          "decode_batch": _DecodeBatch()}


class _State:
    def __init__(self, kind, held):
        self.kind, self.held = kind, held


def prepare(case, seed):
    kind = _KINDS[case["kind"]]
    return _State(kind, kind.prepare(case, seed))


def run(state):
    return state.kind.run(state.held)


def work(case):
    return _KINDS[case["kind"]].work(case)


def tolerance(case):
    return _KINDS[case["kind"]].tolerance(case)


def exact(case, seed):
    return _KINDS[case["kind"]].exact(case, seed)
