"""The performance cases of this framework: what a program on one MI355X has
it do, with the inputs, the work, the tolerance and a 64-bit statement of
each.

Kinds of case:
  qmm      one quantized projection, ops.int4_g64_matmul / int8_pc_matmul:
           decode (a row per sequence), batched decode, prompts
  gemm     one dense product, ops.gemm_bf16 / ops.gemm_f32
  linear   a linear layer's training step compiled from StableHLO: the
           forward product and both gradients (x W, dy W^T, x^T dy)
  sample   the end of a decode step: softmax and argmax over the logits
  chain    the six-op elementwise chain compiled from StableHLO
  layer    one Llama-style decoder layer with int4 weights
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jax-metallib_amd"))

from mi355x import _lib, decoder, ops, programs, runtime  # noqa: E402

DEV = "cuda:0"
BF16 = torch.bfloat16


def listed():
    return [
        # One sequence decoding against one shard (1/8) of a 4096 x 14336
        # projection: the smallest call, launch latency.
        {"name": "int4 shard 1 row", "kind": "qmm", "fmt": "int4", "M": 1, "K": 4096, "N": 1792},
        # The decode step of 16 sequences, the benchmark's headline shape.
        {"name": "int4 decode 16 rows", "kind": "qmm", "fmt": "int4", "M": 16, "K": 4096, "N": 14336},
        # A server's decode batch, per-channel int8 weights.
        {"name": "int8 batch 100 rows", "kind": "qmm", "fmt": "int8", "M": 100, "K": 4096, "N": 14336},
        # A prompt of no particular length through the same projection.
        {"name": "int4 prompt 1000 rows", "kind": "qmm", "fmt": "int4", "M": 1000, "K": 4096, "N": 14336},
        # The decode step with dense bf16 weights.
        {"name": "bf16 decode 16 rows", "kind": "gemm", "dt": "bf16", "batch": 0, "M": 16, "K": 4096, "N": 14336},
        # The benchmark's square product.
        {"name": "bf16 4096^3", "kind": "gemm", "dt": "bf16", "batch": 0, "M": 4096, "K": 4096, "N": 4096},
        # A batch of tokens of no particular size through a projection of no
        # particular width.
        {"name": "bf16 2000 rows", "kind": "gemm", "dt": "bf16", "batch": 0, "M": 2000, "K": 2048, "N": 3000},
        # The benchmark's f32 product.
        {"name": "f32 2048^3", "kind": "gemm", "dt": "f32", "batch": 0, "M": 2048, "K": 2048, "N": 2048},
        # The training step of a classifier head with an odd class count.
        {"name": "bf16 head training step", "kind": "linear", "dt": "bf16", "T": 1024, "D": 1024, "C": 5001},
        # Picking the next token of 64 sequences from a 32001-word vocabulary.
        {"name": "f32 sampling 64 rows", "kind": "sample", "dt": "f32", "R": 64, "C": 32001},
        # The benchmark's elementwise chain.
        {"name": "bf16 chain 8192^2", "kind": "chain", "dt": "bf16", "R": 8192, "C": 8192},
        # One layer of the benchmark's decoder, 4 x 2048 tokens: the largest.
        {"name": "int4 decoder layer", "kind": "layer", "hidden": 2048, "B": 4, "S": 2048},
    ]


def _log(rng, lo, hi, mult=1):
    """A size from lo..hi, spread over its logarithm, a multiple of mult."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(mult, int(round(v / mult)) * mult)


def draw(rng):
    kind = rng.choice(["qmm", "qmm", "qmm", "gemm", "gemm", "gemm", "linear", "linear", "sample", "chain", "layer"])
    if kind == "qmm":
        return {"kind": kind, "fmt": rng.choice(["int4", "int8"]), "M": _log(rng, 1, 4096),
                "K": _log(rng, 1024, 8192, 64), "N": _log(rng, 1000, 14336, 8)}
    if kind == "gemm":
        dt = rng.choice(["bf16", "bf16", "f32"])
        if dt == "bf16" and rng.random() < 0.3:  # attention scores and values over 2..32 heads
            return {"kind": kind, "dt": dt, "batch": rng.randint(2, 32), "M": _log(rng, 64, 2048),
                    "K": _log(rng, 64, 1024, 8), "N": _log(rng, 64, 2048, 8)}
        top = 14336 if dt == "bf16" else 4096
        return {"kind": kind, "dt": dt, "batch": 0, "M": _log(rng, 1, 4096), "K": _log(rng, 256, 4096, 8),
                "N": _log(rng, 256, top, 8)}
    if kind == "linear":
        return {"kind": kind, "dt": rng.choice(["bf16", "f32"]), "T": _log(rng, 64, 2048), "D": _log(rng, 64, 1536),
                "C": _log(rng, 10, 8192)}
    if kind == "sample":
        return {"kind": kind, "dt": rng.choice(["f32", "bf16"]), "R": _log(rng, 1, 4096), "C": _log(rng, 1000, 50000)}
    if kind == "chain":
        return {"kind": kind, "dt": rng.choice(["f32", "bf16"]), "R": _log(rng, 16, 8192), "C": _log(rng, 100, 8192)}
    return {"kind": kind, "hidden": rng.choice([1024, 2048]), "B": rng.randint(1, 4), "S": 128 * rng.randint(1, 16)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _dt(name):
    return torch.float32 if name == "f32" else BF16


def _normal(g, shape, scale, dt):
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(dt)


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device=DEV) * (hi - lo) + lo


def _bytes(g, shape, lo, hi, dt):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=dt)


def _int4(g, K, N, lo, hi):
    """A random int4 group-64 weight: packed bytes, bf16 scales, zero points."""
    return decoder.Int4Weight(_bytes(g, (K // 2, N), 0, 256, torch.uint8), _uniform(g, (K // 64, N), lo, hi).to(BF16),
                              _bytes(g, (K // 64, N), 0, 16, torch.uint8))


def _linear_inputs(case, seed):
    """x, W and the output gradient dy of a linear layer."""
    g, dt = _gen(seed), _dt(case["dt"])
    T, D, C = case["T"], case["D"], case["C"]
    return (_normal(g, (T, D), 1.0, dt), _normal(g, (D, C), D ** -0.5, dt), _normal(g, (T, C), 1.0, dt))


def _linear_program(T, D, C, dt):
    """jax.jit of (x, W, dy) -> (x @ W, dy @ W.T, x.T @ dy), as jax.vjp of a
    linear layer lowers it."""
    x, w, y = (f"tensor<{a}x{b}x{dt}>" for a, b in ((T, D), (D, C), (T, C)))

    def dot(name, a, b, ta, tb, ca, cb, out):
        return (f"    %{name} = stablehlo.dot_general {a}, {b}, contracting_dims = [{ca}] x [{cb}], "
                f"precision = [DEFAULT, DEFAULT] : ({ta}, {tb}) -> {out}\n")

    return ("module @jit_linear_step {\n"
            f"  func.func public @main(%arg0: {x}, %arg1: {w}, %arg2: {y}) -> ({y}, {x}, {w}) {{\n"
            + dot(0, "%arg0", "%arg1", x, w, 1, 0, y)
            + dot(1, "%arg2", "%arg1", y, w, 1, 1, x)
            + dot(2, "%arg0", "%arg2", x, y, 0, 0, w)
            + f"    return %0, %1, %2 : {y}, {x}, {w}\n  }}\n}}\n")


def _chain_input(case, seed):
    return _normal(_gen(seed), (case["R"], case["C"]), 2.0, _dt(case["dt"]))


def _layer_config(case):
    h = case["hidden"]
    return decoder.DecoderConfig(layers=1, hidden=h, heads=h // 128, ffn=4 * h, batch=case["B"], seq=case["S"])


def _layer_inputs(case, seed):
    cfg, g = _layer_config(case), _gen(seed)
    H, A, F = cfg.hidden, cfg.heads * cfg.head_dim, cfg.ffn
    w = [_int4(g, k, n, 0.004, 0.006) for k, n in ((H, 3 * A), (A, H), (H, F), (H, F), (F, H))]
    gains = [_uniform(g, (H,), 0.5, 1.5).to(BF16) for _ in range(2)]
    x = _normal(g, (cfg.tokens, H), 1.0, BF16)
    return cfg, decoder.LayerWeights(gains[0], w[0], w[1], gains[1], w[2], w[3], w[4]), x


_CLIENT = None
_EXECUTABLES = {}  # program text -> compiled, as jit keeps one per shape


def _executable(text):
    global _CLIENT
    if _CLIENT is None:
        _CLIENT = runtime.Client()
    if text not in _EXECUTABLES:
        if len(_EXECUTABLES) >= 64:
            _EXECUTABLES.pop(next(iter(_EXECUTABLES))).close()
        _EXECUTABLES[text] = _CLIENT.compile(text)
    return _EXECUTABLES[text]


def _device_buffer(t):
    """A runtime buffer holding the tensor's values."""
    a = t.cpu()
    if a.dtype == BF16:
        return _CLIENT.buffer(a.view(torch.int16).numpy().view(np.uint16), runtime.BF16)
    return _CLIENT.buffer(a.numpy())


class _View:
    """A runtime buffer's device memory for torch.as_tensor, without a copy."""

    def __init__(self, buf):
        self.buf = buf
        self.__cuda_array_interface__ = {
            "shape": buf.shape, "typestr": "<f4" if buf.type == runtime.F32 else "<i2", "version": 2,
            "data": (_lib.lib().mkrt_buffer_device_pointer(buf._h), False)}


def _tensors(buffers):
    out = []
    for b in buffers:
        t = torch.as_tensor(_View(b), device=DEV)
        out.append(t if t.dtype == torch.float32 else t.view(BF16))
    return out


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind == "qmm":
        M, K, N = case["M"], case["K"], case["N"]
        s = {"kind": kind, "fmt": case["fmt"], "x": _normal(g, (M, K), 1.0, BF16)}
        if case["fmt"] == "int4":
            s["w"] = _int4(g, K, N, 1e-3, 1e-2)
        else:
            s["w"] = (_bytes(g, (K, N), -127, 128, torch.int8), _uniform(g, (N,), 1e-3, 1e-2))
        return s
    if kind == "gemm":
        dt, K, lead = _dt(case["dt"]), case["K"], (case["batch"],) if case["batch"] else ()
        return {"kind": kind, "a": _normal(g, lead + (case["M"], K), K ** -0.25, dt),
                "b": _normal(g, lead + (K, case["N"]), K ** -0.25, dt)}
    if kind == "linear":
        exe = _executable(_linear_program(case["T"], case["D"], case["C"], case["dt"]))
        return {"kind": kind, "exe": exe, "in": [_device_buffer(t) for t in _linear_inputs(case, seed)]}
    if kind == "sample":
        return {"kind": kind, "x": _normal(g, (case["R"], case["C"]), 2.0, _dt(case["dt"]))}
    if kind == "chain":
        exe = _executable(programs.chain6(case["R"], case["C"], case["dt"]))
        return {"kind": kind, "exe": exe, "in": [_device_buffer(_chain_input(case, seed))]}
    cfg, lw, x = _layer_inputs(case, seed)
    lw.w_gateup = decoder.interleave_int4(lw.w_gate, lw.w_up)
    return {"kind": kind, "cfg": cfg, "w": lw, "x": x, "buf": decoder.Buffers(cfg, DEV),
            "rope": decoder.rope_tables(cfg, DEV)}


def run(state):
    kind = state["kind"]
    if kind == "qmm":
        if state["fmt"] == "int4":
            w = state["w"]
            return ops.int4_g64_matmul(state["x"], w.packed, w.scale, w.zero)
        return ops.int8_pc_matmul(state["x"], *state["w"])
    if kind == "gemm":
        return (ops.gemm_f32 if state["a"].dtype == torch.float32 else ops.gemm_bf16)(state["a"], state["b"])
    if kind in ("linear", "chain"):
        out, _done = state["exe"].execute(state["in"])
        return _tensors(out)
    if kind == "sample":
        return ops.softmax(state["x"]), ops.argmax(state["x"])
    buf = state["buf"]
    buf.x.copy_(state["x"])
    decoder.layer_forward(state["cfg"], state["w"], buf, *state["rope"])
    return buf.x


# ---------------------------------------------------------------------------
# Work and tolerance
# ---------------------------------------------------------------------------

def _int4_bytes(K, N):
    return K * N // 2 + 3 * (K // 64) * N


def work(case):
    kind = case["kind"]
    if kind == "qmm":
        M, K, N = case["M"], case["K"], case["N"]
        w = _int4_bytes(K, N) if case["fmt"] == "int4" else K * N + 4 * N
        return {"bytes": w + 2 * M * K + 2 * M * N, "flops": 2 * M * K * N}
    if kind == "gemm":
        M, K, N, b = case["M"], case["K"], case["N"], max(1, case["batch"])
        return {"bytes": b * (M * K + K * N + M * N) * (4 if case["dt"] == "f32" else 2), "flops": 2 * b * M * K * N}
    if kind == "linear":
        T, D, C = case["T"], case["D"], case["C"]
        return {"bytes": 2 * (T * D + D * C + T * C) * (4 if case["dt"] == "f32" else 2), "flops": 6 * T * D * C}
    n = case.get("R", 0) * case.get("C", 0)
    if kind == "sample":
        return {"bytes": 2 * n * (4 if case["dt"] == "f32" else 2) + 4 * case["R"], "flops": 5 * n}
    if kind == "chain":
        return {"bytes": 2 * n * (4 if case["dt"] == "f32" else 2), "flops": 6 * n}
    cfg = _layer_config(case)
    H, A, F = cfg.hidden, cfg.heads * cfg.head_dim, cfg.ffn
    w = sum(_int4_bytes(k, n) for k, n in ((H, 3 * A), (A, H), (H, F), (H, F), (F, H)))
    return {"bytes": w + 4 * cfg.tokens * H + 4 * H + 4 * cfg.seq * cfg.head_dim, "flops": cfg.matmul_flops()}


def tolerance(case):
    kind = case["kind"]
    if kind == "layer":  # bf16 activations between nine steps
        return {"rel": 2e-2}
    if kind == "qmm" or case["dt"] == "bf16":  # bf16 results (and, many rows, weights rounded to bf16)
        return {"rel": 8e-3}
    return {"rel": 5e-6}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

def _dequant(w):
    """An int4 group-64 weight as float64 [K, N]."""
    q = torch.stack([w.packed & 15, w.packed >> 4], 1).reshape(-1, w.packed.shape[1]).double()
    return (q - w.zero.double().repeat_interleave(64, 0)) * w.scale.double().repeat_interleave(64, 0)


def _rmsnorm(x, g, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * g.double()


def _exact_layer(case, seed):
    cfg, w, x = _layer_inputs(case, seed)
    B, S, H, D = cfg.batch, cfg.seq, cfg.heads, cfg.head_dim
    x = x.double()
    qkv = (_rmsnorm(x, w.g_attn, cfg.eps) @ _dequant(w.w_qkv)).view(B, S, 3, H, D).permute(2, 0, 3, 1, 4)
    half = D // 2
    inv = cfg.rope_base ** (-torch.arange(half, dtype=torch.float64, device=DEV) * 2.0 / D)
    ang = torch.arange(S, dtype=torch.float64, device=DEV)[:, None] * inv
    c, s = ang.cos(), ang.sin()

    def rope(t):
        a, b = t[..., :half], t[..., half:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    attn = torch.empty((B, S, H * D), dtype=torch.float64, device=DEV)
    future = torch.ones((S, S), dtype=torch.bool, device=DEV).triu(1)
    for b in range(B):
        q, k, v = rope(qkv[0, b]), rope(qkv[1, b]), qkv[2, b]
        p = (q @ k.transpose(1, 2).contiguous() / math.sqrt(D)).masked_fill_(future, -math.inf).softmax(-1)
        attn[b] = (p @ v.contiguous()).transpose(0, 1).reshape(S, H * D)
    x = x + attn.view(B * S, H * D) @ _dequant(w.w_o)
    h = _rmsnorm(x, w.g_mlp, cfg.eps)
    gate = h @ _dequant(w.w_gate)
    return x + (gate * gate.sigmoid() * (h @ _dequant(w.w_up))) @ _dequant(w.w_down)


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        return _exact_layer(case, seed)
    if kind == "linear":
        x, w, dy = (t.double() for t in _linear_inputs(case, seed))
        return [x @ w, dy @ w.t().contiguous(), x.t().contiguous() @ dy]
    if kind == "chain":
        x = _chain_input(case, seed).double()
        b = x * 1.5 + 0.5
        return [torch.where(x > 0, torch.maximum(torch.log1p(torch.exp(b)), x), b)]
    s = prepare(case, seed)
    if kind == "qmm":
        w = _dequant(s["w"]) if case["fmt"] == "int4" else s["w"][0].double() * s["w"][1].double()
        return s["x"].double() @ w
    if kind == "gemm":
        return s["a"].double() @ s["b"].double()
    x = s["x"].double()  # sample: the softmax, and the first of the largest
    at = torch.arange(x.shape[1], device=DEV)
    first = torch.where(x == x.amax(1, keepdim=True), at, x.shape[1]).amin(1)
    return x.softmax(1), first.int()
