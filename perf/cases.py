"""What a user of this package has it do, as cases that can be timed and checked.

A case is one call (or one training step) through the package's public entry
points: ``triton_mxfp8_grouped_mm`` for the forward and the data gradient,
``triton_mxfp8_wgrad``, the quantizer ``to_mx``, and ``MXFP8GroupedLinear``
for a whole training step.  ``listed()`` names the fixed ones, ``draw`` makes
more of the same ranges, ``prepare`` the operands a program has in hand
before the call, ``run`` the call itself, ``exact`` the same result in 64 bits
from plain torch.  The GEMM cases get their MX operands from ``_to_mx`` below
(plain torch, the same bytes as the package's quantizer), so that preparing
them depends on nothing that a change to the kernels could change.

Run with the repository's root as the working directory.
"""

import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.getcwd(), "grouped-gemms_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import kernels  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_BYTES = {"bf16": 2, "f16": 2, "f32": 4}
_BLOCK = 32

# Tokens per expert: "jagged", cumulative ends at random multiples of 32 (a
# training batch as the benchmark draws it: very uneven groups); "routed",
# every token picks an expert at random (a serving batch: any counts, empty
# experts among them).


def listed():
    """The fixed cases, smallest calls to a whole training step."""
    return [
        # The smallest call: a toy layer, a few thousand rows of work; launches
        # and host time are all there is.
        _gemm("forward smallest", "forward", 4, 1024, 512, 512),
        # Serving one decode step: 64 tokens over 8 experts of a large
        # projection, every expert's weight read for a handful of tokens.
        _gemm("forward decode", "forward", 8, 64, 8192, 5120, groups="routed"),
        # One GPU's share of an expert-parallel layer: one expert, 1/8 of the
        # benchmark's tokens.
        _gemm("forward shard", "forward", 1, 2080, 5120, 5120),
        # An ordinary training forward of the benchmark's sweep, 8 uneven
        # experts, narrow output.
        _gemm("forward training", "forward", 8, 16640, 2048, 5120),
        # Many experts and a hidden size that fills neither the 128-byte lines
        # nor the tiles; fp16 model.
        _gemm("forward many experts", "forward", 32, 16640, 2880, 2880, out="f16"),
        # 4-bit weights under 8-bit activations.
        _gemm("forward mxfp4", "forward", 8, 16640, 8192, 5120, weight="e2m1"),
        # The benchmark's largest product, as the data gradient: grad_out
        # (M, N) times the transposed weight.
        _gemm("dgrad largest", "dgrad", 4, 16640, 8192, 8192),
        # Weight gradient of a training batch.
        _gemm("wgrad training", "wgrad", 4, 16640, 5120, 8192),
        # Weight gradient of a small batch, fp32 gradients: a few hundred
        # tokens per expert, the output is most of the traffic.
        _gemm("wgrad small batch", "wgrad", 8, 2080, 2048, 2048, out="f32"),
        # Quantizing a batch of activations before the forward.
        _quant("quantize activations", (1, 16640, 8192), "e4m3", "bf16"),
        # Quantizing a layer's expert weights to 4 bits for serving.
        _quant("quantize weights mxfp4", (8, 2048, 5120), "e2m1", "bf16"),
        # A training step of one MoE projection: quantize, forward, data and
        # weight gradients (the benchmark's layer).
        _gemm("training step", "step", 8, 16640, 8192, 5120),
    ]


def _gemm(name, op, E, M, N, K, weight="e4m3", out="bf16", groups="jagged"):
    c = {"op": op, "E": E, "M": M, "N": N, "K": K, "weight": weight, "out": out, "groups": groups}
    return dict(c, name=name) if name else c


def _quant(name, shape, elem, src):
    c = {"op": "quantize", "B": shape[0], "R": shape[1], "C": shape[2], "elem": elem, "src": src}
    return dict(c, name=name) if name else c


def _log(rng, lo, hi, step):
    """An integer of [lo, hi], spread over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(-(-lo // step), min(hi // step, round(v / step))) * step


def draw(rng):
    """One more case: any of the operations over the listed cases' ranges."""
    op = rng.choice(("forward", "forward", "forward", "dgrad", "wgrad", "wgrad", "quantize", "step"))
    if op == "quantize":
        B, C = rng.choice((1, 1, 8)), _log(rng, 512, 8192, 32)
        R = _log(rng, 64, 16640 if B == 1 else 4096, rng.choice((1, 32)))
        return _quant(None, (B, R, C), rng.choice(("e4m3", "e4m3", "e2m1")), rng.choice(("bf16", "bf16", "f16", "f32")))
    E = rng.choice((1, 2, 4, 8, 16, 32))
    N, K = _log(rng, 512, 8192, 32), _log(rng, 512, 8192, 32)
    if op == "forward":
        routed = rng.random() < 0.5      # serving batches: any token count
        M = _log(rng, 16, 2048, 1) if routed else _log(rng, 32 * E, 16640, 32)
        return _gemm(None, op, E, M, N, K, weight=rng.choice(("e4m3", "e4m3", "e2m1")),
                     out=rng.choice(("bf16", "bf16", "f16", "f32")), groups="routed" if routed else "jagged")
    M = _log(rng, max(1024, 32 * E), 16640, 32)
    return _gemm(None, op, E, M, N, K, out="bf16" if op == "step" else rng.choice(("bf16", "bf16", "f32")))


# --- inputs ---------------------------------------------------------------


def _offsets(case, seed):
    """Cumulative group ends (a list of E ints, the last M), from the seed."""
    E, M = case["E"], case["M"]
    r = random.Random(seed)
    if case["groups"] == "routed":
        counts = [0] * E
        for _ in range(M):
            counts[r.randrange(E)] += 1
    else:
        cuts = sorted(r.sample(range(1, M // 32), E - 1)) if E > 1 else []
        return [32 * c for c in cuts] + [M]
    ends, at = [], 0
    for n in counts:
        at += n
        ends.append(at)
    return ends


def _randn(shape, std, seed, dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(dtype)


def _to_mx(x, elem="e4m3"):
    """(scales uint8, data) of x along its last dim: FLOOR e8m0 scale per 32
    elements, e4m3 bytes or e2m1 pairs (element 2i in the low nibble)."""
    shape = x.shape
    b = x.reshape(-1, shape[-1] // _BLOCK, _BLOCK).float()
    amax = b.abs().amax(dim=-1, keepdim=True).clamp_min(torch.finfo(torch.float32).tiny)
    s = (((amax.view(torch.int32) >> 23) & 0xFF) - (8 if elem == "e4m3" else 2)).clamp(0, 254)
    v = torch.ldexp(b, 127 - s)
    s = s.to(torch.uint8).reshape(*shape[:-1], shape[-1] // _BLOCK)
    if elem == "e4m3":
        return s, v.clamp(-448.0, 448.0).to(torch.float8_e4m3fn).reshape(shape)
    a = v.abs().clamp(max=6.0)
    # round to nearest even in steps of 0.5 (below 2), 1 (below 4) and 2
    code = torch.where(a < 2, (a * 2).round(), torch.where(a < 4, a.round() + 2, (a / 2).round() + 4))
    code = code.to(torch.uint8) | (torch.signbit(v).to(torch.uint8) << 3)
    code = code.reshape(-1, shape[-1] // 2, 2)
    return s, (code[..., 0] | (code[..., 1] << 4)).reshape(*shape[:-1], shape[-1] // 2)


def _dequant(s, q, elem="e4m3"):
    """The values of MX data in float64."""
    if elem == "e4m3":
        v = q.float()
    else:
        grid = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], device=q.device)
        v = grid[torch.stack((q & 15, q >> 4), dim=-1).int()].reshape(*q.shape[:-1], 2 * q.shape[-1])
    v = v.reshape(*s.shape, _BLOCK).double()
    return torch.ldexp(v, (s.int() - 127).unsqueeze(-1)).reshape(*s.shape[:-1], s.shape[-1] * _BLOCK)


def _operands(case, seed):
    """The unquantized operands of a GEMM case: the pair its product takes."""
    E, M, N, K = case["E"], case["M"], case["N"], case["K"]
    if case["op"] == "forward":
        return _randn((M, K), 1.0, 2 * seed), _randn((E, N, K), 0.02, 2 * seed + 1)
    if case["op"] == "dgrad":
        return _randn((M, N), 1.0, 2 * seed), _randn((E, K, N), 0.02, 2 * seed + 1)
    if case["op"] == "wgrad":     # token-major: grad_out^T and input^T
        return _randn((N, M), 1.0, 2 * seed), _randn((K, M), 1.0, 2 * seed + 1)
    return _randn((M, K), 1.0, 3 * seed), _randn((E, N, K), 0.02, 3 * seed + 1), _randn((M, N), 1.0, 3 * seed + 2)


def prepare(case, seed):
    """What a program holds before the call: MX operands and group ends, the
    tensor to quantize, or the layer with its batch and output gradient."""
    if case["op"] == "quantize":
        shape = (case["R"], case["C"]) if case["B"] == 1 else (case["B"], case["R"], case["C"])
        std = 1.0 if case["elem"] == "e4m3" else 0.02
        return {"op": "quantize", "x": _randn(shape, std, seed, _DTYPES[case["src"]]),
                "elem": torch.float8_e4m3fn if case["elem"] == "e4m3" else torch.float4_e2m1fn_x2}
    offs = torch.tensor(_offsets(case, seed), dtype=torch.int32, device="cuda")
    if case["op"] == "step":
        x, w, go = _operands(case, seed)
        layer = kernels.MXFP8GroupedLinear(case["E"], case["K"], case["N"], device="cuda")
        with torch.no_grad():
            layer.weight.copy_(w)
        return {"op": "step", "layer": layer, "x": x.requires_grad_(), "go": go, "offs": offs}
    a, b = _operands(case, seed)
    sa, qa = _to_mx(a)
    sb, qb = _to_mx(b, case["weight"])
    return {"op": case["op"], "qa": qa, "sa": sa, "qb": qb, "sb": sb, "offs": offs, "out": _DTYPES[case["out"]]}


def run(state):
    """One pass."""
    s = state
    if s["op"] == "quantize":
        scales, data = kernels.to_mx(s["x"], s["elem"])
        return scales, data.view(torch.uint8)
    if s["op"] == "step":
        s["x"].grad = s["layer"].weight.grad = None
        out = s["layer"](s["x"], s["offs"])
        out.backward(s["go"])
        return out, s["x"].grad, s["layer"].weight.grad
    if s["op"] == "wgrad":
        return kernels.triton_mxfp8_wgrad(s["qa"], s["sa"], s["qb"], s["sb"], s["offs"], out_dtype=s["out"])
    return kernels.triton_mxfp8_grouped_mm(s["qa"], s["qb"], s["sa"], s["sb"], s["offs"], out_dtype=s["out"])


# --- what a case takes and gives ------------------------------------------


def work(case):
    """Bytes and operations the path cannot do without: each input read once,
    each output written once, two operations per multiply-add."""
    if case["op"] == "quantize":
        n = case["B"] * case["R"] * case["C"]
        q = 1 if case["elem"] == "e4m3" else 0.5
        return {"bytes": n * (_BYTES[case["src"]] + q + 1 / 32), "flops": 0}
    E, M, N, K, o = case["E"], case["M"], case["N"], case["K"], _BYTES[case["out"]]
    mx = 1 + 1 / 32
    if case["op"] == "forward":
        w = mx if case["weight"] == "e4m3" else 0.5 + 1 / 32
        used = sum(b > a for a, b in zip([0] + _offsets(case, 1), _offsets(case, 1)))   # experts that got tokens
        return {"bytes": M * K * mx + used * N * K * w + o * M * N, "flops": 2 * M * N * K}
    if case["op"] == "dgrad":
        return {"bytes": M * N * mx + E * N * K * mx + o * M * K, "flops": 2 * M * N * K}
    if case["op"] == "wgrad":
        return {"bytes": M * (N + K) * mx + o * E * N * K, "flops": 2 * M * N * K}
    # x, w and grad_out in; out, grad_x and grad_w out, all 16 bits
    return {"bytes": 2 * 2 * (M * K + E * N * K + M * N), "flops": 6 * M * N * K}


def tolerance(case):
    """Quantized bytes are exact.  A product with 32-bit sums differs between
    implementations by the order of its sums, and by one rounding to the
    output type where that tips: four times the distance to the 64-bit result,
    2**-8 at most per value in bf16 (1.7e-3 over the result), 2**-11 in f16
    (2.1e-4); an f32 result keeps the matrix unit's own sums (1.4e-5).  A
    weight gradient is rounded to bf16 whatever its output type is."""
    if case["op"] == "quantize":
        return "exact"
    if case["op"] == "wgrad" or case["out"] == "bf16":
        return {"rel": 7e-3, "max": 3.2e-2}
    if case["out"] == "f16":
        return {"rel": 8e-4, "max": 4e-3}
    return {"rel": 6e-5, "max": 1e-3}


def _grouped(a, b, offs):
    """out[s:e] = a[s:e] @ b[g]^T in float64."""
    out = torch.empty((a.shape[0], b.shape[1]), dtype=torch.float64, device=a.device)
    at = 0
    for g, end in enumerate(offs):
        if end > at:
            out[at:end] = a[at:end] @ b[g].t()
        at = end
    return out


def _grouped_w(a, b, offs):
    """out[g] = a[:, s:e] @ b[:, s:e]^T in float64."""
    out = torch.zeros((len(offs), a.shape[0], b.shape[0]), dtype=torch.float64, device=a.device)
    at = 0
    for g, end in enumerate(offs):
        if end > at:
            out[g] = a[:, at:end] @ b[:, at:end].t()
        at = end
    return out


def exact(case, seed):
    """What run() returns, from plain torch: the quantized bytes, or the
    products of the MX operands in 64 bits."""
    if case["op"] == "quantize":
        s, q = _to_mx(prepare(case, seed)["x"], case["elem"])
        return s, q.view(torch.uint8)
    offs = _offsets(case, seed)
    if case["op"] == "step":
        x, w, go = _operands(case, seed)

        def mx(t):
            return _dequant(*_to_mx(t.contiguous()))

        out = _grouped(mx(x), mx(w), offs)
        grad_x = _grouped(mx(go), mx(w.transpose(1, 2)), offs)
        return out, grad_x, _grouped_w(mx(go.t()), mx(x.t()), offs)
    a, b = _operands(case, seed)
    a, b = _dequant(*_to_mx(a)), _dequant(*_to_mx(b, case["weight"]), case["weight"])
    return _grouped_w(a, b, offs) if case["op"] == "wgrad" else _grouped(a, b, offs)
