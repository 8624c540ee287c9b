"""The workloads this framework's speed is measured on.

Each case is one pass through the public operators that mlx_amd.runtime.Context
offers: the quantized matmul of a linear layer (decode, small batches and
prefill, over bit widths, group sizes and data types), the same fused with an
output bias and activation, two of them in a row as a decode MLP, the
dequantizer, the quantizer, and the plugin ABI's dense f32 matmul.

listed() holds the named cases, draw() gives more of the same ranges, run()
does one pass on what prepare() laid out, and exact() is the same result in
64 bits from plain torch.  Inputs come from the seed alone, on the GPU.
"""
import ctypes
import math

import torch

from mlx_amd import abi
from mlx_amd.runtime import Context

DT = {"f32": abi.FLOAT32, "f16": abi.FLOAT16, "bf16": abi.BFLOAT16}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
ACT = {"none": abi.ACT_NONE, "relu": abi.ACT_RELU, "silu": abi.ACT_SILU, "gelu": abi.ACT_GELU}

# the largest listed product: drawn cases stay below it
MOST_MACS = 2048 * 4096 * 14336


def linear(name, M, K, N, bits, group, dtype, outliers=False, bias="", act="none"):
    return {"name": name, "op": "linear", "M": M, "K": K, "N": N, "bits": bits, "group": group, "dtype": dtype,
            "outliers": outliers, "bias": bias, "act": act}


def listed():
    return [
        # one token through a square 4-bit projection in f32, the reference
        # core's own tensor type: the smallest call, launch latency counts
        linear("decode_f32_m1", 1, 4096, 4096, 4, 64, "f32"),
        # one decoded token through a 4-bit MLP of an 8B-class model: up
        # projection with SiLU, then the down projection (long K)
        {"name": "decode_mlp_4bit_m1", "op": "mlp", "M": 1, "K": 4096, "N": 14336, "bits": 4, "group": 64, "dtype": "f16"},
        # eight decoded tokens (a small serving batch) through the same up projection
        linear("decode_4bit_m8", 8, 4096, 14336, 4, 64, "f16"),
        # one token, codes that straddle words, weights with outliers
        linear("decode_6bit_m1", 1, 4096, 11008, 6, 64, "f16", outliers=True),
        # a serving batch at the GEMV / GEMM crossover, 8-bit codes
        linear("batch_8bit_m32", 32, 8192, 8192, 8, 128, "bf16"),
        # a larger serving batch, 3-bit codes with outliers
        linear("batch_3bit_m64", 64, 4096, 11008, 3, 64, "f16", outliers=True),
        # the same square f32 projection as the first case for a batch of prompts
        linear("batch_f32_m64", 64, 4096, 4096, 4, 64, "f32"),
        # prefill of a whole 2048-token prompt, 4-bit: the largest call
        linear("prefill_4bit_m2048", 2048, 4096, 14336, 4, 64, "bf16"),
        # prefill of a prompt of odd length through a down projection whose K
        # is no power of two, 6-bit codes, with the fused bias and GELU
        linear("prefill_6bit_odd", 509, 11008, 4096, 6, 64, "f16", bias="f16", act="gelu"),
        # unpacking a weight matrix (weight export, or a dense library call after it)
        {"name": "dequantize_4bit", "op": "dequantize", "N": 14336, "K": 4096, "bits": 4, "group": 64, "dtype": "f16", "out": "f16"},
        # packing an f32 weight matrix at load time
        {"name": "quantize_4bit", "op": "quantize", "N": 14336, "K": 4096, "bits": 4, "group": 64, "dtype": "f16", "src": "f32"},
        # the plugin ABI's dense f32 matmul, ragged on every side
        {"name": "matmul_f32", "op": "matmul", "M": 1000, "K": 2000, "N": 3000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, group, lo, hi):
    """A row length: a multiple of 1024, 256 or 64 (the group where larger), as layers have them."""
    step = max(group, rng.choice([1024, 1024, 256, 64]))
    return max(1, round(_log(rng, lo, hi) / step)) * step


def draw(rng):
    op = rng.choices(["linear", "mlp", "dequantize", "quantize", "matmul"], [12, 1, 2, 2, 2])[0]
    if op == "matmul":
        return {"op": op, "M": _log(rng, 1, 2000), "K": _log(rng, 16, 4000), "N": _log(rng, 16, 4000)}
    group = rng.choice([32, 64, 64, 64, 128])
    bits = rng.choice([2, 3, 4, 4, 4, 5, 6, 8, 8])
    dtype = rng.choice(["f32", "f16", "f16", "bf16", "bf16"])
    if op in ("dequantize", "quantize"):
        c = {"op": op, "N": _log(rng, 100, 14336), "K": _width(rng, group, 256, 8192), "bits": bits, "group": group,
             "dtype": dtype}
        c["out" if op == "dequantize" else "src"] = rng.choice(["f32", "f16", "bf16"])
        return c
    K, N = _width(rng, group, 512, 14336), _log(rng, 256, 14336)
    if op == "mlp":
        return {"op": op, "M": rng.randint(1, 8), "K": min(K, 8192), "N": _width(rng, group, 1024, 14336),
                "bits": bits, "group": group, "dtype": dtype}
    M = _log(rng, 1, 2048 if dtype != "f32" else 128)
    M = max(1, min(M, MOST_MACS // (K * N)))
    bias = rng.choice(["", "", "", dtype])
    act = rng.choice(["relu", "silu", "gelu"]) if bias else "none"
    return {"op": op, "M": M, "K": K, "N": N, "bits": bits, "group": group, "dtype": dtype,
            "outliers": rng.random() < 0.25, "bias": bias, "act": act}


# --- the packed format, in plain torch ------------------------------------------------


def _weights(gen, N, K, outliers=False):
    """N(0, 0.02), with 1 % of the entries times 20 where asked."""
    w = torch.randn(N, K, generator=gen, device="cuda") * 0.02
    if outliers:
        w = torch.where(torch.rand(N, K, generator=gen, device="cuda") < 0.01, w * 20, w)
    return w


def _quantized(w, bits, group, dtype):
    """(codes int32 [N, K], scales, biases [N, K / group]): affine min / max groups."""
    N, K = w.shape
    g = w.view(N, K // group, group)
    lo, hi = g.amin(-1), g.amax(-1)
    levels = 2 ** bits - 1
    s, b = ((hi - lo) / levels).to(TORCH[dtype]), lo.to(TORCH[dtype])
    q = ((g - b.float()[..., None]) / s.float()[..., None]).round().clamp(0, levels)
    return q.to(torch.int32).view(N, K), s, b


def _packed(q, bits):
    """int32 [N, K * bits / 32]: row n's codes as a little-endian bit stream."""
    N, K = q.shape
    q = q.view(N, K // 32, 32)
    words = torch.zeros(N, K // 32, bits, dtype=torch.int64, device=q.device)
    for i in range(32):
        at, sh = divmod(i * bits, 32)
        code = q[..., i].to(torch.int64) << sh
        words[..., at] |= code & 0xFFFFFFFF
        if sh + bits > 32:
            words[..., at + 1] |= code >> 32
    return words.to(torch.int32).view(N, K * bits // 32)


def _dequantized(q, s, b, group):
    """The weights in 64 bits."""
    return torch.addcmul(b.double()[..., None], q.double().view(q.shape[0], -1, group), s.double()[..., None]).view(q.shape)


def _activated(y, act):
    if act == "relu":
        return torch.relu(y)
    if act == "silu":
        return torch.nn.functional.silu(y)
    if act == "gelu":
        return torch.nn.functional.gelu(y)
    return y


def _layer(gen, c, N, K):
    return _quantized(_weights(gen, N, K, c.get("outliers", False)), c["bits"], c["group"], c["dtype"])


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _inputs(case, seed):
    """What the path is given: torch tensors on the GPU, from the seed alone."""
    gen, c = _generator(seed), case
    randn = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    if c["op"] == "matmul":
        return {"a": randn(c["M"], c["K"]), "b": randn(c["K"], c["N"])}
    if c["op"] == "quantize":
        return {"w": _weights(gen, c["N"], c["K"]).to(TORCH[c["src"]])}
    if c["op"] == "dequantize":
        return {"layer": _layer(gen, c, c["N"], c["K"])}
    x = randn(c["M"], c["K"]).to(TORCH[c["dtype"]])
    if c["op"] == "mlp":
        return {"x": x, "up": _layer(gen, c, c["N"], c["K"]), "down": _layer(gen, c, c["K"], c["N"])}
    return {"x": x, "layer": _layer(gen, c, c["N"], c["K"]),
            "bias": randn(c["N"]).to(TORCH[c["bias"]]) if c["bias"] else None}


# --- device buffers ---------------------------------------------------------------------

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = Context(0)
    return _context


class _Array:
    """A plugin buffer, and a torch tensor over the same memory (`t`): the
    handle is the plugin's record of the buffer, whose first word is the
    device address.  The tensor keeps the buffer alive, and the last of the
    two to go frees it."""

    class _Owner:
        def __init__(self, buf, shape, typestr):
            self.buf = buf
            address = ctypes.c_void_p.from_address(buf.handle).value
            self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (address, False), "version": 2}

        def __del__(self):
            self.buf.free()

    def __init__(self, shape, dtype):
        shape = tuple(shape)
        size = torch.empty(0, dtype=dtype).element_size()
        self.buf = _ctx().alloc(math.prod(shape) * size)
        owner = self._Owner(self.buf, shape, {4: "<i4", 2: "<i2"}[size])
        self.t = torch.as_tensor(owner, device="cuda").view(dtype)


def _on_device(t):
    a = _Array(t.shape, t.dtype)
    _ctx().sync()  # the buffer's zero fill, before torch writes it
    a.t.copy_(t)
    return a


def _layer_on_device(layer, bits):
    q, s, b = layer
    return [_on_device(_packed(q, bits)), _on_device(s), _on_device(b)]


def prepare(case, seed):
    c, given = case, _inputs(case, seed)
    ctx = _ctx()
    dt = DT[c["dtype"]] if "dtype" in c else None
    if c["op"] == "matmul":
        a, b = _on_device(given["a"]), _on_device(given["b"])
        out = _Array((c["M"], c["N"]), torch.float32)
        keep, outs = [a, b, out], out.t
        calls = [(ctx.matmul_f32, (a.buf, b.buf, out.buf, c["M"], c["K"], c["N"]))]
    elif c["op"] == "quantize":
        w = _on_device(given["w"])
        wq = _Array((c["N"], c["K"] * c["bits"] // 32), torch.int32)
        s, b = (_Array((c["N"], c["K"] // c["group"]), TORCH[c["dtype"]]) for _ in range(2))
        keep, outs = [w, wq, s, b], {"w_q": wq.t, "scales": s.t, "biases": b.t}
        calls = [(ctx.quantize, (w.buf, wq.buf, s.buf, b.buf, c["N"], c["K"], c["group"], c["bits"], DT[c["src"]], dt))]
    elif c["op"] == "dequantize":
        keep = _layer_on_device(given["layer"], c["bits"])
        out = _Array((c["N"], c["K"]), TORCH[c["out"]])
        calls = [(ctx.dequantize, (*[a.buf for a in keep], out.buf, c["N"], c["K"], c["group"], c["bits"], dt, DT[c["out"]]))]
        keep, outs = keep + [out], out.t
    elif c["op"] == "mlp":
        x, h = _on_device(given["x"]), _Array((c["M"], c["N"]), TORCH[c["dtype"]])
        y = _Array((c["M"], c["K"]), TORCH[c["dtype"]])
        up, down = _layer_on_device(given["up"], c["bits"]), _layer_on_device(given["down"], c["bits"])
        calls = [(ctx.quantized_matmul_fused, (x.buf, *[a.buf for a in up], None, h.buf, c["M"], c["K"], c["N"],
                                               c["group"], c["bits"], dt, dt, dt, dt, ACT["silu"])),
                 (ctx.quantized_matmul, (h.buf, *[a.buf for a in down], y.buf, c["M"], c["N"], c["K"],
                                         c["group"], c["bits"], dt, dt, dt))]
        keep, outs = [x, h, y] + up + down, {"h": h.t, "y": y.t}
    else:
        x, layer = _on_device(given["x"]), _layer_on_device(given["layer"], c["bits"])
        y = _Array((c["M"], c["N"]), TORCH[c["dtype"]])
        shape = (c["M"], c["K"], c["N"], c["group"], c["bits"])
        ops = [a.buf for a in layer]
        keep, outs = [x, y] + layer, y.t
        if c["bias"]:
            bias = _on_device(given["bias"])
            keep.append(bias)
            calls = [(ctx.quantized_matmul_fused, (x.buf, *ops, bias.buf, y.buf, *shape, dt, dt, DT[c["bias"]], dt, ACT[c["act"]]))]
        else:
            calls = [(ctx.quantized_matmul, (x.buf, *ops, y.buf, *shape, dt, dt, dt))]
    ctx.sync()
    torch.cuda.synchronize()  # the plugin has a stream of its own
    return {"calls": calls, "outs": outs, "keep": keep}


def run(state):
    for op, args in state["calls"]:
        op(*args)
    return state["outs"]


# --- what a pass needs, and what it gives -----------------------------------------------


def _layer_bytes(c, N, K):
    return N * K * c["bits"] // 8 + 2 * N * (K // c["group"]) * SIZE[c["dtype"]]


def work(case):
    c = case
    if c["op"] == "matmul":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 4 * (M * K + K * N + M * N), "flops": 2 * M * K * N}
    if c["op"] == "quantize":
        return {"bytes": c["N"] * c["K"] * SIZE[c["src"]] + _layer_bytes(c, c["N"], c["K"]), "flops": 4 * c["N"] * c["K"]}
    if c["op"] == "dequantize":
        return {"bytes": c["N"] * c["K"] * SIZE[c["out"]] + _layer_bytes(c, c["N"], c["K"]), "flops": 2 * c["N"] * c["K"]}
    M, K, N = c["M"], c["K"], c["N"]
    if c["op"] == "mlp":
        return {"bytes": 2 * _layer_bytes(c, N, K) + M * (2 * K + 2 * N) * SIZE[c["dtype"]], "flops": 4 * M * K * N}
    extra = N * SIZE[c["bias"]] if c["bias"] else 0
    return {"bytes": _layer_bytes(c, N, K) + M * (K + N) * SIZE[c["dtype"]] + extra, "flops": 2 * M * K * N}


def tolerance(case):
    # dense f32: every sum runs in ascending k with a rounding per multiply
    # and add, as the reference's CPU backend does it; packing and unpacking
    # are defined to the bit
    if case["op"] in ("matmul", "quantize", "dequantize"):
        return "exact"
    # Measured against exact(): 2e-7 to 8e-7 of f32's sums, 2e-4 to 3e-4 in
    # f16, 1.7e-3 to 2.3e-3 in bf16 (the output's rounding and, where the
    # products run on the matrix cores, that of the dequantized weights).
    # Four times that, and a few units in the last place for one value.
    if case["dtype"] == "f32":
        return {"rel": 3e-6, "max": 4e-5}
    return {"rel": 1.2e-3, "max": 1e-2} if case["dtype"] == "f16" else {"rel": 9e-3, "max": 6e-2}


def exact(case, seed):
    c, given = case, _inputs(case, seed)
    if c["op"] == "matmul":
        return given["a"].double() @ given["b"].double()
    if c["op"] == "quantize":
        g = given["w"].double().view(c["N"], -1, c["group"])
        lo, hi = g.amin(-1), g.amax(-1)
        return {"w_q": None, "scales": (hi - lo) / (2 ** c["bits"] - 1), "biases": lo}
    if c["op"] == "dequantize":
        return _dequantized(*given["layer"], c["group"])
    x = given["x"].double()
    if c["op"] == "mlp":
        h = torch.nn.functional.silu(x @ _dequantized(*given["up"], c["group"]).t())
        return {"h": h, "y": h @ _dequantized(*given["down"], c["group"]).t()}
    y = x @ _dequantized(*given["layer"], c["group"]).t()
    if c["bias"]:
        y = y + given["bias"].double()
    return _activated(y, c["act"])
