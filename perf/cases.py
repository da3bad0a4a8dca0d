"""What the performance of this library is measured on: twelve calls that its users make, and a
generator of further ones over the same ranges.

A case is a dict of plain values.  `kind` says which public entry points a pass goes through:

  linear  one call with packed operands: `entry` is gemm (int32 output), s32 (int32 with a bias),
          f32, f16 or bf16 (scaled outputs: row scales, column scales, and a bias where `bias`);
  static  a layer whose weights were converted once: per pass the activations are converted
          (fp6_convert) and multiplied (linear_fp6_converted, output type `entry`);
  block   the seven linear layers of one decoder block (four hidden x hidden, two ffn x hidden, one
          hidden x ffn) for m tokens, captured into a HIP graph once and replayed per pass, as a
          decode loop does;
  pack    int32 values -> packed s4 on the device;  unpack  the way back.

Activations are normal(0, 2) rounded and clamped to [-8, 7], weights uniform in [-8, 7].
"""
import math

import torch

import int4linear_amd as lib

OUT_DTYPE = {"gemm": torch.int32, "s32": torch.int32, "f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _linear(name, entry, m, n, k, bias=False):
    return {"name": name, "kind": "linear", "entry": entry, "m": m, "n": n, "k": k, "bias": bias}


def listed():
    return [
        # one token through a 4096 x 4096 projection, called eagerly: the smallest call a decode loop makes
        _linear("token 1x4096x4096", "gemm", 1, 4096, 4096),
        # a decode step of sixteen sequences: all linear layers of one block, replayed as a graph
        {"name": "block of 16 tokens", "kind": "block", "m": 16, "hidden": 4096, "ffn": 14336},
        # sixty-four sequences through the down projection, output in the next layer's type
        _linear("decode 64x4096x14336", "f16", 64, 4096, 14336),
        # logits of sixteen sequences over a large vocabulary: the longest weight stream
        _linear("logits 16x128256x8192", "f32", 16, 128256, 8192),
        # a short prompt, or a large decode batch, through the up projection
        _linear("chunk 128x14336x4096", "bf16", 128, 14336, 4096),
        # the smallest and a ragged shape of the validation suite
        _linear("square 1024", "gemm", 1024, 1024, 1024),
        _linear("ragged 1000x3000x4096", "s32", 1000, 3000, 4096, bias=True),
        # K a multiple of the packer's word only, all three sizes odd multiples of it or odd
        _linear("odd K 333x1111x4104", "bf16", 333, 1111, 4104, bias=True),
        # a prompt of 2048 tokens against weights converted when the model was loaded
        {"name": "prompt 2048x14336x4096", "kind": "static", "entry": "bf16", "m": 2048, "n": 14336, "k": 4096, "bias": False},
        # the square the headline figure is quoted on: the largest call
        _linear("square 8192", "gemm", 8192, 8192, 8192),
        # quantised activations of 2048 tokens to the packed layout, and packed weights back
        {"name": "pack 2048x4096", "kind": "pack", "m": 2048, "n": 4096},
        {"name": "unpack 4096x4096", "kind": "unpack", "m": 4096, "n": 4096},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _columns(rng, low, high):
    """A row count of W: half of them multiples of 64, as layers have them, the others anything."""
    n = _log_int(rng, low, high)
    return max(64, n // 64 * 64) if rng.random() < 0.5 else n


def _depth(rng, low, high):
    """K: mostly multiples of 256 or 128, some of 64 or of the packer's word of 8."""
    step = rng.choice([256, 256, 256, 256, 128, 128, 64, 8])
    return max(step, _log_int(rng, low, high) // step * step)


MOST_PRODUCTS = 8192 ** 3 // 2   # half the largest listed case's multiply-adds
MOST_WEIGHTS = 128256 * 8192 // 2


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["static", "block", "pack", "unpack"])
    if kind in ("pack", "unpack"):
        while True:
            m, n = _log_int(rng, 1, 8192), _log_int(rng, 64, 16384)
            if m * n <= 1 << 25:
                return {"kind": kind, "m": m, "n": n}
    if kind == "block":
        hidden = rng.choice([2048, 3072, 4096, 5120])
        return {"kind": kind, "m": _log_int(rng, 1, 64), "hidden": hidden, "ffn": rng.choice([5, 6, 7]) * hidden // 2 // 256 * 256}
    while True:
        if kind == "static":
            m, n, k = _log_int(rng, 256, 8192), _columns(rng, 1024, 16384), _depth(rng, 1024, 16384)
            entry = rng.choice(["s32", "f32", "f16", "bf16"])
        else:
            m, n, k = _log_int(rng, 1, 8192), _columns(rng, 128, 65536), _depth(rng, 256, 16384)
            entry = rng.choice(["gemm", "gemm", "s32", "f32", "f16", "bf16"])
        if m * n * k <= MOST_PRODUCTS and n * k <= MOST_WEIGHTS:
            return {"kind": kind, "entry": entry, "m": m, "n": n, "k": k, "bias": entry != "gemm" and rng.random() < 0.5}


# ---- inputs ------------------------------------------------------------------------------


def _weights(g, rows, k):
    """Packed uniform s4: every byte value equally likely is two independent uniform nibbles."""
    return torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, device="cuda", generator=g)


def _activation_values(g, rows, k):
    return torch.randn((rows, k), device="cuda", generator=g).mul_(2.0).round_().clamp_(-8, 7).to(torch.int32)


def _activations(g, rows, k):
    nibbles = (_activation_values(g, rows, k) & 0xF).to(torch.uint8)
    return (nibbles[:, 0::2] | (nibbles[:, 1::2] << 4)).contiguous()


def _scales(g, count):
    return torch.rand(count, device="cuda", generator=g).mul_(0.02).add_(0.001)


def _epilogue_operands(g, entry, m, n, bias):
    scaled = entry in ("f32", "f16", "bf16")
    return (torch.randint(-2000, 2000, (n,), dtype=torch.int32, device="cuda", generator=g) if bias else None,
            _scales(g, m) if scaled else None, _scales(g, n) if scaled else None)


def prepare(case, seed):
    lib.init()
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind, m = case["kind"], case["m"]
    if kind == "pack":
        n = case["n"]
        return {"case": case, "src": _activation_values(g, m, n), "dst": torch.empty((m, (n + 7) // 8), dtype=torch.int32, device="cuda")}
    if kind == "unpack":
        n = case["n"]
        words = torch.randint(-(1 << 31), 1 << 31, (m, (n + 7) // 8), dtype=torch.int64, device="cuda", generator=g).to(torch.int32)
        return {"case": case, "src": words, "dst": torch.empty((m, n), dtype=torch.int32, device="cuda")}
    if kind == "block":
        return _prepare_block(case, g)
    n, k, entry = case["n"], case["k"], case["entry"]
    state = {"case": case, "x": _activations(g, m, k), "w": _weights(g, n, k),
             "y": torch.empty((m, n), dtype=OUT_DTYPE[entry], device="cuda")}
    state["bias"], state["row_scale"], state["col_scale"] = _epilogue_operands(g, entry, m, n, case["bias"])
    if kind == "static":
        state["x_conv"] = torch.empty(lib.fp6_operand_bytes(m, k), dtype=torch.uint8, device="cuda")
        state["w_conv"] = torch.empty(lib.fp6_operand_bytes(n, k), dtype=torch.uint8, device="cuda")
        lib.fp6_convert(state["w"], state["w_conv"], n, k)
    return state


def _prepare_block(case, g):
    m, hidden, ffn = case["m"], case["hidden"], case["ffn"]
    x_hidden, x_ffn = _activations(g, m, hidden), _activations(g, m, ffn)
    layers = []
    for n, k in [(hidden, hidden)] * 4 + [(ffn, hidden)] * 2 + [(hidden, ffn)]:
        _, row_scale, col_scale = _epilogue_operands(g, "bf16", m, n, False)
        layers.append((x_hidden if k == hidden else x_ffn, _weights(g, n, k), row_scale, col_scale,
                       torch.empty((m, n), dtype=torch.bfloat16, device="cuda"), n, k))

    def step():
        for x, w, row_scale, col_scale, y, n, k in layers:
            lib.linear_bf16(x, w, None, row_scale, col_scale, y, m, n, k)

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return {"case": case, "layers": layers, "graph": graph, "y": [layer[4] for layer in layers]}


# ---- one pass ----------------------------------------------------------------------------


def run(state):
    case = state["case"]
    kind, m = case["kind"], case["m"]
    if kind == "block":
        state["graph"].replay()
        return state["y"]
    n = case["n"]
    if kind == "pack":
        lib.pack_device(state["src"], state["dst"], m, n)
        return state["dst"]
    if kind == "unpack":
        lib.unpack_device(state["src"], state["dst"], m, n)
        return state["dst"]
    k, entry, y = case["k"], case["entry"], state["y"]
    if kind == "static":
        lib.fp6_convert(state["x"], state["x_conv"], m, k)
        lib.linear_fp6_converted(state["x_conv"], state["w_conv"], state["bias"], state["row_scale"], state["col_scale"], y,
                                 entry, m, n, k)
    elif entry == "gemm":
        lib.gemm_s4s4s32(state["x"], state["w"], y, m, n, k)
    elif entry == "s32":
        lib.linear_s32(state["x"], state["w"], state["bias"], y, m, n, k)
    else:
        layer = {"f32": lib.linear_f32, "f16": lib.linear_f16, "bf16": lib.linear_bf16}[entry]
        layer(state["x"], state["w"], state["bias"], state["row_scale"], state["col_scale"], y, m, n, k)
    return y


# ---- what a pass cannot do without, and how exact it is ------------------------------------


def _layer_work(entry, m, n, k, bias, w_bytes_per_element=0.5):
    out = 2 if entry in ("f16", "bf16") else 4
    moved = m * k // 2 + n * k * w_bytes_per_element + m * n * out + (4 * n if bias else 0)
    if entry in ("f32", "f16", "bf16"):
        moved += 4 * (m + n)
    return moved, 2.0 * m * n * k


def work(case):
    kind, m = case["kind"], case["m"]
    if kind in ("pack", "unpack"):
        n = case["n"]
        return {"bytes": 4 * m * n + 4 * m * ((n + 7) // 8), "flops": 0}
    if kind == "block":
        hidden, ffn = case["hidden"], case["ffn"]
        parts = [_layer_work("bf16", m, n, k, False) for n, k in [(hidden, hidden)] * 4 + [(ffn, hidden)] * 2 + [(hidden, ffn)]]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    moved, flops = _layer_work(case["entry"], m, case["n"], case["k"], case["bias"], 0.75 if kind == "static" else 0.5)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """The integer sums are exact, and the interface fixes every rounding after them (one conversion
    to float32, one rounding per multiplication in the order written, one to the output type), so
    another correct implementation gives the same bits in every output type."""
    return "exact"
