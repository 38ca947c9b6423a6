"""Performance cases of the pack / mmt4d / unpack / conv_nchwc entry points.

Each case is a piece of work as a program on top of this library has it done,
through the public binding (`iree_amd.ukernel`) in its default state, on
operands resident in device memory:

  matmul    row-major A [M, K] times B ([N, K] or [K, N]) into row-major C:
            pack A, pack B, mmt4d, unpack. What a compiled program does with a
            matmul of two activations, and what the library's own headline
            chain does.
  layers    one pass of M rows (tokens) through `count` linear layers whose
            weights were packed when the model was loaded: per layer pack the
            activations, mmt4d, and the epilogue the program has chosen
            (unpack, the fused store into a row-major matrix, or the fused
            dequantizing store of quantized layers). Small M is decoding, large
            M prefill. Several layers, each with weights of its own, stand for
            a model's walk through its weights in decoding.
  relayout  a matrix brought into tiles and, where unpack has the type, back:
            what loading weights or handing over a large operand costs.
  conv      one convolution layer of an image network in the [N][C/c0][H][W][c0]
            layout.

`listed()` holds one case for each part of the range, `draw()` picks others
from the same ranges.
"""
from __future__ import annotations

import math

import torch

from iree_amd import ukernel as uk

# element type -> (mmt4d type flags, pack type of the operands, torch operand
# type, torch result type, bytes per operand element, unpack type of the result)
_TYPES = {
    "s8": (uk.MMT4D_TYPE_S8S8S32, uk.PACK_TYPE_I8I8, torch.int8, torch.int32, 1, uk.UNPACK_TYPE_I32I32),
    "s8s4": (uk.MMT4D_TYPE_S8S4S32 | uk.MMT4D_ALLOW_GENERIC_FALLBACK_TILE_FUNCTION, uk.PACK_TYPE_I8I8,
             torch.int8, torch.int32, 1, uk.UNPACK_TYPE_I32I32),
    "f16": (uk.MMT4D_TYPE_F16F16F32, uk.PACK_TYPE_F16F16, torch.float16, torch.float32, 2, uk.UNPACK_TYPE_F32F32),
    "bf16": (uk.MMT4D_TYPE_BF16BF16F32, uk.PACK_TYPE_BF16BF16, torch.bfloat16, torch.float32, 2,
             uk.UNPACK_TYPE_F32F32),
    # bf16 in and out with one rounding at the end, as bf16 models run
    "bf16bf16": (uk.MMT4D_TYPE_BF16BF16BF16 | uk.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, uk.PACK_TYPE_BF16BF16,
                 torch.bfloat16, torch.bfloat16, 2, uk.UNPACK_TYPE_BF16BF16),
    "f32": (uk.MMT4D_TYPE_F32F32F32, uk.PACK_TYPE_F32F32, torch.float32, torch.float32, 4, uk.UNPACK_TYPE_F32F32),
    "f8": (uk.MMT4D_TYPE_F8E4M3FNF8E4M3FNF32, uk.PACK_TYPE_I8I8, torch.uint8, torch.float32, 1,
           uk.UNPACK_TYPE_F32F32),
}
_RELAYOUT_TYPES = {
    "i8": (uk.PACK_TYPE_I8I8, None, torch.int8),
    "f16": (uk.PACK_TYPE_F16F16, uk.UNPACK_TYPE_F16F16, torch.float16),
    "f32": (uk.PACK_TYPE_F32F32, uk.UNPACK_TYPE_F32F32, torch.float32),
}


def listed():
    return [
        # The smallest: the size of a unit test or of a small head, the tile of the CPU library.
        dict(name="matmul_s8_small", kind="matmul", dtype="s8", m=100, n=70, k=96, m0=16, n0=16, k0=2, rhs="nk"),
        # An ordinary quantized product in the CPU library's tile.
        dict(name="matmul_s8_1024", kind="matmul", dtype="s8", m=1024, n=1024, k=1024, m0=16, n0=16, k0=2, rhs="nk"),
        # The benchmark's default chain.
        dict(name="matmul_f16_4096", kind="matmul", dtype="f16", m=4096, n=4096, k=4096, m0=16, n0=16, k0=16,
             rhs="nk"),
        # Nothing divides anything, right-hand side as linalg.matmul has it, the tile the query answers with.
        dict(name="matmul_bf16_ragged_kn", kind="matmul", dtype="bf16", m=1000, n=1501, k=777, m0=16, n0=16, k0=8,
             rhs="kn"),
        # f32 in the CPU library's tile, odd sizes.
        dict(name="matmul_f32_ragged_kn", kind="matmul", dtype="f32", m=515, n=1027, k=769, m0=16, n0=16, k0=1,
             rhs="kn"),
        # Decoding of a batch of 16 with 8-bit weights, up-projections of four layers, with bias accumulators.
        dict(name="decode_s8", kind="layers", dtype="s8", m=16, n=14336, k=4096, m0=32, n0=16, k0=8, count=4,
             epilogue="dequant", bias=True),
        # Decoding of one sequence with 4-bit weights, down-projections of four layers.
        dict(name="decode_s8s4", kind="layers", dtype="s8s4", m=1, n=4096, k=14336, m0=16, n0=16, k0=32, count=4,
             epilogue="dequant", bias=False),
        # A short prompt, bf16 in and out.
        dict(name="prefill_bf16_short", kind="layers", dtype="bf16bf16", m=200, n=4096, k=14336, m0=16, n0=16, k0=8,
             count=1, epilogue="fused", bias=False),
        # The largest: a long prompt in 8-bit floats.
        dict(name="prefill_f8_long", kind="layers", dtype="f8", m=2048, n=28672, k=8192, m0=16, n0=16, k0=32,
             count=1, epilogue="unpack", bias=False),
        # The large relayout, rows that are not 16-byte aligned, both directions.
        dict(name="relayout_f32_large", kind="relayout", dtype="f32", rows=12288, cols=12289, t0=16, t1=1,
             transpose="outer"),
        # A layer of an image network in training batch size ...
        dict(name="conv_3x3_batch", kind="conv", batch=16, ic=256, oc=256, oh=56, ow=56, f=3, stride=1),
        # ... and a late one for a single image.
        dict(name="conv_3x3_single", kind="conv", batch=1, ic=512, oc=512, oh=7, ow=7, f=3, stride=1),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# Tiles per type: the one iree_uk_query_tile_sizes_2d answers with (16-byte
# rows), a wider one where configurations use it, and the CPU library's.
_TILES = {"s8": [(16, 16, 16), (16, 16, 2), (32, 16, 8)], "s8s4": [(16, 16, 32), (16, 16, 16)],
          "f16": [(16, 16, 8), (16, 16, 16)], "bf16": [(16, 16, 8), (16, 16, 2)], "bf16bf16": [(16, 16, 8)],
          "f32": [(16, 16, 4), (16, 16, 1)], "f8": [(16, 16, 32), (16, 16, 16)]}
# The most multiply-adds a drawn case of a type has: what keeps it below the
# cost of the largest listed case.
_MOST = {"s8": 3e11, "s8s4": 2e11, "f16": 1.2e11, "bf16": 1.2e11, "bf16bf16": 1.2e11, "f32": 1e10, "f8": 3e11}


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "layers", "layers", "relayout", "conv"])
    if kind == "matmul":
        dtype = rng.choice(["s8", "f16", "bf16", "f32", "f8"])
        m0, n0, k0 = rng.choice(_TILES[dtype])
        m, n, k = (_log_int(rng, 64, 4096) for _ in range(3))
        while float(m) * n * k > _MOST[dtype]:
            m, n, k = (max(64, x * 3 // 4) for x in (m, n, k))
        return dict(kind=kind, dtype=dtype, m=m, n=n, k=k, m0=m0, n0=n0, k0=k0, rhs=rng.choice(["nk", "kn"]))
    if kind == "layers":
        dtype = rng.choice(["s8", "s8", "s8s4", "f16", "bf16bf16", "f8"])
        m0, n0, k0 = rng.choice(_TILES[dtype])
        m = _log_int(rng, 1, 2048)
        # Layer widths are multiples of 128 in practice.
        n, k = (128 * _log_int(rng, 8, 128) for _ in range(2))
        count = 4 if m <= 64 else 1
        while float(count) * m * n * k > _MOST[dtype]:
            m = max(1, m * 3 // 4)
        epilogue = rng.choice(["unpack", "dequant"] if dtype in ("s8", "s8s4") else ["unpack", "fused"])
        return dict(kind=kind, dtype=dtype, m=m, n=n, k=k, m0=m0, n0=n0, k0=k0, count=count, epilogue=epilogue,
                    bias=epilogue == "dequant" and rng.random() < 0.5)
    if kind == "relayout":
        dtype = rng.choice(["i8", "f16", "f32"])
        transpose = rng.choice(["none", "outer", "inner_outer"])
        t0, t1 = {"i8": [(16, 16), (16, 2)], "f16": [(16, 8), (16, 16)],
                  "f32": [(16, 4), (16, 1)]}[dtype][rng.randrange(2)]
        return dict(kind=kind, dtype=dtype, rows=_log_int(rng, 256, 12288), cols=_log_int(rng, 256, 12288), t0=t0,
                    t1=t1, transpose=transpose)
    size = _log_int(rng, 7, 112)
    ic, oc = (16 * _log_int(rng, 1, 32) for _ in range(2))
    f, stride = rng.choice([(1, 1), (3, 1), (3, 1), (3, 2), (7, 2)])
    batch = _log_int(rng, 1, 16)
    while float(batch) * size * size * ic * oc * f * f > 2.9e10:
        ic, oc = max(16, ic // 32 * 16), max(16, oc // 32 * 16)
    return dict(kind=kind, batch=batch, ic=ic, oc=oc, oh=size, ow=size, f=f, stride=stride)


# ------------------------------------------------------------------- inputs
def _operand(shape, dtype, weights, gen):
    """Random values of an operand: uniform bytes for quantized weights, a
    clipped normal for quantized activations, N(0, 1) for floats, scaled to the
    type's range for 8-bit floats."""
    if dtype in ("s8", "s8s4", "i8"):
        if weights:
            return torch.randint(-128, 128, shape, generator=gen, device="cuda", dtype=torch.int8)
        t = torch.randn(shape, generator=gen, device="cuda") * 40.0
        return t.round_().clamp_(-128, 127).to(torch.int8)
    t = torch.randn(shape, generator=gen, device="cuda")
    if dtype == "f8":
        t *= 448.0 / t.abs().max()
        return t.to(torch.float8_e4m3fn).view(torch.uint8)
    return t.to({"f16": torch.float16, "bf16": torch.bfloat16, "bf16bf16": torch.bfloat16, "f32": torch.float32}[dtype])


def _tiles(case):
    cd = lambda a, b: -(-a // b)  # noqa: E731
    return cd(case["m"], case["m0"]), cd(case["n"], case["n0"]), cd(case["k"], case["k0"])


def _pack_args(src, rows, cols, dst, tile0, tile1, flags):
    """Arguments of one pack call: a rows x cols row-major matrix into tiles
    that are tile0 x tile1 once transposed the way `flags` says."""
    s0, s1 = tile0, tile1
    if flags & uk.PACK_TRANSPOSE_INNER:
        s0, s1 = s1, s0
    o0, o1 = -(-rows // s0), -(-cols // s1)
    if flags & uk.PACK_TRANSPOSE_OUTER:
        o0, o1 = o1, o0
    return (src.data_ptr(), 0, cols, 1, dst.data_ptr(), 0, o1 * tile0 * tile1, tile0 * tile1, rows, cols, o0, o1,
            tile0, tile1, 0, flags)


def _prepare_matmul(case, gen):
    flags, pack, tin, tout, _, unpack = _TYPES[case["dtype"]]
    m, n, k, m0, n0, k0 = (case[x] for x in ("m", "n", "k", "m0", "n0", "k0"))
    m1, n1, k1 = _tiles(case)
    kn = case["rhs"] == "kn"
    a = _operand((m, k), case["dtype"], False, gen)
    b = _operand((k, n) if kn else (n, k), case["dtype"], True, gen)
    lhs = torch.empty(m1 * k1 * m0 * k0, dtype=tin, device="cuda")
    rhs = torch.empty(n1 * k1 * n0 * k0, dtype=tin, device="cuda")
    acc = torch.empty(m1 * n1 * m0 * n0, dtype=tout, device="cuda")
    out = torch.empty((m, n), dtype=tout, device="cuda")
    both = uk.PACK_TRANSPOSE_INNER | uk.PACK_TRANSPOSE_OUTER
    return {
        "keep": (a, b, lhs, rhs, acc), "out": out,
        "pack_a": _pack_args(a, m, k, lhs, m0, k0, pack),
        "pack_b": _pack_args(b, k, n, rhs, n0, k0, pack | both) if kn else _pack_args(b, n, k, rhs, n0, k0, pack),
        "mmt4d": (lhs.data_ptr(), 0, k1 * m0 * k0, rhs.data_ptr(), 0, k1 * n0 * k0, acc.data_ptr(), 0,
                  n1 * m0 * n0, m1, n1, k1, m0, n0, k0, flags),
        "unpack": (acc.data_ptr(), 0, n1 * m0 * n0, m0 * n0, out.data_ptr(), 0, n, 1, m1, n1, m0, n0, m, n, unpack),
    }


def _prepare_layers(case, gen):
    lib = uk.load()
    flags, pack, tin, tout, _, unpack = _TYPES[case["dtype"]]
    m, n, k, m0, n0, k0 = (case[x] for x in ("m", "n", "k", "m0", "n0", "k0"))
    m1, n1, k1 = _tiles(case)
    layers = []
    for _ in range(case["count"]):
        act = _operand((m, k), case["dtype"], False, gen)
        if case["dtype"] == "s8s4":  # two weights a byte, in tiles as a model file holds them
            rhs = torch.randint(-128, 128, (n1 * k1 * n0 * k0 // 2,), generator=gen, device="cuda", dtype=torch.int8)
        else:
            w = _operand((n, k), case["dtype"], True, gen)
            rhs = torch.empty(n1 * k1 * n0 * k0, dtype=tin, device="cuda")
            lib.pack(*_pack_args(w, n, k, rhs, n0, k0, pack))
        lhs = torch.empty(m1 * k1 * m0 * k0, dtype=tin, device="cuda")
        layer = {"pack": _pack_args(act, m, k, lhs, m0, k0, pack)}
        operands = (lhs.data_ptr(), 0, k1 * m0 * k0, rhs.data_ptr(), 0, k1 * n0 * k0)
        sizes = (m1, n1, k1, m0, n0, k0)
        if case["epilogue"] == "dequant":
            out = torch.empty((m, n), dtype=torch.float32, device="cuda")
            row = torch.rand(m, generator=gen, device="cuda") * 0.02 + 0.001
            col = torch.rand(n, generator=gen, device="cuda") * 0.02 + 0.001
            acc = None
            if case["bias"]:
                acc = torch.randint(-2 ** 15, 2 ** 15, (m1 * n1 * m0 * n0,), generator=gen, device="cuda",
                                    dtype=torch.int32)
            layer["dequant"] = (*operands, acc.data_ptr() if case["bias"] else None, 0, n1 * m0 * n0, out.data_ptr(),
                                0, n, m, n, row.data_ptr(), col.data_ptr(), *sizes,
                                flags | (uk.MMT4D_ACCUMULATE if case["bias"] else 0))
            layer["keep"] = (act, rhs, lhs, row, col, acc)
        elif case["epilogue"] == "fused":
            out = torch.empty((m, n), dtype=tout, device="cuda")
            layer["fused"] = (*operands, out.data_ptr(), 0, n, m, n, *sizes, flags)
            layer["keep"] = (act, rhs, lhs)
        else:
            acc = torch.empty(m1 * n1 * m0 * n0, dtype=tout, device="cuda")
            out = torch.empty((m, n), dtype=tout, device="cuda")
            layer["mmt4d"] = (*operands, acc.data_ptr(), 0, n1 * m0 * n0, *sizes, flags)
            layer["unpack"] = (acc.data_ptr(), 0, n1 * m0 * n0, m0 * n0, out.data_ptr(), 0, n, 1, m1, n1, m0, n0,
                               m, n, unpack)
            layer["keep"] = (act, rhs, lhs, acc)
        layer["out"] = out
        layers.append(layer)
    return {"layers": layers}


def _prepare_relayout(case, gen):
    pack, unpack, t = _RELAYOUT_TYPES[case["dtype"]]
    rows, cols, t0, t1 = case["rows"], case["cols"], case["t0"], case["t1"]
    flags = {"none": 0, "outer": uk.PACK_TRANSPOSE_OUTER,
             "inner_outer": uk.PACK_TRANSPOSE_INNER | uk.PACK_TRANSPOSE_OUTER}[case["transpose"]]
    src = _operand((rows, cols), case["dtype"], True, gen)
    s0, s1 = (t1, t0) if flags & uk.PACK_TRANSPOSE_INNER else (t0, t1)
    tiles = torch.empty(-(-rows // s0) * -(-cols // s1) * t0 * t1, dtype=t, device="cuda")
    args = _pack_args(src, rows, cols, tiles, t0, t1, pack | flags)
    state = {"keep": src, "tiles": tiles, "pack": args, "out": [tiles]}
    if unpack is not None:
        back = torch.empty((rows, cols), dtype=t, device="cuda")
        # The transposition flags of the two calls have the same values.
        state["unpack"] = (tiles.data_ptr(), 0, args[6], t0 * t1, back.data_ptr(), 0, cols, 1, args[10], args[11],
                           t0, t1, rows, cols, unpack | flags)
        state["out"].append(back)
    return state


def _conv_sizes(case):
    h = (case["oh"] - 1) * case["stride"] + case["f"]
    w = (case["ow"] - 1) * case["stride"] + case["f"]
    x = case["batch"] * case["ic"] * h * w
    return h, w, x, case["oc"] * case["ic"] * case["f"] ** 2, case["batch"] * case["oc"] * case["oh"] * case["ow"]


def _prepare_conv(case, gen):
    h, w, nx, nf, ny = _conv_sizes(case)
    c0 = k0 = 16
    ico, oco, f, oh, ow = case["ic"] // c0, case["oc"] // k0, case["f"], case["oh"], case["ow"]
    x = torch.randn(nx, generator=gen, device="cuda")
    flt = torch.randn(nf, generator=gen, device="cuda")
    y = torch.empty(ny, device="cuda")
    return {"keep": (x, flt), "out": y,
            "conv": (x.data_ptr(), 0, ico * h * w * c0, h * w * c0, w * c0, flt.data_ptr(), 0,
                     ico * f * f * c0 * k0, f * f * c0 * k0, f * c0 * k0, y.data_ptr(), 0, oco * oh * ow * k0,
                     oh * ow * k0, ow * k0, case["batch"], oco, oh, ow, ico, f, f, k0, c0, case["stride"],
                     case["stride"], 0x01)}


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    make = {"matmul": _prepare_matmul, "layers": _prepare_layers, "relayout": _prepare_relayout,
            "conv": _prepare_conv}[case["kind"]]
    state = make(case, gen)
    state["kind"] = case["kind"]
    state["lib"] = uk.load()
    return state


# ---------------------------------------------------------------- the passes
def run(state):
    lib, kind = state["lib"], state["kind"]
    if kind == "matmul":
        lib.pack(*state["pack_a"])
        lib.pack(*state["pack_b"])
        lib.mmt4d(*state["mmt4d"])
        lib.unpack(*state["unpack"])
        return state["out"]
    if kind == "layers":
        for layer in state["layers"]:
            lib.pack(*layer["pack"])
            if "dequant" in layer:
                lib.mmt4d_dequant_unpack(*layer["dequant"])
            elif "fused" in layer:
                lib.mmt4d_unpack(*layer["fused"])
            else:
                lib.mmt4d(*layer["mmt4d"])
                lib.unpack(*layer["unpack"])
        return [layer["out"] for layer in state["layers"]]
    if kind == "relayout":
        lib.pack(*state["pack"])
        if "unpack" in state:
            lib.unpack(*state["unpack"])
        return state["out"]
    lib.conv_nchwc(*state["conv"])
    return state["out"]


def work(case):
    """Bytes: every operand of every call read once and every result written
    once; the tiled operands are buffers of the caller's, so the calls hand
    them over in memory. Operations: those of the unpadded sizes."""
    kind = case["kind"]
    if kind == "conv":
        _, _, nx, nf, ny = _conv_sizes(case)
        return {"bytes": 4.0 * (nx + nf + ny),
                "flops": 2.0 * ny * case["ic"] * case["f"] ** 2}
    if kind == "relayout":
        es = {"i8": 1, "f16": 2, "f32": 4}[case["dtype"]]
        both = 1 if case["dtype"] == "i8" else 2
        return {"bytes": 2.0 * case["rows"] * case["cols"] * es * both, "flops": 0.0}
    m, n, k = case["m"], case["n"], case["k"]
    es = _TYPES[case["dtype"]][4]
    out = 2 if case["dtype"] == "bf16bf16" else 4
    if kind == "matmul":
        return {"bytes": 3.0 * (m * k + n * k) * es + 3.0 * m * n * out, "flops": 2.0 * m * n * k}
    weights = n * k * (0.5 if case["dtype"] == "s8s4" else es)
    results = {"unpack": 3, "fused": 1, "dequant": 2 if case["bias"] else 1}[case["epilogue"]]
    return {"bytes": case["count"] * (3.0 * m * k * es + weights + results * m * n * out),
            "flops": 2.0 * case["count"] * m * n * k}


def tolerance(case):
    """Integers and moved bytes are exact, dequantized integers too (the scales
    are applied in one fixed order). Floats: about four times the distance from
    the same product in float64 (2-norm). f32 sums: 4e-7 for f16 at K = 4096, 5e-7
    for f32 at K = 769, 9e-7 for the 3x3 convolution of 256 channels. 8-bit
    floats: 1.5e-5, how the matrix instruction aligns the terms it adds up at
    once. 16-bit results: 3.9e-5 from the rounded float64 product, the results
    that round the other way, which are one unit in the last place (2^-7) off."""
    if case["kind"] == "relayout" or case.get("dtype") in ("s8", "s8s4"):
        return "exact"
    return {"f8": {"rel": 6e-5}, "bf16bf16": {"rel": 1.6e-4, "max": 0.03}}.get(case.get("dtype"), {"rel": 4e-6})
