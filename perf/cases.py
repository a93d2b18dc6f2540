"""The work a user of this framework has it do, as cases that can be timed: whole `.ttnn` programs through the runtime
(`submit` / `to_host`) and the kernel library's entry points on tensors that stay on the GPU.

listed() names one or two points of every family, draw() gives another point of the same ranges, prepare() makes what a
program has in hand before the call, run() is one pass, work() is what the pass cannot do without, tolerance() how far two
correct implementations of the same precision may lie apart.
"""
import math

import numpy as np
import torch

import __graft_entry__ as entry

entry.load_package()
from ttmlir_amd import harness, hip, programs, runtime as rt  # noqa: E402

# (hidden, query heads, kv heads, head dim, ffn) of the decoder layers: the configuration of the benchmark, and two smaller ones
LAYERS = [(4096, 32, 8, 128, 14336), (2048, 32, 8, 64, 8192), (1024, 8, 8, 128, 2816)]
WEIGHTS = {"bfp8": hip.BFP8B, "bfp4": hip.BFP4B, "bf16": hip.BF16}
FLOATS = {"f32": (hip.F32, torch.float32, 4), "bf16": (hip.BF16, torch.bfloat16, 2)}
TILE_BYTES = {"bfp8": 1088, "bfp4": 576, "bf16": 2048, "f32": 4096}


def listed():
    return [
        # one small operation from host tensors to a host tensor, layout changes on the device: what a single-op program
        # under test or the first call of a session is; all latency
        dict(name="matmul_program_256", kind="matmul_program", m=256, k=512, n=256),
        # one serving step of a decoder layer, 32 sequences at the end of a 2048-token context: the step's activations,
        # rotary rows and positions come from the host, caches and weights are resident, the result goes back.  The caches are
        # the runtime's own tensors, which a serving loop never reads back: the rows a step writes show in its result through
        # the attention over them, and attention_decode returns its caches whole
        dict(name="decode_step_32", kind="decode_step", layer=0, users=32, max_seq=2048, pos=2047),
        # the MLP block of a short prompt (or a chunk of a long one)
        dict(name="mlp_512", kind="mlp", layer=0, tokens=512),
        # a whole decoder layer over a 2048-token prompt: the largest call
        dict(name="prefill_layer_2048", kind="prefill_layer", layer=0, seq=2048),
        # a projection of a decode step (weight streaming) and of a prompt (matrix cores), with bias and activation
        dict(name="linear_32", kind="linear", m=32, k=4096, n=14336, weight="bfp8", act="gelu", bias=True),
        dict(name="linear_2048", kind="linear", m=2048, k=4096, n=14336, weight="bfp8", act="gelu", bias=True),
        # weights that were left in bf16, a token count that is no multiple of anything
        dict(name="linear_77_bf16", kind="linear", m=77, k=4096, n=4096, weight="bf16", act="", bias=False),
        # attention of a prompt, causal, grouped queries
        dict(name="attention_prefill_2048", kind="attention_prefill", batch=1, heads=32, kv_heads=8, seq=2048, dim=128, window=-1),
        # attention of a decode step: the new key and value rows go into the caches, then every user attends over its own
        # context length
        dict(name="attention_decode_32", kind="attention_decode", users=32, heads=32, kv_heads=8, max_seq=2048, dim=128, paged=False),
        # weights or cache contents into block float and back
        dict(name="bfp8_8192", kind="layout", format="bfp8", dtype="f32", batch=1, rows=8192, cols=8192),
        # tile order and back for a tensor whose extents are no multiples of the tile
        dict(name="tile_ragged", kind="layout", format="tile", dtype="bf16", batch=3, rows=1000, cols=3001),
        # the row-wise and element-wise operations between the projections
        dict(name="rms_norm_2048", kind="tile_op", op="rms_norm", dtype="bf16", rows=2048, cols=4096),
    ]


# ------------------------------------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A feature width: usually whole tiles, now and then not."""
    w = _log(rng, lo, hi)
    return w if rng.random() < 0.2 else max(32, w // 32 * 32)


def draw(rng):
    kind = rng.choice(["matmul_program", "decode_step", "mlp", "prefill_layer", "linear", "linear", "attention_prefill", "attention_decode",
                       "layout", "tile_op", "tile_op"])
    if kind == "matmul_program":
        return dict(kind=kind, m=_log(rng, 16, 1024), k=_log(rng, 32, 2048), n=_log(rng, 32, 1024))
    if kind == "decode_step":
        max_seq = 32 * _log(rng, 8, 64)
        return dict(kind=kind, layer=rng.randrange(3), users=_log(rng, 1, 32), max_seq=max_seq, pos=rng.randrange(max_seq // 2, max_seq))
    if kind == "mlp":
        return dict(kind=kind, layer=rng.randrange(3), tokens=_log(rng, 1, 1024))
    if kind == "prefill_layer":
        return dict(kind=kind, layer=rng.randrange(3), seq=_log(rng, 64, 2047))
    if kind == "linear":
        return dict(kind=kind, m=_log(rng, 1, 2048), k=_width(rng, 512, 8192), n=_width(rng, 512, 14336),
                    weight=rng.choice(["bfp8", "bfp8", "bfp4", "bf16"]), act=rng.choice(["", "gelu", "silu"]), bias=rng.random() < 0.5)
    if kind == "attention_prefill":
        heads, kv = rng.choice([(32, 8), (32, 32), (16, 4), (8, 8)])
        seq = _log(rng, 64, 4096)
        return dict(kind=kind, batch=rng.choice([1, 1, 2, 4]), heads=heads, kv_heads=kv, seq=seq, dim=rng.choice([64, 128]),
                    window=rng.choice([-1, -1, -1, max(32, seq // 8)]))
    if kind == "attention_decode":
        heads, kv = rng.choice([(32, 8), (32, 8), (16, 4), (8, 8)])
        return dict(kind=kind, users=_log(rng, 1, 32), heads=heads, kv_heads=kv, max_seq=64 * _log(rng, 4, 64), dim=rng.choice([64, 128]),
                    paged=rng.random() < 0.3)
    if kind == "layout":
        return dict(kind=kind, format=rng.choice(["tile", "bfp8", "bfp4"]), dtype=rng.choice(["f32", "bf16"]), batch=rng.choice([1, 1, 2, 3]),
                    rows=_log(rng, 32, 4096), cols=_width(rng, 64, 8192))
    return dict(kind=kind, op=rng.choice(["rms_norm", "softmax", "sum", "add", "gelu"]), dtype=rng.choice(["f32", "bf16"]),
                rows=_log(rng, 32, 8192), cols=_width(rng, 128, 8192))


# ------------------------------------------------------------------------------------------------ inputs
_device = None


def _dev():
    """The process's runtime device, opened once."""
    global _device
    if _device is None:
        _device = rt.open_mesh_device()
    return _device


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(dtype)


def _tiles(x):
    """The TILE image of a row-major device tensor, as a flat tensor of the padded extent."""
    x = x if x.dim() > 1 else x.reshape(1, -1)
    rows, cols = x.shape[-2:]
    batch = x.numel() // (rows * cols)
    out = torch.empty(batch * (-(-rows // 32) * 32) * (-(-cols // 32) * 32), dtype=x.dtype, device=x.device)
    hip.call("ttm_tilize", hip.ptr(x.contiguous()), hip.ptr(out), batch, rows, cols, x.element_size(), hip.current_stream())
    return out


def _zero_tiles(batch, rows, cols, dtype):
    return torch.zeros(batch * (-(-rows // 32) * 32) * (-(-cols // 32) * 32), dtype=dtype, device="cuda")


def _count_tiles(rows, cols):
    return -(-rows // 32) * -(-cols // 32)


def _resident(binary, program, tensors, first=0):
    """Tensors in the layouts the program's inputs ask for, kept across calls."""
    return [rt.to_layout(rt.from_torch(t.cpu()), _dev(), rt.get_layout(binary, program, first + i), retain=True) for i, t in enumerate(tensors)]


def _matmul_program(m, k, n):
    pb = rt.ProgramBuilder()
    DT, TL, ST = rt.DataType, rt.TensorLayout, rt.StorageType
    pb.begin_program("matmul")
    a, b = pb.input((m, k), DT.BFloat16, TL.RowMajor, ST.Host), pb.input((k, n), DT.BFloat16, TL.RowMajor, ST.Host)
    c = pb.matmul(pb.to_layout(pb.to_device(a), TL.Tile), pb.to_layout(pb.to_device(b), TL.Tile))
    pb.output(pb.from_device(pb.to_layout(c, TL.RowMajor)))
    pb.end_program()
    return pb.finish()


def _layer_weights(g, layer):
    hidden, heads, kv, dim, ffn = LAYERS[layer]
    norm = lambda: (1.0 + 0.02 * torch.randn((hidden,), generator=g, device="cuda")).to(torch.bfloat16)
    mat = lambda a, b: _randn(g, (a, b), 0.02)
    return [norm(), mat(hidden, heads * dim), mat(hidden, kv * dim), mat(hidden, kv * dim), mat(heads * dim, hidden), norm(),
            mat(hidden, ffn), mat(hidden, ffn), mat(ffn, hidden)]


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = dict(case)
    if kind == "matmul_program":
        s["binary"] = rt.Binary.load_from_memory(_matmul_program(case["m"], case["k"], case["n"]))
        s["inputs"] = [_randn(g, (case["m"], case["k"])).cpu(), _randn(g, (case["k"], case["n"])).cpu()]
        _dev()
    elif kind == "decode_step":
        hidden, heads, kv, dim, ffn = LAYERS[case["layer"]]
        users, max_seq, pos = case["users"], case["max_seq"], case["pos"]
        s["binary"] = binary = rt.Binary.load_from_memory(programs.decode_layer(users, hidden, heads, kv, dim, ffn, max_seq, trace=True))
        s["main"] = binary.get_num_programs() - 1
        angle = pos * 10000.0 ** (-torch.arange(0, dim, 2, device="cuda") / dim).repeat(2).reshape(1, 1, 1, dim)
        # what a step brings along: token activations, the rotary rows of the position, the position
        s["step"] = [_randn(g, (users, hidden)).cpu(), angle.cos().to(torch.bfloat16).cpu(), angle.sin().to(torch.bfloat16).cpu(),
                     torch.tensor([pos], dtype=torch.int32), torch.full((users,), pos, dtype=torch.int32)]
        caches = [_randn(g, (users, kv, max_seq, dim)) for _ in range(2)]
        s["resident"] = _resident(binary, s["main"], caches + _layer_weights(g, case["layer"]), first=5)
    elif kind == "mlp":
        hidden, _, _, _, ffn = LAYERS[case["layer"]]
        s["binary"] = binary = rt.Binary.load_from_memory(programs.c4_mlp(case["tokens"], hidden, ffn))
        w = _layer_weights(g, case["layer"])
        s["main"], s["resident"] = 1, _resident(binary, 1, [_randn(g, (case["tokens"], hidden))] + w[5:])
    elif kind == "prefill_layer":
        hidden, heads, kv, dim, ffn = LAYERS[case["layer"]]
        s["binary"] = binary = rt.Binary.load_from_memory(programs.c5_decoder(case["seq"], hidden, heads, kv, dim, ffn))
        s["main"], s["resident"] = 1, _resident(binary, 1, [_randn(g, (1, case["seq"], hidden))] + _layer_weights(g, case["layer"]))
    elif kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        s["a"] = _tiles(_randn(g, (m, k)))
        w = _randn(g, (k, n), 0.02, torch.float32)
        if case["weight"] == "bf16":
            s["w"] = _tiles(w.to(torch.bfloat16))
        else:
            s["w"] = torch.empty(_count_tiles(k, n) * TILE_BYTES[case["weight"]], dtype=torch.uint8, device="cuda")
            hip.call("ttm_bfp_pack", hip.ptr(w), hip.F32, hip.ROW_MAJOR, hip.ptr(s["w"]), WEIGHTS[case["weight"]], 1, k, n, hip.current_stream())
        s["b"] = _tiles(_randn(g, (n,), 0.02)) if case["bias"] else None
        s["out"] = _zero_tiles(1, m, n, torch.bfloat16)
    elif kind == "attention_prefill":
        b, h, kv, seq, dim = (case[x] for x in ("batch", "heads", "kv_heads", "seq", "dim"))
        s["q"], s["k"], s["v"] = (_tiles(_randn(g, (b, n, seq, dim))) for n in (h, kv, kv))
        s["out"] = torch.zeros_like(s["q"])
    elif kind == "attention_decode":
        users, h, kv, max_seq, dim = (case[x] for x in ("users", "heads", "kv_heads", "max_seq", "dim"))
        block = 64
        if case["paged"]:     # every user's pages lie anywhere in the pool
            shape = (users * (max_seq // block), kv, block, dim)
            order = torch.randperm(shape[0], generator=g, device="cuda")
            s["pages"] = order.reshape(users, max_seq // block).to(torch.int32)
        else:
            shape, s["pages"] = (users, kv, max_seq, dim), None
        s["k"], s["v"] = _tiles(_randn(g, shape)), _tiles(_randn(g, shape))
        s["q"], s["k_new"], s["v_new"] = (_tiles(_randn(g, (users, n, dim))) for n in (h, kv, kv))
        # context lengths between a quarter of the cache and all of it
        s["cur"] = torch.randint(max_seq // 4, max_seq, (users,), generator=g, device="cuda").to(torch.int32)
        s["out"] = torch.zeros_like(s["q"])
    elif kind == "layout":
        _, dtype, _ = FLOATS[case["dtype"]]
        shape = (case["batch"], case["rows"], case["cols"])
        x = _randn(g, shape, 1.0, torch.float32)
        # a few large values among many small ones, as trained weights and activations have
        x = torch.where(torch.rand(shape, generator=g, device="cuda") < 0.01, x * 100.0, x)
        s["x"] = x.to(dtype)
        tiles = case["batch"] * _count_tiles(case["rows"], case["cols"])
        if case["format"] == "tile":
            s["packed"] = _zero_tiles(case["batch"], case["rows"], case["cols"], dtype)
        else:
            s["packed"] = torch.empty(tiles * TILE_BYTES[case["format"]], dtype=torch.uint8, device="cuda")
        s["back"] = torch.empty_like(s["x"])
    elif kind == "tile_op":
        _, dtype, _ = FLOATS[case["dtype"]]
        rows, cols = case["rows"], case["cols"]
        s["x"] = _tiles(_randn(g, (rows, cols), 1.0, dtype))
        s["w"] = _tiles(1.0 + _randn(g, (cols,), 0.02, dtype)) if case["op"] == "rms_norm" else None
        s["y"] = _tiles(_randn(g, (rows, cols), 1.0, dtype)) if case["op"] == "add" else None
        s["shape"] = np.array([rows, cols], dtype=np.int64)
        s["out"] = _zero_tiles(1, rows, 1 if case["op"] == "sum" else cols, dtype)
    else:
        raise ValueError("unknown kind %r" % kind)
    torch.cuda.synchronize()     # the runtime has a stream of its own
    return s


# ------------------------------------------------------------------------------------------------ one pass
def run(s):
    kind = s["kind"]
    if kind == "matmul_program":
        return harness.execute(s["binary"], 0, s["inputs"], device=_dev())[0]
    if kind == "decode_step":
        # new host tensors in every step, as a serving loop makes them; the result lives in the trace's own output slot
        step = [rt.from_torch(t) for t in s["step"]]
        (out,) = rt.submit(_dev(), s["binary"], s["main"], step + s["resident"])
        return rt.to_torch(rt.to_host(out, untilize=True)[0])
    if kind in ("mlp", "prefill_layer"):
        # device tensors are opaque handles: a program's result is read with to_host
        (out,) = rt.submit(_dev(), s["binary"], s["main"], s["resident"])
        host = rt.to_host(out, untilize=True)[0]
        rt.deallocate_tensor(out, force=True)
        return rt.to_torch(host)
    stream = hip.current_stream()
    if kind == "linear":
        hip.call("ttm_linear", hip.ptr(s["a"]), hip.BF16, hip.ptr(s["w"]), WEIGHTS[s["weight"]], 0, hip.ptr(s["b"]) if s["bias"] else None,
                 hip.BF16, hip.TILE, hip.ptr(s["out"]), hip.BF16, 1, 1, s["m"], s["n"], s["k"], hip.ACT[s["act"]], stream)
        return s["out"]
    if kind == "attention_prefill":
        hip.call("ttm_sdpa_windowed", hip.ptr(s["q"]), hip.ptr(s["k"]), hip.ptr(s["v"]), None, 1, 1, hip.ptr(s["out"]), hip.BF16, s["batch"],
                 s["heads"], s["kv_heads"], s["seq"], s["seq"], s["dim"], 1, 0.0, 0, s["window"], None, stream)
        return s["out"]
    if kind == "attention_decode":
        users, kv, max_seq, dim = s["users"], s["kv_heads"], s["max_seq"], s["dim"]
        block = 64 if s["paged"] else max_seq
        blocks, pages, table = users * (max_seq // block), max_seq // block, hip.ptr(s["pages"]) if s["paged"] else None
        cur = hip.ptr(s["cur"])
        for cache, new in ((s["k"], s["k_new"]), (s["v"], s["v_new"])):
            hip.call("ttm_paged_update_cache", hip.ptr(cache), hip.ptr(new), cur, table, hip.BF16, blocks, kv, block, dim, users,
                     pages if s["paged"] else 0, 0, stream)
        hip.call("ttm_sdpa_decode", hip.ptr(s["q"]), hip.ptr(s["k"]), hip.ptr(s["v"]), cur, None, 1, table, pages if s["paged"] else 0,
                 block if s["paged"] else 0, blocks if s["paged"] else 0, hip.ptr(s["out"]), hip.BF16, users, s["heads"], kv, max_seq, dim, 1,
                 0.0, stream)
        return s["out"], s["k"], s["v"]
    if kind == "layout":
        code, _, size = FLOATS[s["dtype"]]
        x, packed, back = hip.ptr(s["x"]), hip.ptr(s["packed"]), hip.ptr(s["back"])
        batch, rows, cols = s["batch"], s["rows"], s["cols"]
        if s["format"] == "tile":
            hip.call("ttm_tilize", x, packed, batch, rows, cols, size, stream)
            hip.call("ttm_untilize", packed, back, batch, rows, cols, size, stream)
        else:
            fmt = WEIGHTS[s["format"]]
            hip.call("ttm_bfp_pack", x, code, hip.ROW_MAJOR, packed, fmt, batch, rows, cols, stream)
            hip.call("ttm_bfp_unpack", packed, fmt, back, code, hip.ROW_MAJOR, batch, rows, cols, stream)
        return s["packed"], s["back"]
    code = FLOATS[s["dtype"]][0]
    x, out, rows, cols = hip.ptr(s["x"]), hip.ptr(s["out"]), s["rows"], s["cols"]
    if s["op"] == "rms_norm":
        hip.call("ttm_rms_norm", x, hip.ptr(s["w"]), hip.TILE, None, hip.TILE, out, code, 1, rows, cols, 1e-5, stream)
    elif s["op"] == "softmax":
        hip.call("ttm_softmax_lastdim", x, out, code, 1, rows, cols, stream)
    elif s["op"] == "sum":
        hip.call("ttm_reduce_lastdim", programs.REDUCE["sum"], x, out, code, 1, rows, cols, stream)
    elif s["op"] == "add":
        shape = s["shape"].ctypes.data
        hip.call("ttm_eltwise_binary", programs.BINARY["add"], x, shape, hip.ptr(s["y"]), shape, out, shape, 2, code, hip.TILE, stream)
    else:
        hip.call("ttm_eltwise_unary", programs.UNARY["gelu"], x, out, code, hip.TILE, 1, rows, cols, 0.0, stream)
    return s["out"]


# ------------------------------------------------------------------------------------------------ what a pass is worth
def _layer_weight_bytes(layer, mlp_only=False):
    hidden, heads, kv, dim, ffn = LAYERS[layer]
    bfp8 = _count_tiles(hidden, ffn) * 2
    if not mlp_only:
        bfp8 += 2 * _count_tiles(hidden, heads * dim) + 2 * _count_tiles(hidden, kv * dim)
    return bfp8 * TILE_BYTES["bfp8"] + _count_tiles(ffn, hidden) * TILE_BYTES["bfp4"] + 2 * hidden * (1 if mlp_only else 2)


def _layer_flops(layer, tokens, mlp_only=False):
    hidden, heads, kv, dim, ffn = LAYERS[layer]
    return 2.0 * tokens * hidden * (3 * ffn + (0 if mlp_only else (2 * heads + 2 * kv) * dim))


def work(case):
    kind = case["kind"]
    if kind == "matmul_program":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 2 * (m * k + k * n + m * n), "flops": 2.0 * m * k * n}
    if kind == "decode_step":
        hidden, heads, kv, dim, _ = LAYERS[case["layer"]]
        users, keys = case["users"], case["pos"] + 1
        return {"bytes": _layer_weight_bytes(case["layer"]) + 4 * users * kv * keys * dim + 4 * users * hidden,
                "flops": _layer_flops(case["layer"], users) + 4.0 * users * heads * keys * dim}
    if kind == "mlp":
        return {"bytes": _layer_weight_bytes(case["layer"], True) + 4 * case["tokens"] * LAYERS[case["layer"]][0],
                "flops": _layer_flops(case["layer"], case["tokens"], True)}
    if kind == "prefill_layer":
        hidden, heads, _, dim, _ = LAYERS[case["layer"]]
        seq = case["seq"]
        return {"bytes": _layer_weight_bytes(case["layer"]) + 4 * seq * hidden,
                "flops": _layer_flops(case["layer"], seq) + 4.0 * heads * dim * (seq * (seq + 1) // 2)}
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 2 * (m * k + m * n) + _count_tiles(k, n) * TILE_BYTES[case["weight"]] + (2 * n if case["bias"] else 0),
                "flops": 2.0 * m * k * n}
    if kind == "attention_prefill":
        b, h, kv, seq, dim, window = (case[x] for x in ("batch", "heads", "kv_heads", "seq", "dim", "window"))
        w = seq if window < 0 else min(window, seq)
        pairs = w * (w + 1) // 2 + (seq - w) * w
        return {"bytes": 2 * b * seq * dim * (2 * h + 2 * kv), "flops": 4.0 * b * h * pairs * dim}
    if kind == "attention_decode":
        users, h, kv, max_seq, dim = (case[x] for x in ("users", "heads", "kv_heads", "max_seq", "dim"))
        keys = users * max_seq * 5 // 8       # the mean context length is five eighths of the cache
        return {"bytes": 4 * keys * kv * dim + 4 * users * (h + 2 * kv) * dim, "flops": 4.0 * keys * h * dim}
    if kind == "layout":
        size = FLOATS[case["dtype"]][2]
        packed = case["batch"] * _count_tiles(case["rows"], case["cols"]) * TILE_BYTES[case["dtype"] if case["format"] == "tile" else case["format"]]
        return {"bytes": 2 * (case["batch"] * case["rows"] * case["cols"] * size + packed), "flops": 0}
    size, n = FLOATS[case["dtype"]][2], case["rows"] * case["cols"]
    reads = 2 if case["op"] == "add" else 1
    return {"bytes": size * (n * reads + (case["rows"] if case["op"] == "sum" else n)), "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "layout":
        return "exact"
    if kind == "tile_op" and case["dtype"] == "f32":
        return {"rel": 1e-5}
    return {"rel": 1e-2}      # bf16 operands and results, fp32 accumulation
