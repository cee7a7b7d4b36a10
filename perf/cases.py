"""What a user of this framework has it do, as measured cases: whole networks resident on the device, networks loaded
from a kmodel file and fed from host memory, decode steps of a language model, and the single operators of the C ABI on
device buffers and (through `nncase_amd.kernels`) on host arrays.

Every case has a "kind"; the ranges a kind stands for are those of its branch of draw().  Models, weights and model files
are made once per process and shared (a user's program has them on disk); what the seed decides is the data.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from nncase_amd import kernels, kmodel, llm, quant
from nncase_amd import netbuilder as nb
from nncase_amd import runtime as rt
from nncase_amd.runtime import Context, qp

FULL = (-rt.FLT_MAX, rt.FLT_MAX)
TORCH = {"u8": torch.uint8, "i8": torch.int8, "i16": torch.int16, "i32": torch.int32, "f16": torch.float16, "f32": torch.float32}
NUMPY = {"u8": np.uint8, "i8": np.int8, "i16": np.int16, "i32": np.int32, "f16": np.float16, "f32": np.float32}
CODE = {k: rt.NP_TO_DT[np.dtype(v)] for k, v in NUMPY.items()}
SIZE = {k: np.dtype(v).itemsize for k, v in NUMPY.items()}


def listed():
    return [
        # one camera image classified with everything resident: the latency of a chain of short launches
        {"name": "classify one image", "kind": "net", "model": "mobilenet_v2", "hw": 224, "batch": 1},
        # the same network as a server batches it, at the size the benchmark is quoted on
        {"name": "classify a batch", "kind": "net", "model": "mobilenet_v2", "hw": 224, "batch": 64},
        # detection at the benchmark's resolution and batch: dense 3x3 layers, concats, three f32 heads
        {"name": "detect in a batch", "kind": "net", "model": "yolov5s", "hw": 640, "batch": 16},
        # what an nncase program does: a kmodel file loaded once, then host image in, host detections out, one at a time
        {"name": "kmodel, host image", "kind": "kmodel", "model": "yolov5s", "hw": 640, "batch": 1},
        # one generated token for 32 conversations, recorded as two lanes like the benchmark
        {"name": "decode 32 sequences", "kind": "decode", "layers": 24, "batch": 32, "ctx": 2048, "vocab": 151936, "lanes": 2},
        # one generated token for a single user: nothing to share the weights' trip with
        {"name": "decode one sequence", "kind": "decode", "layers": 24, "batch": 1, "ctx": 700, "vocab": 151936, "lanes": 1},
        # attention alone over many long contexts with the head geometry of larger models
        {"name": "attention, long contexts", "kind": "attention", "batch": 48, "q_heads": 32, "kv_heads": 8, "head_dim": 128,
         "ctx": 6000, "out": "f16"},
        # a large product whose sides fit no tile, result as float32
        {"name": "matmul, ragged", "kind": "matmul", "m": 5000, "k": 3000, "n": 2100, "out": "f32"},
        # a strided 3x3 layer with channel counts that are no multiple of anything, as in pruned networks
        {"name": "conv, odd channels", "kind": "conv", "batch": 6, "hw": 77, "cin": 90, "cout": 203, "k": 3, "stride": 2,
         "depthwise": False, "out": "u8"},
        # activations handed from a float16 part of a graph to a quantised one
        {"name": "quantize a tensor", "kind": "cast", "count": 25_000_001, "src": "f16", "dst": "u8"},
        # a feature map brought into channel-blocked form for another module, channels that fill no block
        {"name": "pack channels", "kind": "layout", "op": "pack", "batch": 24, "c": 75, "hw": 80, "lanes": 32, "dtype": "f16"},
        # the drop-in kernel call on host tensors: operands up, one convolution, result down
        {"name": "host conv2d call", "kind": "host", "op": "conv2d", "batch": 1, "hw": 28, "c": 96, "n": 128, "k": 3, "out": "u8"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["net", "net", "kmodel", "decode", "decode", "attention", "matmul", "conv", "cast", "layout", "host"])
    case = {"kind": kind}
    if kind in ("net", "kmodel"):
        most = {"net": (64, 16), "kmodel": (16, 4)}[kind]
        if rng.random() < 0.5:
            case.update(model="mobilenet_v2", hw=rng.randint(96, 224), batch=_log(rng, 1, most[0]))
        else:
            case.update(model="yolov5s", hw=32 * rng.randint(8, 20), batch=_log(rng, 1, most[1]))
    elif kind == "decode":
        lanes = rng.choice([1, 2])
        case.update(layers=rng.randint(4, 24), batch=max(1, _log(rng, 1, 64) // lanes) * lanes, ctx=_log(rng, 64, 2048),
                    vocab=rng.choice([32000, 151936]), lanes=lanes)
    elif kind == "attention":
        q, kv, d = rng.choice([(14, 2, 64), (12, 12, 64), (32, 8, 128), (28, 4, 128)])
        ctx = _log(rng, 64, 16000)
        case.update(batch=_log(rng, 1, max(1, min(256, 1_500_000_000 // (ctx * kv * d * 4)))), q_heads=q, kv_heads=kv, head_dim=d,
                    ctx=ctx, out=rng.choice(["f16", "f32"]))
    elif kind == "matmul":
        case.update(m=_log(rng, 1, 32768), k=_log(rng, 64, 4096), n=_log(rng, 64, 4096), out=rng.choice(["f32", "u8"]))
    elif kind == "conv":
        depthwise, hw = rng.random() < 0.3, rng.randint(7, 160)
        cin = _log(rng, 8, 640)
        case.update(batch=_log(rng, 1, max(1, min(64, 100_000_000 // (hw * hw * 640)))), hw=hw, cin=cin, cout=cin if depthwise else _log(rng, 8, 640),
                    k=rng.choice([1, 3, 3, 5]), stride=rng.choice([1, 1, 2]), depthwise=depthwise, out=rng.choice(["u8", "u8", "f32"]))
    elif kind == "cast":
        src, dst = rng.choice([("f32", "u8"), ("f16", "u8"), ("f32", "i8"), ("f32", "i16"), ("u8", "f32"), ("u8", "f16"), ("i32", "f32")])
        case.update(count=_log(rng, 1000, 100_000_000), src=src, dst=dst)
    elif kind == "layout":
        hw, c, dtype = rng.randint(7, 224), _log(rng, 3, 512), rng.choice(["u8", "f16", "f32"])
        most = max(1, min(64, 200_000_000 // (hw * hw * c * SIZE[dtype])))
        case.update(op=rng.choice(["pack", "unpack", "nchw_to_nhwc", "nhwc_to_nchw"]), batch=_log(rng, 1, most), c=c, hw=hw,
                    lanes=rng.choice([4, 16, 32]), dtype=dtype)
    elif rng.random() < 0.5:
        case.update(op="conv2d", batch=_log(rng, 1, 8), hw=rng.randint(7, 64), c=_log(rng, 8, 256), n=_log(rng, 8, 256),
                    k=rng.choice([1, 3]), out=rng.choice(["u8", "f32"]))
    else:
        case.update(op="mat_mul", batch=1, hw=_log(rng, 1, 1024), c=_log(rng, 64, 1024), n=_log(rng, 64, 1024), k=1,
                    out=rng.choice(["u8", "f32"]))
    return case


# ------------------------------------------------------------------------------------------------ what a program keeps
@functools.lru_cache(maxsize=None)
def _context():
    return Context(0)


@functools.lru_cache(maxsize=4)
def _graph(model, hw):
    """The quantised network, calibrated on one image."""
    g = {"mobilenet_v2": nb.mobilenet_v2, "yolov5s": nb.yolov5s}[model](input_hw=hw)
    return nb.quantize_graph(g, np.random.default_rng(3).random((1, hw, hw, 3), dtype=np.float32), calib_batch=1)


@functools.lru_cache(maxsize=4)
def _model_file(model, hw, batch):
    return kmodel.compile_quant_graph(_graph(model, hw), batch)


@functools.lru_cache(maxsize=2)
def _decoder_weights(layers, vocab):
    """A checkpoint of the benchmark's decoder shape, int8 per output channel, the vocabulary head tied to the embedding
    and the residual branches small beside it, so that the greedy token has a margin as it has in a trained model."""
    cfg = llm.DecoderConfig(layers=layers, vocab=vocab)
    rng = np.random.default_rng(5)
    qd, kvd = cfg.q_heads * cfg.head_dim, cfg.kv_heads * cfg.head_dim

    def lin(n, k, std):
        return rng.integers(-127, 128, (n, k), dtype=np.int8), np.full(n, std / 73.3, np.float32)

    def gain():
        return (1.0 + 0.1 * rng.standard_normal(cfg.hidden)).astype(np.float16)

    def layer():
        return {"ln1": gain(), "qkv": lin(qd + 2 * kvd, cfg.hidden, cfg.hidden ** -0.5),
                "qkv_bias": (rng.standard_normal(qd + 2 * kvd) * 0.1).astype(np.float32), "o": lin(cfg.hidden, qd, qd ** -0.5 * 0.2),
                "ln2": gain(), "gate_up": lin(2 * cfg.mlp, cfg.hidden, cfg.hidden ** -0.5),
                "down": lin(cfg.hidden, cfg.mlp, cfg.mlp ** -0.5 * 0.2)}

    head = lin(vocab, cfg.hidden, cfg.hidden ** -0.5)
    return cfg, {"layers": [layer() for _ in range(layers)], "embedding": head[0].astype(np.float16) * np.float16(0.5 / 73.3),
                 "ln_f": gain(), "lm_head": head}


class _Device:
    """A tensor on the device as torch sees it, over memory the framework allocated."""

    def __init__(self, buf, shape, dtype):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(int(s) for s in shape), "typestr": np.dtype(NUMPY[dtype]).str,
                                         "data": (buf.ptr, False), "version": 2}


def _view(buf, shape, dtype):
    return torch.as_tensor(_Device(buf, shape, dtype), device="cuda")


def _upload(values):
    """A framework buffer holding a torch tensor's values, made on the GPU."""
    name = next(k for k, t in TORCH.items() if t == values.dtype)
    buf = _context().alloc(values.numel() * values.element_size())
    _view(buf, values.shape, name).copy_(values)
    return buf


def _result(shape, dtype):
    buf = _context().alloc(math.prod(shape) * SIZE[dtype])
    view = _view(buf, shape, dtype)
    view.zero_()
    return buf, view


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _codes(g, shape):
    """Activations as calibration leaves them: a bell over the 256 codes."""
    return (torch.randn(shape, generator=g, device="cuda") * 40 + 110).clamp_(0, 255).to(torch.uint8)


def _weights(rng, shape):
    """Quantised weights of a layer: (codes, zero point, scale)."""
    fan_in = math.prod(shape[1:]) if len(shape) == 4 else shape[0]
    return quant.quantize_weights((rng.standard_normal(shape, dtype=np.float32) * np.float32(fan_in ** -0.5)))


X_QP, Y_QP = qp(110, 0.02), qp(118, 0.021)   # a layer's input and output at the spread that _codes and _weights give


def _conv_out(c):
    p = c["k"] // 2
    return (c["hw"] + 2 * p - c["k"]) // c["stride"] + 1


def _layout_shapes(c):
    """(plain NCHW shape, the other one) of a layout case."""
    n, ch, hw = c["batch"], c["c"], c["hw"]
    plain = [n, ch, hw, hw]
    return plain, [n, -(-ch // c["lanes"]), hw, hw, c["lanes"]] if c["op"] in ("pack", "unpack") else [n, hw, hw, ch]


def _context_lengths(c):
    """Lengths between an eighth of the largest and the largest, the same total for every seed."""
    return np.linspace(max(1, c["ctx"] // 8), c["ctx"], c["batch"] + 1)[1:].astype(np.int32)


# ------------------------------------------------------------------------------------------------ the four functions
def prepare(case, seed):
    ctx, c, kind = _context(), case, case["kind"]
    g, rng = _generator(seed), np.random.default_rng(seed)
    s = {"kind": kind, "case": c, "ctx": ctx}
    if kind in ("net", "kmodel"):
        qg = _graph(c["model"], c["hw"])
        image = rng.random((c["batch"],) + tuple(qg.input_shape), dtype=np.float32)
        if kind == "kmodel":
            s["model"] = rt.LoadedKModel(ctx, _model_file(c["model"], c["hw"], c["batch"]))
            s["image"] = image.reshape(s["model"].input_shape)
        else:
            s["model"] = m = nb.HipModel(ctx, qg, c["batch"])
            m.set_input(image)
            s["out"] = []
            for buf, j in zip(m.outputs_f32, qg.output_nodes):
                ch, h, w = qg.nodes[j].out_shape
                s["out"].append(_view(buf, (c["batch"], h, w, ch), "f32"))
    elif kind == "decode":
        cfg, weights = _decoder_weights(c["layers"], c["vocab"])
        lens = rng.permutation(_context_lengths(c))
        blocks = -(-(c["ctx"] + 1) // cfg.block_size)
        total = c["batch"] * blocks
        table = rng.permutation(total).reshape(c["batch"], blocks).astype(np.int32)
        empty = np.zeros((total, cfg.kv_heads, cfg.block_size, cfg.head_dim), np.float16)
        flat = empty.reshape(total, cfg.kv_heads, cfg.head_dim, cfg.block_size)
        s["model"] = d = llm.HipDecoder(ctx, cfg, weights, c["batch"], blocks, table, lens, [empty] * cfg.layers, [flat] * cfg.layers,
                                        lanes=c["lanes"])
        for layer in d.layers:                      # the conversations so far
            for cache in (layer["k"], layer["v"]):
                _view(cache, (empty.size,), "f16").normal_(generator=g)
        d.set_tokens(rng.integers(0, c["vocab"], c["batch"]).astype(np.int32))
        # The logits depend on every layer's appended rows; of the caches themselves the last layer's are handed back.
        s["out"] = {"logits": _view(d.logits, (c["batch"], c["vocab"]), "f32"), "tokens": _view(d.next_tokens, (c["batch"],), "i32"),
                    "k": _view(d.layers[-1]["k"], empty.shape, "f16"), "v": _view(d.layers[-1]["v"], flat.shape, "f16")}
    elif kind == "attention":
        b, hq, hkv, dim, blk = c["batch"], c["q_heads"], c["kv_heads"], c["head_dim"], 16
        blocks = -(-c["ctx"] // blk)
        total = b * blocks
        table = rng.permutation(total).reshape(b, blocks).astype(np.int32)
        half = {"generator": g, "device": "cuda", "dtype": torch.float16}
        s["q"], s["k"], s["v"] = (_upload(torch.randn(shape, **half)) for shape in ((b, hq, dim), (total, hkv, blk, dim), (total, hkv, dim, blk)))
        s["table"], s["lens"] = ctx.to_device(table), ctx.to_device(rng.permutation(_context_lengths(c)))
        s["y"], s["out"] = _result((b, hq, dim), c["out"])
        s["args"] = rt.PagedAttnArgs(b, hq, hkv, dim, blk, blocks, total, dim ** -0.5, CODE[c["out"]])
    elif kind == "matmul":
        w, zw, sw = _weights(rng, (c["k"], c["n"]))
        s["x"] = _upload(_codes(g, (c["m"], c["k"])))
        s["w"] = ctx.prepack_matmul(w, None, qp(zw, sw), expected_rows=c["m"])
        s["y"], s["out"] = _result((c["m"], c["n"]), c["out"])
        s["args"] = rt.MatmulArgs(c["m"], X_QP, Y_QP, FULL[0], FULL[1], CODE[c["out"]])
    elif kind == "conv":
        n, hw, cin, cout, k, st, p, o = c["batch"], c["hw"], c["cin"], c["cout"], c["k"], c["stride"], c["k"] // 2, _conv_out(c)
        groups = cin if c["depthwise"] else 1
        w, zw, sw = _weights(rng, (cout, cin // groups, k, k))
        s["x"] = _upload(_codes(g, (n, hw, hw, cin)))
        s["w"] = ctx.prepack_conv2d(w, rng.integers(-200, 200, cout).astype(np.int32), qp(zw, sw), groups, expected_pixels=n * o * o)
        s["y"], s["out"] = _result((n, o, o, cout), c["out"])
        s["args"] = rt.Conv2dArgs(n, hw, hw, st, st, 1, 1, p, p, p, p, X_QP, Y_QP, FULL[0], FULL[1], CODE[c["out"]])
    elif kind == "cast":
        src = TORCH[c["src"]]
        if src.is_floating_point:
            x = (torch.randn(c["count"], generator=g, device="cuda") * 1.5).to(src)
        else:
            x = _codes(g, (c["count"],)).to(src)
        s["x"] = _upload(x)
        s["qp"] = qp(0, 3e-4) if c["dst"] == "i16" else qp(0, 0.045) if c["dst"] == "i8" else qp(121, 0.045)
        s["y"], s["out"] = _result((c["count"],), c["dst"])
    elif kind == "layout":
        plain, other = _layout_shapes(c)
        back = c["op"] in ("unpack", "nhwc_to_nchw")
        bits = {1: torch.uint8, 2: torch.int16, 4: torch.int32}[SIZE[c["dtype"]]]
        x = torch.randint(0, 200, other if back else plain, generator=g, device="cuda", dtype=bits)
        s["x"] = _upload(x)
        s["y"], s["out"] = _result(plain if back else other, {torch.uint8: "u8", torch.int16: "i16", torch.int32: "i32"}[bits])
        s["plain"] = plain
    else:
        m, k = (c["hw"], c["c"]) if c["op"] == "mat_mul" else (0, 0)
        shape = (m, k) if m else (c["batch"], c["c"], c["hw"], c["hw"])
        s["x"] = np.clip(rng.standard_normal(shape, dtype=np.float32) * 40 + 110, 0, 255).astype(np.uint8)
        w, zw, sw = _weights(rng, (k, c["n"]) if m else (c["n"], c["c"], c["k"], c["k"]))
        s["w"], s["w_qp"], s["bias"] = w, qp(zw, sw), rng.integers(-200, 200, c["n"]).astype(np.int32)
    torch.cuda.synchronize()
    return s


def run(s):
    ctx, kind, c = s["ctx"], s["kind"], s["case"]
    if kind == "net":
        s["model"].invoke()
        return s["out"]
    if kind == "kmodel":
        return s["model"].run(s["image"])
    if kind == "decode":
        d = s["model"]
        d.step()
        ctx.add_i32(d.ctx_lens, c["batch"], -1)     # the token is taken back: the next pass generates it again
        return s["out"]
    if kind == "attention":
        ctx.paged_attention_decode(s["q"], s["k"], s["v"], s["table"], s["lens"], s["y"], s["args"])
    elif kind == "matmul":
        ctx.qmatmul(s["x"], s["w"], s["y"], s["args"])
    elif kind == "conv":
        ctx.qconv2d(s["x"], s["w"], s["y"], s["args"])
    elif kind == "cast":
        call = ctx.quantize if c["src"] in ("f16", "f32") else ctx.dequantize
        call(s["x"], CODE[c["src"]], s["y"], CODE[c["dst"]], c["count"], s["qp"])
    elif kind == "layout":
        n, ch, h, w = s["plain"]
        if c["op"] in ("pack", "unpack"):
            (ctx.pack if c["op"] == "pack" else ctx.unpack)(s["x"], s["y"], SIZE[c["dtype"]], s["plain"], [1], [c["lanes"]])
        else:
            (ctx.nchw_to_nhwc if c["op"] == "nchw_to_nhwc" else ctx.nhwc_to_nchw)(s["x"], s["y"], SIZE[c["dtype"]], n, ch, h, w)
    elif c["op"] == "conv2d":
        p = c["k"] // 2
        return kernels.conv2d(s["x"], s["w"], s["bias"], (1, 1), ((p, p), (p, p)), (1, 1), 1, FULL, X_QP, s["w_qp"], Y_QP,
                              NUMPY[c["out"]], ctx=ctx)
    else:
        return kernels.mat_mul(s["x"], s["w"], X_QP, s["w_qp"], Y_QP, NUMPY[c["out"]], s["bias"], ctx=ctx)
    return s["out"]


def work(case):
    c, kind = case, case["kind"]
    if kind in ("net", "kmodel"):
        qg, b = _graph(c["model"], c["hw"]), c["batch"]
        constants = sum(n.weights.size + 4 * n.bias.size for n in qg.nodes if n.weights is not None)
        ends = 4 * (math.prod(qg.input_shape) + sum(math.prod(qg.nodes[j].out_shape) for j in qg.output_nodes))
        return {"bytes": b * ends + constants, "flops": 2 * b * sum(qg.macs_per_image.values())}
    if kind == "decode":
        cfg = llm.DecoderConfig(layers=c["layers"], vocab=c["vocab"])
        qd, kvd, b = cfg.q_heads * cfg.head_dim, cfg.kv_heads * cfg.head_dim, c["batch"]
        per_layer = (qd + 2 * kvd) * cfg.hidden + cfg.hidden * qd + 3 * cfg.mlp * cfg.hidden
        tokens = int(_context_lengths(c).sum()) + b
        weights = cfg.layers * per_layer + cfg.vocab * cfg.hidden
        return {"bytes": weights + cfg.layers * tokens * kvd * 2 * 2 + b * cfg.vocab * 4,
                "flops": 2 * b * weights + cfg.layers * tokens * 4 * qd}
    if kind == "attention":
        tokens, d = int(_context_lengths(c).sum()), c["head_dim"]
        return {"bytes": tokens * c["kv_heads"] * d * 4 + c["batch"] * c["q_heads"] * d * (2 + SIZE[c["out"]]), "flops": 4 * tokens * c["q_heads"] * d}
    if kind == "matmul" or (kind == "host" and c["op"] == "mat_mul"):
        m, k, n = (c["m"], c["k"], c["n"]) if kind == "matmul" else (c["hw"], c["c"], c["n"])
        return {"bytes": m * k + k * n + m * n * SIZE[c["out"]], "flops": 2 * m * k * n}
    if kind in ("conv", "host"):
        cin, cout, st = (c["cin"], c["cout"], c["stride"]) if kind == "conv" else (c["c"], c["n"], 1)
        o = _conv_out({"hw": c["hw"], "k": c["k"], "stride": st})
        reduction = c["k"] * c["k"] * (1 if c.get("depthwise") else cin)
        pixels = c["batch"] * o * o
        return {"bytes": c["batch"] * c["hw"] * c["hw"] * cin + cout * (reduction + 4) + pixels * cout * SIZE[c["out"]], "flops": 2 * pixels * cout * reduction}
    if kind == "cast":
        return {"bytes": c["count"] * (SIZE[c["src"]] + SIZE[c["dst"]]), "flops": 0}
    plain, other = _layout_shapes(c)
    return {"bytes": (math.prod(plain) + math.prod(other)) * SIZE[c["dtype"]], "flops": 0}


def tolerance(case):
    """Integer paths and the float32 values of codes are exact.  Attention accumulates in float32 over float16 operands;
    a decode step stores its hidden state as float16 between operators."""
    if case["kind"] == "attention":
        return {"rel": 1e-3 if case["out"] == "f16" else 1e-4}
    if case["kind"] == "decode":
        return {"rel": 1e-2}
    return "exact"
