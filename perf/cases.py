"""What the speed of this library is measured on: structured-linear work as its users call it.

Kinds of case
  call     one operator call through the function a configuration names (triton_funcs.*), issued eagerly: what the layer
           harness and a program's own modules do
  step     the linears of one transformer block, one after the other; graph = True replays them from a HIP graph captured
           once, as a serving loop does for decode (prefill issues them eagerly)
  module   a wrapper module (models.wrappers) with bias and the activation of an MLP handed to its output stage
  verify   the float32 names, which return their intermediates as well
  pack     the weight quantizer: float factors to int8 / packed int4 codes and scales, once per layer of a loaded checkpoint
  network  a DiT-XL/2 forward with its attention and MLP linears replaced

Sizes are those of configs/layers/*.yaml, configs/networks/dit_xl.yaml and bench.py, and generic ones beside them.  Rows are
the tokens of a call: 1 for decode of one sequence, 2 to 16 for small batches, tens for large ones, hundreds and thousands for
prefill, and odd numbers throughout, since prompts are not powers of two long.
"""
import contextlib
import io
import math
import os
import sys

import torch

# the package's folder is not an importable name: its modules are imported from inside it, as bench.py and the tests do
_PKG = os.path.join(os.getcwd(), "mem-efficient-blr_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

# (in, out, BLAST blocks, BLAST rank, Monarch blocks, Monarch rank, low rank) of configs/layers/*.yaml
LAYERS = {
    "gpt2s.c_attn": (768, 2304, 6, 192, 4, 192, 192),
    "gpt2s.c_fc": (768, 3072, 4, 128, 4, 128, 128),
    "gpt2s.c_proj": (3072, 768, 6, 192, 4, 192, 192),
    "vit_b.attn_qkv": (768, 2304, 3, 128, 4, 128, 128),
    "vit_b.fc1": (768, 3072, 3, 128, 4, 128, 128),
    "vit_b.fc2": (3072, 768, 3, 128, 4, 128, 128),
    "dit_xl.adaln": (1152, 6912, 9, 256, 4, 256, 256),
    "dit_xl.qkv": (1152, 3456, 16, 288, 4, 288, 288),
    "dit_xl.proj": (1152, 1152, 16, 288, 4, 288, 288),
    "dit_xl.fc1": (1152, 4608, 16, 576, 4, 576, 576),
    "dit_xl.fc2": (4608, 1152, 16, 576, 4, 576, 576),
    "llama1b.qo": (2048, 2048, 16, 256, 16, 256, 256),
    "llama1b.gate": (2048, 8192, 16, 512, 16, 512, 512),
    "llama1b.up": (2048, 8192, 16, 768, 16, 768, 768),
    "llama1b.down": (8192, 2048, 16, 768, 16, 768, 768),
    "llama7b.qkvo": (4096, 4096, 16, 512, 4, 1024, 1024),
    "llama7b.gate_up": (4096, 22016, 16, 1024, 4, 1024, 1024),
    "llama7b.down": (11008, 4096, 16, 1024, 4, 1024, 1024),
}
# the linears of one block, in the order a forward calls them
BLOCKS = {
    "gpt2s": ("gpt2s.c_attn", "gpt2s.c_fc", "gpt2s.c_proj"),
    "vit_b": ("vit_b.attn_qkv", "vit_b.fc1", "vit_b.fc2"),
    "llama1b": ("llama1b.qo", "llama1b.qo", "llama1b.gate", "llama1b.up", "llama1b.down"),
    "llama7b": ("llama7b.qkvo",) * 4 + ("llama7b.gate_up", "llama7b.down"),
}
BLAST = ("blast_full", "blast_bmm")
QUANT = ("int8", "int4")
MONARCH = ("monarch_right", "monarch_right_ideal", "monarch_right_left")
OPS = BLAST + QUANT + MONARCH + ("low_rank", "dense")
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _linear(op, layer):
    """The (in, out, blocks, rank) that an operator uses on a layer."""
    i, o, b, r, mb, mr, lr = LAYERS[layer]
    if op in MONARCH:
        return i, o, mb, mr
    if op == "low_rank":
        return i, o, 1, lr
    if op == "dense":
        return i, o, 1, 0
    return i, o, b, r


def _call(op, layer, rows, dtype, **more):
    i, o, b, r = _linear(op, layer)
    return dict({"kind": "call", "op": op, "in": i, "out": o, "b": b, "rank": r, "rows": rows, "dtype": dtype}, **more)


def listed():
    return [
        # a GPT-2 sized layer for one token: nothing but latency
        _call("blast_full", "gpt2s.c_fc", 1, "f16", name="call-blast-small-m1"),
        # the headline: a Llama-7B block's six BLAST linears for one token, replayed by a serving loop
        {"name": "decode-blast-7b-m1", "kind": "step", "graph": True, "net": "llama7b", "op": "blast_full", "rows": 1, "dtype": "f16"},
        # the same block with int8 factors, a batch of four sequences
        {"name": "decode-int8-7b-m4", "kind": "step", "graph": True, "net": "llama7b", "op": "int8", "rows": 4, "dtype": "f16"},
        # batched decode, one large layer called eagerly
        _call("monarch_right_left", "llama7b.gate_up", 16, "bf16", name="call-monarch-gate_up-m16"),
        # a short prompt (or a wide decode batch) through a 1B block: between weight streaming and matrix work, a ragged row count
        {"name": "chunk-blast-1b-m61", "kind": "step", "graph": False, "net": "llama1b", "op": "blast_bmm", "rows": 61, "dtype": "bf16"},
        # eight 224x224 images (197 tokens each) through a ViT-B MLP's first linear with bias and GELU
        _call("blast_full", "vit_b.fc1", 1576, "bf16", name="module-blast-vit-fc1", kind="module", bias=True, act="gelu_tanh"),
        # the verification names the layer harness compares with the torch baselines
        _call("blast_full", "gpt2s.c_fc", 128, "f32", name="verify-blast-c_fc-m128", kind="verify"),
        # prefill of a 2048-token prompt through a Llama-7B block
        {"name": "prefill-blast-7b-m2048", "kind": "step", "graph": False, "net": "llama7b", "op": "blast_full", "rows": 2048, "dtype": "f16"},
        # a prompt of 1000 tokens through the gated MLP's fused projection
        _call("low_rank", "llama7b.gate_up", 1000, "bf16", name="module-lowrank-gated-m1000", kind="module", bias=False, act="silu_mul"),
        # the dense layer that the structured ones are held against
        _call("dense", "llama7b.down", 2048, "f16", name="call-dense-down-m2048"),
        # sixteen images through DiT-XL/2 with BLAST linears: the other half of the headline
        {"name": "network-dit-blast-16", "kind": "network", "op": "blast", "images": 16, "tokens": 256, "dtype": "f16"},
        # packing a Llama-7B layer's factors into int4 while a checkpoint is loaded
        _call("int4", "llama7b.gate_up", 1, "f32", name="pack-int4-gate_up", kind="pack"),
    ]


def _rows(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, op):
    """A layer of the configurations, or as often as not a generic one: block sizes and ranks in eights, not only powers of two."""
    if rng.random() < 0.6:
        return _linear(op, rng.choice(sorted(LAYERS)))
    if op == "dense":
        return 8 * _rows(rng, 64, 1024), 8 * _rows(rng, 64, 2048), 1, 0
    if op == "low_rank":
        return 8 * _rows(rng, 64, 1024), 8 * _rows(rng, 64, 2048), 1, 8 * _rows(rng, 16, 128)
    if op in MONARCH:
        b = rng.choice((2, 4, 8, 16))
        return b * 8 * _rows(rng, 8, 1024 // b), b * 8 * _rows(rng, 8, 1024 // b), b, 16 * _rows(rng, 8, 64)
    b = rng.choice((2, 3, 4, 6, 8, 12, 16))
    return b * 8 * _rows(rng, 8, 1024 // b), b * 8 * _rows(rng, 8, 1024 // b), b, 8 * _rows(rng, 16, 128)


def draw(rng):
    kind = rng.choices(("call", "step", "module", "verify", "pack", "network"), (40, 25, 15, 7, 6, 7))[0]
    if kind == "network":
        return {"kind": kind, "op": rng.choice(("blast", "low_rank", "dense")), "images": rng.randint(1, 16), "tokens": rng.choice((64, 256)), "dtype": "f16"}
    dtype = rng.choice(("f16", "bf16"))
    if kind == "step":
        graph = rng.random() < 0.5
        return {"kind": kind, "graph": graph, "net": rng.choice(sorted(BLOCKS)), "op": rng.choice(OPS),
                "rows": _rows(rng, 1, 16) if graph else _rows(rng, 1, 2048), "dtype": dtype}
    if kind == "verify":
        op = rng.choice(("blast_full", "blast_bmm", "monarch_right_left", "low_rank", "dense"))
        i, o, b, r = _linear(op, rng.choice(sorted(LAYERS)))
        return {"kind": kind, "op": op, "in": i, "out": o, "b": b, "rank": r, "rows": _rows(rng, 32, 1024), "dtype": "f32"}
    if kind == "pack":
        op = rng.choice(QUANT)
        i, o, b, r = _shape(rng, op)
        return {"kind": kind, "op": op, "in": i, "out": o, "b": b, "rank": r, "rows": 1, "dtype": rng.choice(("f32", "f16"))}
    op = rng.choice(OPS)
    i, o, b, r = _shape(rng, op)
    case = {"kind": kind, "op": op, "in": i, "out": o, "b": b, "rank": r, "rows": _rows(rng, 1, 4096), "dtype": dtype}
    if kind == "module":
        case["bias"] = rng.random() < 0.7
        case["act"] = rng.choice(("", "gelu_tanh", "silu", "silu_mul") if o // b % 16 == 0 else ("", "gelu_tanh", "silu"))
    return case


# ---- making the inputs ------------------------------------------------------------------------------------------------

def _randn(gen, dtype, *shape, fan_in=1):
    return torch.randn(shape, device="cuda", generator=gen).mul_(fan_in ** -0.5).to(dtype)


def _func(op, dtype):
    end = "fp32" if dtype == "f32" else "fp16"
    if op in BLAST:
        return "triton_funcs.blast_kernels.triton_%s_%s" % (op, end)
    if op in QUANT:
        return "triton_funcs.blast_sym_quant_kernels.triton_blast_bmm_%s_fp16" % op
    family = "monarch" if op in MONARCH else op
    return "triton_funcs.%s_kernels.triton_%s_%s" % (family, op, end)


def _resolve(path):
    from models.wrappers import resolve
    return resolve(path)[1]


def _factors(gen, op, i, o, b, r, dtype):
    """The operator's weights in the layout its function takes."""
    if op == "dense":
        return (_randn(gen, dtype, i, o, fan_in=i),)
    if op == "low_rank":
        return _randn(gen, dtype, i, r, fan_in=r), _randn(gen, dtype, r, o, fan_in=r)
    if op in MONARCH:
        second = (b, r, o // b) if op == "monarch_right_left" else (b, o // b, r)
        return _randn(gen, dtype, b, i // b, r, fan_in=i // b), _randn(gen, dtype, *second, fan_in=r)
    V = _randn(gen, dtype, b, i // b, r, fan_in=r)
    if op == "blast_full":
        return _randn(gen, dtype, b, r, o // b, fan_in=r), V, _randn(gen, dtype, b, b, r)
    return _randn(gen, dtype, b, o // b, r, fan_in=r), V, _randn(gen, dtype, r, b, b)


def _prepare_linear(gen, op, i, o, b, r, rows, dtype):
    dt = DTYPES[dtype]
    if op in QUANT:
        from triton_funcs.blast_sym_quant_kernels import quantize_blast_factors
        U, V, S = _factors(gen, op, i, o, b, r, torch.float32)
        weights = quantize_blast_factors(U, V, 8 if op == "int8" else 4) + (S.to(dt),)
    else:
        weights = _factors(gen, op, i, o, b, r, dt)
    return _resolve(_func(op, dtype)), (_randn(gen, dt, 1, rows, i),) + weights


def _prepare_module(case):
    from models.wrappers import BlastLinear, DenseLinear, LowRankLinear, MonarchLinear, QuantBlastLinear
    op, dt = case["op"], DTYPES[case["dtype"]]
    common = dict(func_path=_func(op, case["dtype"]), device="cuda", dtype=dt, bias=case["bias"])
    if op == "dense":
        m = DenseLinear(case["in"], case["out"], **common)
    elif op == "low_rank":
        m = LowRankLinear(case["in"], case["out"], rank=case["rank"], **common)
    elif op in MONARCH:
        m = MonarchLinear(case["in"], case["out"], b=case["b"], rank=case["rank"], **common)
    elif op in QUANT:
        m = QuantBlastLinear(case["in"], case["out"], b=case["b"], rank=case["rank"], bits=8 if op == "int8" else 4, **common)
    else:
        m = BlastLinear(case["in"], case["out"], b=case["b"], rank=case["rank"], **common)
    m.fused_act = case["act"] or None
    return m.eval()


def _prepare_network(case):
    from models.dit_xl import CustomDiT
    from utils import load_yaml
    cfg = load_yaml(os.path.join(_PKG, "configs", "networks", "dit_xl.yaml"))[case["op"]]
    cfg = {k: {"rank": v.get("rank"), "b": v.get("b"), "func": v["triton"]["func"]} for k, v in cfg.items()}
    side = 2 * int(case["tokens"] ** 0.5)
    dt = DTYPES[case["dtype"]]
    with torch.device("cuda"), contextlib.redirect_stdout(io.StringIO()):
        model = CustomDiT(layer_configs=cfg, method=case["op"], dtype=dt, device="cuda", input_size=side)
    n = case["images"]
    x = torch.randn(n, 4, side, side, device="cuda").to(dt)
    return model, (x, torch.randint(0, 1000, (n,), device="cuda"), torch.randint(0, 1000, (n,), device="cuda"))


def _capture(calls):
    """The calls in a HIP graph, warmed up and captured on a stream of its own, and the tensors that a replay writes."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for f, args in calls:
            f(*args)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        outs = [f(*args) for f, args in calls]
    return graph, outs


def prepare(case, seed):
    gen = torch.Generator("cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "step":
        calls = [_prepare_linear(gen, case["op"], *_linear(case["op"], name), case["rows"], case["dtype"]) for name in BLOCKS[case["net"]]]
        if case["graph"]:
            graph, outs = _capture(calls)
            return {"graph": graph, "outs": outs, "calls": calls}
        return {"calls": calls}
    if kind == "pack":
        U, V, _ = _factors(gen, case["op"], case["in"], case["out"], case["b"], case["rank"], DTYPES[case["dtype"]])
        return {"pack": (U, V, 8 if case["op"] == "int8" else 4)}
    torch.manual_seed(seed)                                     # the modules draw their own parameters
    if kind == "module":
        return {"model": _prepare_module(case), "inputs": (_randn(gen, DTYPES[case["dtype"]], 1, case["rows"], case["in"]),)}
    if kind == "network":
        model, inputs = _prepare_network(case)
        return {"model": model, "inputs": inputs}
    return {"calls": [_prepare_linear(gen, case["op"], case["in"], case["out"], case["b"], case["rank"], case["rows"], case["dtype"])]}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    if "calls" in state:
        return [f(*args) for f, args in state["calls"]]
    if "pack" in state:
        from triton_funcs.blast_sym_quant_kernels import quantize_blast_factors
        u, v = quantize_blast_factors(*state["pack"])
        return u.codes, u.scales, v.codes, v.scales
    with torch.no_grad():
        return state["model"](*state["inputs"])


# ---- what a pass cannot do without ------------------------------------------------------------------------------------

def _linear_work(op, i, o, b, r, rows, dtype, out_columns=None):
    e = 4 if dtype == "f32" else 2
    acts = e * rows * (i + (o if out_columns is None else out_columns))
    if op == "dense":
        return e * i * o + acts, 2 * rows * i * o
    if op == "low_rank" or op in MONARCH:
        return e * r * (i + o) + acts, 2 * rows * r * (i + o)
    flops = 2 * rows * r * (i + o + b * b)
    if op in QUANT:
        return r * (i + o) * (8 if op == "int8" else 4) // 8 + 2 * (o + b * r) + e * b * b * r + acts, flops
    return e * r * (i + o + b * b) + acts, flops


def work(case):
    kind, op = case["kind"], case["op"]
    if kind == "step":
        each = [_linear_work(op, *_linear(op, name), case["rows"], case["dtype"]) for name in BLOCKS[case["net"]]]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    if kind == "pack":                                          # weights read once, codes and scales written once
        n = case["rank"] * (case["in"] + case["out"])
        codes = n if op == "int8" else n // 2
        return {"bytes": n * (4 if case["dtype"] == "f32" else 2) + codes + 2 * (case["out"] + case["b"] * case["rank"]), "flops": 0}
    if kind == "network":                                       # weights of every block once, the linears, adaLN and attention
        rows, n, depth, h = case["images"] * case["tokens"], case["images"], 28, 1152
        size = {"blast": "blast_bmm"}.get(op, op)
        each = [_linear_work(size, *_linear(size, "dit_xl." + name), rows, case["dtype"]) for name in ("qkv", "proj", "fc1", "fc2")]
        if op == "dense":
            weights = 2 * 12 * h * h
        else:
            weights = sum(b - 2 * rows * (_linear(size, "dit_xl." + name)[0] + _linear(size, "dit_xl." + name)[1])
                          for (b, _), name in zip(each, ("qkv", "proj", "fc1", "fc2")))
        flops = sum(f for _, f in each) + 4 * rows * case["tokens"] * h + 2 * n * h * 6 * h
        return {"bytes": depth * (weights + 2 * 6 * h * h) + 2 * n * case["tokens"] * 4 * 4 * 3, "flops": depth * flops}
    columns = case["out"] // 2 if case.get("act") == "silu_mul" else None
    by, fl = _linear_work(op, case["in"], case["out"], case["b"], case["rank"], case["rows"], case["dtype"], columns)
    if kind == "module" and case["bias"]:
        by += (4 if case["dtype"] == "f32" else 2) * case["out"]
    if kind == "verify":                                        # the intermediates are results too
        by += 4 * case["rows"] * {"low_rank": case["rank"], "dense": 0}.get(op, (2 if op in BLAST else 3 if op in MONARCH else 1) * case["b"] * case["rank"])
    return {"bytes": by, "flops": fl}


def tolerance(case):
    if case["kind"] == "pack":
        return "exact"                                          # codes and scales are defined to the bit
    # about four times what the paths show against themselves in 64 bits: f16 7e-4 (max 4e-3), bf16 4e-3 (3e-2), f32 1e-6 over the
    # longest reductions; 28 layers of f16 1.6e-3 (7e-3)
    if case["kind"] == "network":
        return {"rel": 6e-3, "max": 3e-2}
    rel = {"f16": 3e-3, "bf16": 2e-2, "f32": 1e-5}[case["dtype"]]
    return {"rel": rel, "max": 6 * rel}
