"""What a user of this framework has it do, as cases that can be timed and compared: the quantised and corrected linears
of a decoder layer at every number of token rows that occurs in serving and evaluation, and the decoder around them.

A case is a dict of plain values; its `kind` says which entry points it goes through:

  linears  the wrappers a converted and patched model holds (`CudaW4A16Linear`, `AddSVDCorrection` with the group cache),
           called on given activations: `layers` layers of `groups` ("all": q|k|v, o, gate|up, down; "qkv": that group
           alone).  `selected` is the part of the groups that carries a correction ("all", "half", "none": GlowQ-S).
           `graph` 1: recorded once into a HIP graph and replayed, as a serving loop does with few token rows;
           0: called from Python.  `fp32` 1: fp32 outputs (the modules' default), else fp16 (what `_configure_cuda_w4a16_env`
           sets).  `bias` 1: q, k and v carry a bias.
  step     one token through `GreedyDecoder(fused=True)`: the recorded step of the whole decoder (norms, group launches,
           attention over the cache, lm_head, pick) at `context` cached tokens.
  window   `Decoder.forward_tokens` over `rows` tokens from an empty cache: the prompt of a generation, or one window of
           a perplexity evaluation.

Weights ~ N(0, 0.02) are quantised by the framework's own converter (int4, asymmetric, groups of 128 columns), right
factors ~ N(0, 1/K), left factors ~ N(0, 0.01), activations ~ N(0, 1), all made on the GPU from the seed.  With several
layers the weights of a pass exceed the last-level cache, as in a real decode loop.
"""
from __future__ import annotations

import math
import os

import torch
import torch.nn as nn

from glowq_amd.correction import AddSVDCorrection, MiniGroupCache
from glowq_amd.decode import DecoderConfig, GreedyDecoder, build_decoder
from glowq_amd.linear import CudaW4A16Linear

GROUP = 128

# hidden, query heads, key/value heads, head size, intermediate
LLAMA_8B = dict(hidden=4096, heads=32, kv_heads=8, head_dim=128, inter=14336)
QWEN_7B = dict(hidden=3584, heads=28, kv_heads=4, head_dim=128, inter=18944)
QWEN_14B = dict(hidden=5120, heads=40, kv_heads=8, head_dim=128, inter=17408)
OPT_1B = dict(hidden=2048, heads=32, kv_heads=32, head_dim=64, inter=8192)


def _linears(name, shape, rows, rank, layers=1, groups="all", selected="all", bias=0, fp32=0, graph=0):
    case = dict(kind="linears", **shape, rows=rows, rank=rank, layers=layers, groups=groups, selected=selected, bias=bias,
                fp32=fp32, graph=graph)
    return dict(name=name, **case) if name else case


def _step(name, shape, rank, layers, context, max_len, vocab):
    case = dict(kind="step", **shape, rank=rank, layers=layers, context=context, max_len=max_len, vocab=vocab)
    return dict(name=name, **case) if name else case


def _window(name, shape, rows, rank, layers, vocab):
    case = dict(kind="window", **shape, rows=rows, rank=rank, layers=layers, vocab=vocab)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # One attention group on one token, called from Python: the smallest call a program makes.
        _linears("qkv_1row_call", OPT_1B, rows=1, rank=64, groups="qkv"),
        # Single-stream decode: the linears of an 8B layer on one token.
        _linears("layer8b_1row", LLAMA_8B, rows=1, rank=128, layers=4, graph=1),
        # A small decode batch.
        _linears("layer8b_4rows", LLAMA_8B, rows=4, rank=128, layers=4, graph=1),
        # A decode batch with the correction on half of the groups (GlowQ-S, rank 256).
        _linears("layer14b_half_16rows", QWEN_14B, rows=16, rank=256, layers=4, selected="half", graph=1),
        # A large, ragged decode batch.
        _linears("layer14b_57rows", QWEN_14B, rows=57, rank=256, layers=2, graph=1),
        # A short prompt, called from Python.
        _linears("layer8b_100rows", LLAMA_8B, rows=100, rank=128, layers=2),
        # A medium prompt on a model with biases and the modules' default fp32 outputs.
        _linears("layer7b_fp32_333rows", QWEN_7B, rows=333, rank=128, bias=1, fp32=1),
        # A full evaluation window or long prompt.
        _linears("layer7b_2048rows", QWEN_7B, rows=2048, rank=128, bias=1),
        # A long ragged prompt with the correction on half of the groups: the others are bare quantised linears.
        _linears("layer14b_half_1500rows", QWEN_14B, rows=1500, rank=256, layers=2, selected="half"),
        # One generated token of a decoder of eight 8B layers, its cache as full as after a prompt of 640 tokens ...
        _step("token8b_640ctx", LLAMA_8B, rank=128, layers=8, context=640, max_len=1024, vocab=128256),
        # ... and late in a long conversation.
        _step("token8b_7000ctx", LLAMA_8B, rank=128, layers=4, context=7000, max_len=8192, vocab=32000),
        # The prompt of a generation through the whole decoder.
        _window("prompt8b_512", LLAMA_8B, rows=512, rank=128, layers=4, vocab=32000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_shape(rng):
    """Decoder shapes from about 1B to 14B.  Widths are multiples of 256 in most models and of 128 in a few."""
    head_dim = rng.choice((64, 128, 128))
    unit = 128 if rng.random() < 0.2 else 256
    hidden = _log_int(rng, 1536, 5120) // unit * unit
    heads = hidden // head_dim
    kv_heads = heads // rng.choice([d for d in (1, 2, 4, 5, 6, 7, 8) if heads % d == 0])
    inter = int(hidden * rng.uniform(2.5, 5.0)) // unit * unit
    return dict(hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=head_dim, inter=min(inter, 18432))


def draw(rng):
    while True:
        shape = _draw_shape(rng)
        rank = rng.choice((32, 64, 128, 128, 256))
        kind = rng.choice(("call", "decode", "decode", "prompt", "prompt", "step", "window"))
        if kind == "call":
            case = _linears(None, shape, _log_int(rng, 1, 4), rank, groups="qkv", bias=rng.choice((0, 1)))
        elif kind == "decode":
            case = _linears(None, shape, _log_int(rng, 1, 64), rank, layers=rng.choice((2, 3, 4)),
                            selected=rng.choice(("all", "all", "half", "none")), graph=1)
        elif kind == "prompt":
            case = _linears(None, shape, _log_int(rng, 65, 2048), rank, selected=rng.choice(("all", "all", "half")),
                            bias=rng.choice((0, 1)), fp32=rng.choice((0, 0, 1)))
        elif kind == "step":
            max_len = rng.choice((1024, 4096, 8192))
            case = _step(None, shape, rank, rng.choice((2, 4, 6)), _log_int(rng, 64, max_len - 16), max_len, 32000)
        else:
            case = _window(None, shape, _log_int(rng, 65, 2048), rank, rng.choice((1, 2, 3)), 32000)
        if all(work(case)[k] <= max(work(c)[k] for c in listed()) for k in ("bytes", "flops")):
            return case


# ------------------------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------------------------
def _layer_groups(case):
    """(members (role, rows out), columns in) of each group of a layer."""
    qd, kd = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    groups = [((("q", qd), ("k", kd), ("v", kd)), case["hidden"])]
    if case.get("groups", "all") == "all":
        groups += [((("o", case["hidden"]),), qd), ((("gate", case["inter"]), ("up", case["inter"])), case["hidden"]),
                   ((("down", case["hidden"]),), case["inter"])]
    return groups


def _corrected(case, layer, group):
    selected = case.get("selected", "all")
    return selected == "all" or (selected == "half" and (layer + group) % 2 == 0)


def _select_outputs(case):
    dtype = "fp32" if case.get("fp32") else "fp16"
    if os.environ.get("W4A16_KERNEL_OUT_DTYPE") != dtype:
        os.environ["W4A16_KERNEL_OUT_DTYPE"] = dtype  # the modules honour the switch on their next forward


def _normal(gen, *size, std=1.0):
    return torch.empty(*size, dtype=torch.float16, device="cuda").normal_(0.0, std, generator=gen)


def _make_modules(case, gen):
    """[(modules of a group, its input)] over the layers of a "linears" case."""
    todo = []
    for layer in range(case["layers"]):
        for g, (members, cols) in enumerate(_layer_groups(case)):
            cache = MiniGroupCache() if len(members) > 1 else None
            R = _normal(gen, case["rank"], cols, std=cols ** -0.5)
            mods = []
            for role, rows_out in members:
                lin = nn.Linear(cols, rows_out, bias=bool(case["bias"]) and role in ("q", "k", "v"), dtype=torch.float16,
                                device="cuda")
                with torch.no_grad():
                    lin.weight.normal_(0.0, 0.02, generator=gen)
                    if lin.bias is not None:
                        lin.bias.normal_(0.0, 0.1, generator=gen)
                mod = CudaW4A16Linear.from_float(lin, GROUP)
                L = _normal(gen, rows_out, case["rank"], std=0.01)
                if _corrected(case, layer, g):
                    mod = AddSVDCorrection(mod, L, R, role=role if cache is not None else "solo", is_group=cache is not None,
                                           group_cache=cache, alpha_svd=1.0)
                mods.append(mod.eval())
            todo.append((mods, _normal(gen, case["rows"], cols)))
    return todo


def _forward_all(todo):
    return [mod(x) for mods, x in todo for mod in mods]


@torch.no_grad()
def prepare(case, seed):
    _select_outputs(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case}
    if case["kind"] == "linears":
        state["todo"] = _make_modules(case, gen)
        if case["graph"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _forward_all(state["todo"])
                side.synchronize()
                state["graph"] = torch.cuda.CUDAGraph()
                with torch.cuda.graph(state["graph"], stream=side):
                    state["outputs"] = _forward_all(state["todo"])
            torch.cuda.current_stream().wait_stream(side)
        return state

    length = case["max_len"] if case["kind"] == "step" else case["rows"]
    cfg = DecoderConfig(hidden=case["hidden"], layers=case["layers"], heads=case["heads"], kv_heads=case["kv_heads"],
                        head_dim=case["head_dim"], intermediate=case["inter"], vocab=case["vocab"], max_len=length,
                        group_size=GROUP, rank=case["rank"])
    with torch.device("cuda"):
        model, _, _ = build_decoder(cfg, seed=seed)
    prompt = torch.randint(0, cfg.vocab, (case["context"] if case["kind"] == "step" else case["rows"],), generator=gen,
                           device="cuda")
    if case["kind"] == "step":
        dec = GreedyDecoder(model, use_graph=True, fused=True)
        dec.generate(prompt, 2)  # records the step, fills the cache
        state.update(decoder=dec, token=prompt[-1:].clone())
    else:
        dec = GreedyDecoder(model, use_graph=False)
        state.update(decoder=dec, tokens=prompt, positions=torch.arange(prompt.numel(), device="cuda"))
    return state


# ------------------------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------------------------
@torch.no_grad()
def run(state):
    case = state["case"]
    if case["kind"] == "linears":
        if case["graph"]:
            state["graph"].replay()
            return state["outputs"]
        _select_outputs(case)
        return _forward_all(state["todo"])
    dec = state["decoder"]
    if case["kind"] == "step":
        dec.tok.copy_(state["token"])
        dec.pos.fill_(case["context"])
        dec.graph.replay()
        return [dec.fused.logits] + [t for pair in dec.caches for t in pair]
    _select_outputs(case)
    logits = dec.model.forward_tokens(state["tokens"], state["positions"], dec.caches, dec.cos, dec.sin, from_empty_cache=True)
    return [logits] + [t for pair in dec.caches for t in pair]


# ------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------------------------------
def work(case):
    rows = case.get("rows", 1)
    in_bytes = flops = 0
    for layer in range(case["layers"]):
        for g, (members, cols) in enumerate(_layer_groups(case)):
            out = sum(n for _, n in members)
            groups = -(-cols // GROUP)
            # codes, scales, zero-points
            in_bytes += out * cols // 2 + out * groups * 2 + out * (-(-groups // 8)) * 4
            flops += 2 * rows * out * cols
            if _corrected(case, layer, g):
                in_bytes += 2 * case["rank"] * (cols + out)
                flops += 2 * rows * case["rank"] * (cols + out)
            if case["kind"] == "linears":  # activations of the linears are inputs and outputs of the pass
                in_bytes += rows * (2 * cols + (4 if case["fp32"] else 2) * out)
    if case["kind"] == "linears":
        return {"bytes": in_bytes, "flops": flops}
    qd, kd = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    hidden, vocab, layers = case["hidden"], case["vocab"], case["layers"]
    in_bytes += 2 * vocab * hidden + 2 * rows * hidden + 4 * layers * hidden  # lm_head, embedding rows, norm weights
    flops += 2 * rows * vocab * hidden
    if case["kind"] == "step":
        in_bytes += layers * 4 * kd * (case["context"] + 1)       # the cache read, one row of it written
        flops += layers * 4 * qd * (case["context"] + 1)
        return {"bytes": in_bytes + 2 * vocab, "flops": flops}
    in_bytes += layers * 4 * kd * rows                            # the cache written
    flops += layers * 4 * qd * (rows * (rows + 1) // 2)           # causal
    return {"bytes": in_bytes + 2 * rows * vocab, "flops": flops}


def tolerance(case):
    if case["kind"] == "linears":
        # fp16 outputs and an fp16 r, and from a few rows on a dequantised weight that may or may not be rounded to fp16:
        # 2.1e-4 to 2.8e-4 against a float64 evaluation over these ranges
        return {"rel": 1.2e-3}
    # every layer rounds its activations to fp16 several times: up to 3.0e-3 against a float64 evaluation of the window,
    # up to 3.2e-3 between the recorded step and the same token through the modules
    return {"rel": 1.2e-2}
