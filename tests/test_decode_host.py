"""When the decoder's layers take the library's row kernels and when tensor expressions, on the CPU."""
import itertools

import pytest
import torch
import torch.fx
import torch.nn.functional as F
from torch.overrides import TorchFunctionMode

from glowq_amd import decode
from glowq_amd import kernels as kernels_module

CFG = decode.DecoderConfig(hidden=64, layers=1, heads=4, kv_heads=2, head_dim=16, intermediate=128, vocab=32, max_len=24)


@pytest.fixture()
def model():
    """One layer in fp32 (the CPU's norm has no fp16 weights for fp32 rows)."""
    torch.manual_seed(0)
    m = decode.Decoder(CFG)
    m.model.layers.append(decode.DecoderLayer(CFG))
    return m.float().eval()


def caches(length=CFG.max_len):
    return [tuple(torch.zeros(CFG.kv_heads, length, CFG.head_dim) for _ in range(2))]


class Recorder:
    """Stands in for the library: computes what its row kernels compute and writes down their names."""

    def __init__(self):
        self.calls = []

    def add_rmsnorm_out(self, x, delta, weight, x_out, h, eps):
        self.calls.append("norm" if delta is None else "add_norm")
        if delta is not None:
            x = x_out.copy_(x + delta)
        h.copy_(F.rms_norm(x, (x.size(-1),), weight, eps))

    def silu_mul(self, gate, up, out):
        self.calls.append("gate")
        out.copy_(F.silu(gate) * up)

    def rope_append(self, q, k, v, cos, sin, pos, q_out, k_out, cache_k, cache_v):
        self.calls.append("append")
        T, d = cos.shape
        for src, dst in ((q, q_out), (k, k_out)):
            dst.copy_(decode._rope(src.view(T, -1, d).transpose(0, 1), cos, sin).transpose(0, 1).reshape(T, -1))
        ok = (pos >= 0) & (pos < cache_k.size(1))  # a position outside writes no row
        cache_k[:, pos[ok]] = k_out.view(T, -1, d)[ok].transpose(0, 1)
        cache_v[:, pos[ok]] = v.view(T, -1, d)[ok].transpose(0, 1)


@pytest.fixture()
def kernels(monkeypatch):
    """The row kernels as a recorder, with the CPU's tensors taken for fit."""
    rec = Recorder()
    monkeypatch.setattr(decode, "load_w4a16_extension", lambda: rec)
    monkeypatch.setattr(decode, "_row_kernels", lambda *tensors: True)
    return rec


def forward(model, T=5, length=CFG.max_len, start=0):
    store = caches(length)
    cos, sin = model.rope_tables("cpu")
    with torch.no_grad():
        logits = model.forward_tokens(torch.arange(T), torch.arange(start, start + T), store, cos, sin, from_empty_cache=True)
    return [logits, *store[0]]


ALL = ["norm", "append", "add_norm", "gate", "norm"]


def layer_inputs(model, T=5):
    cos, sin = model.rope_tables("cpu")
    pos = torch.arange(T)
    mask = torch.where(torch.arange(CFG.max_len)[None] <= pos[:, None], 0.0, float("-inf"))
    return (torch.randn(T, CFG.hidden), cos[:T], sin[:T], *caches()[0], pos, mask)


@pytest.mark.parametrize("part", ["norm", "mlp", "attention", "layer"])
def test_layers_can_be_traced_symbolically(model, part):
    layer, args = model.model.layers[0], layer_inputs(model)
    mod = {"norm": layer.input_layernorm, "mlp": layer.mlp, "attention": layer.self_attn, "layer": layer}[part]
    with torch.no_grad():
        args = args if part in ("attention", "layer") else args[:1]
        traced = torch.fx.symbolic_trace(mod, {"delta": None} if part == "norm" else None)
        got = traced(*args, None) if part == "norm" else traced(*args)
        assert torch.equal(got, mod(*args))


def test_batched_rows_stay_expressions():
    """A tensor under torch.func.vmap has no address to look at."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode(), torch.no_grad():
        with torch.device("cuda"):
            norm = decode.RMSNorm(64, 1e-5)
        x = torch.empty(3, 5, 64, dtype=torch.float16, device="cuda")
        assert torch.func.vmap(norm)(x).shape == x.shape


def test_rows_that_nobody_watches_take_the_kernels(model, kernels, monkeypatch):
    with_kernels = forward(model)
    assert kernels.calls == ALL
    with torch.device("cpu"):  # a function mode that looks at factories only
        forward(model)
    assert kernels.calls == 2 * ALL
    monkeypatch.undo()
    for a, b in zip(with_kernels, forward(model)):
        assert torch.allclose(a, b, atol=1e-5)
    assert kernels.calls == 2 * ALL


def test_rows_in_inference_mode_take_the_kernels(model, kernels):
    want = forward(model)
    with torch.inference_mode():
        got = forward(model)
    assert kernels.calls == 2 * ALL and all(torch.equal(a, b) for a, b in zip(got, want))


def test_function_modes_see_the_expressions(model, kernels):
    seen = []

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    with Watch():
        forward(model)
    assert kernels.calls == []
    assert seen.count("rms_norm") == 3 and seen.count("silu") == 1 and seen.count("index_copy_") == 2


def test_a_torch_without_the_probes_takes_the_expressions(model, kernels, monkeypatch):
    monkeypatch.setattr(kernels_module, "_PROBES", (None,) + kernels_module._PROBES[1:])
    forward(model)
    assert kernels.calls == []


@pytest.mark.parametrize("where", ["class", "instance", "call", "hook", "compiled"])
def test_a_replaced_norm_is_called(model, kernels, monkeypatch, where):
    """The residual add rides on the norm's launch only where calling the norm is nothing but its own forward."""
    norm, own, calls = model.model.layers[0].post_attention_layernorm, decode.RMSNorm.forward, []

    def forward_instead(self, x, delta=None):
        calls.append(self)
        return own(self, x, delta)
    if where == "class":
        monkeypatch.setattr(decode.RMSNorm, "forward", forward_instead)
    elif where == "instance":
        norm.forward = forward_instead.__get__(norm)
    elif where == "call":
        call = torch.nn.Module.__call__
        monkeypatch.setattr(torch.nn.Module, "__call__", lambda self, *a, **kw: (calls.append(self), call(self, *a, **kw))[1])
    elif where == "hook":
        norm.register_forward_hook(lambda mod, args, out: calls.append(mod))
    else:
        norm._compiled_call_impl = lambda *args: (calls.append(norm), own(norm, *args))[1]
    forward(model)
    assert norm in calls and "add_norm" not in kernels.calls


def test_positions_outside_a_short_cache_are_refused(model, kernels):
    """A cache shorter than the rotary tables: torch's index_copy_ appends, and refuses a position outside."""
    expressions = ["norm", "add_norm", "gate", "norm"]
    short, full = forward(model, length=8), forward(model)
    assert kernels.calls == expressions + ALL
    assert torch.allclose(short[0], full[0], atol=1e-5) and torch.allclose(short[1], full[1][:, :8], atol=1e-5)
    with pytest.raises(IndexError):
        forward(model, length=8, start=4)
    with pytest.raises(IndexError):
        forward(model, length=CFG.max_len, start=CFG.max_len - 2)
    kernels.calls.clear()
    forward(model, length=CFG.max_len + 8, start=CFG.max_len - 5)
    assert kernels.calls == ALL


def test_positions_that_nothing_has_checked_are_left_to_index_copy(model, kernels):
    """A layer called by itself, and rows of the tables that belong to other positions."""
    x, cos, sin, ck, cv, pos, mask = layer_inputs(model)
    with torch.no_grad():
        model.model.layers[0](x, cos, sin, ck, cv, pos, mask)
        assert "append" not in kernels.calls
        with pytest.raises(IndexError):
            model.model.layers[0](x, cos, sin, ck, cv, pos + CFG.max_len - 2, None)
        decode._note_positions(cos, pos, CFG.max_len)
        assert decode._inside_cache(cos, pos, ck, cv)
        assert not decode._inside_cache(cos, pos.clone(), ck, cv) and not decode._inside_cache(cos, pos, ck[:, 1:], cv[:, 1:])
        pos += CFG.max_len
        assert not decode._inside_cache(cos, pos, ck, cv)


def test_caches_from_an_iterator(model, kernels):
    """Pairs of caches may come from any iterable, an endless one included; pairs past the layers are not looked at."""
    want, pair = forward(model), caches()[0]
    assert decode._positions_end(torch.arange(5), 24, [pair]) == 24
    cos, sin = model.rope_tables("cpu")
    with torch.no_grad():
        logits = model.forward_tokens(torch.arange(5), torch.arange(5), itertools.repeat(pair), cos, sin, from_empty_cache=True)
    assert all(torch.equal(a, b) for a, b in zip([logits, *pair], want)) and kernels.calls == 2 * ALL
    with torch.no_grad():
        again = model.forward_tokens(torch.arange(5), torch.arange(5), [pair, None], cos, sin, from_empty_cache=True)
    assert torch.equal(again, logits)
