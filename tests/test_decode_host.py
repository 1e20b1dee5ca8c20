"""When the decoder's layers take the library's row kernels and when tensor expressions, on the CPU."""
import pytest
import torch
import torch.fx

from glowq_amd import decode

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
