"""A forward set on a submodule's instance or class (as dispatch and instrumentation libraries
do) is called: the block's shorter paths stand aside for it, as they do for hooks."""

import types

import pytest
import torch
from torch import nn

import complexity_deep.layer as layer_mod
from complexity_deep import _native as nat
from complexity_deep.attention import _plain_linear, _plain_norm

H = 64


def _block():
    return layer_mod.TransformerBlock(H, 128, 2, 1, num_experts=2, vocab_size=32)


@pytest.mark.parametrize("name", [None, "self_attn", "mlp", "self_attn.o_proj"])
def test_generation_step_honours_a_replaced_forward(monkeypatch, name):
    calls = []
    monkeypatch.setattr(nat, "host", lambda: types.SimpleNamespace(block_step=lambda *a: calls.append(a)))
    block = _block().bfloat16()
    if name is not None:
        m = block.get_submodule(name)
        m.forward = m.forward
    route = types.SimpleNamespace(perm=None, offsets=None, num_experts=2)
    assert block.step(torch.zeros(1, 1, H, dtype=torch.bfloat16), None, None, route) is None
    assert len(calls) == (1 if name is None else 0)


def test_block_forward_gives_a_replaced_mlp_forward_no_residual(monkeypatch):
    block = _block()
    x, seen = torch.ones(1, 2, H), []
    monkeypatch.setattr(layer_mod, "add_rms_norm", lambda *a: (x, x))
    block.input_layernorm, block.mu_guidance = nn.Identity(), None
    block.self_attn.forward = lambda *a, **k: (x, None)

    def mlp(normed, token_ids=None, route=None, residual=None):
        seen.append(residual)
        return 2 * normed

    block.mlp.forward = mlp
    out = block(x)[0]
    assert seen == [None] and torch.equal(out, 3 * x)


def test_predicates_see_instance_forwards_and_global_hooks():
    lin, norm = nn.Linear(8, 8, bias=False), nn.RMSNorm(8, eps=1e-6)
    assert _plain_linear(lin) and _plain_norm(norm, 8)
    handle = nn.modules.module.register_module_forward_pre_hook(lambda m, a: None)
    try:
        assert not _plain_linear(lin) and not _plain_norm(norm, 8)
    finally:
        handle.remove()
    lin.forward, norm.forward = lin.forward, norm.forward
    assert not _plain_linear(lin) and not _plain_norm(norm, 8)


def test_an_output_projection_without_a_weight_of_its_own_is_called():
    attn = _block().self_attn
    inner = attn.o_proj
    attn.o_proj = nn.Sequential(inner, nn.Dropout(0.0))
    x = torch.randn(1, 2, H)
    assert torch.equal(attn._out_proj(x, None), inner(x))


def _step_calls(monkeypatch, block):
    """How often a step of the block reaches the native block_step."""
    calls = []
    monkeypatch.setattr(nat, "host", lambda: types.SimpleNamespace(block_step=lambda *a: calls.append(a)))
    route = types.SimpleNamespace(perm=None, offsets=None, num_experts=2)
    assert block.step(torch.zeros(1, 1, H, dtype=torch.bfloat16), None, None, route) is None
    return len(calls)


@pytest.mark.parametrize("cls,name", [
    (None, None), (layer_mod.ComplexityAttention, "forward"), (layer_mod.TokenRoutedMLP, "forward"),
    (layer_mod.MuGuidance, "fused"), (layer_mod.TransformerBlock, "_mlp"), (nn.Linear, "forward"),
    (nn.Module, "__call__")])
def test_generation_step_honours_a_method_replaced_on_its_class(monkeypatch, cls, name):
    block = _block().bfloat16()
    if cls is not None:
        own = getattr(cls, name)
        monkeypatch.setattr(cls, name, lambda self, *a, **k: own(self, *a, **k))
    assert _step_calls(monkeypatch, block) == (1 if cls is None else 0)


@pytest.mark.parametrize("path,name", [("", "_mlp"), ("", "forward_fused"), ("mu_guidance", "fused")])
def test_generation_step_honours_a_method_replaced_on_an_instance(monkeypatch, path, name):
    block = _block().bfloat16()
    m = block.get_submodule(path)
    setattr(m, name, getattr(m, name))
    assert _step_calls(monkeypatch, block) == 0


def test_predicates_see_class_forwards(monkeypatch):
    lin, norm = nn.Linear(8, 8, bias=False), nn.RMSNorm(8, eps=1e-6)
    assert _plain_linear(lin) and _plain_norm(norm, 8)
    for m in (lin, norm):
        own = type(m).forward
        monkeypatch.setattr(type(m), "forward", lambda self, x, own=own: own(self, x))
    assert not _plain_linear(lin) and not _plain_norm(norm, 8)


def test_a_layer_that_provides_forward_fused_alone(monkeypatch):
    """An object with forward_fused and no step in a layer's place serves calls of few rows too."""
    import complexity_deep.modeling as modeling

    class Layer(nn.Module):
        use_token_routed_mlp = False

        def __init__(self):
            super().__init__()
            self.input_layernorm = nn.LayerNorm(H)

        def forward_fused(self, h, normed, next_norm, **kw):
            return h + 1, normed + 1, None, None

    model = modeling.ComplexityModel(modeling.ComplexityConfig(
        vocab_size=32, hidden_size=H, intermediate_size=128, num_hidden_layers=2, num_attention_heads=2,
        num_key_value_heads=1, num_experts=2))
    model.layers = nn.ModuleList([Layer(), Layer()])
    monkeypatch.setattr(modeling, "embedding", lambda ids, w: torch.zeros(*ids.shape, H))
    monkeypatch.setattr(modeling, "rms_norm", lambda h, w, eps: h)
    monkeypatch.setattr(modeling, "linear", lambda x, w: x)
    with torch.no_grad():
        out = model(torch.zeros(1, 1, dtype=torch.long))
    assert torch.equal(out.logits, torch.full((1, 1, H), 2.0))


def _hook(m):
    m.register_forward_hook(lambda *a: None)


def _own_forward(m):
    m.forward = m.forward


@pytest.mark.parametrize("change", [None, _hook, _own_forward])
@pytest.mark.parametrize("name", ["q_norm", "k_norm", "rotary_emb"])
def test_heads_of_other_dims_honour_a_replaced_norm_or_rotary_forward(change, name):
    """Heads of 40 took their norms and rotary tables through the submodules' forwards: the
    kernels stand in for them only where those are as written."""
    attn = layer_mod.ComplexityAttention(320, 8, 4)
    assert attn.other_head_dim
    if change is not None:
        change(getattr(attn, name))
        assert not attn.other_head_dim


def test_heads_of_other_dims_honour_a_rotary_forward_replaced_on_the_class(monkeypatch):
    attn = layer_mod.ComplexityAttention(320, 8, 4)
    cls = type(attn.rotary_emb)
    own = cls.forward
    monkeypatch.setattr(cls, "forward", lambda self, n: own(self, n))
    assert not attn.other_head_dim
