"""What LAPruneLlama leaves in a model's modules (CPU): the single-token forwards
are bound to the modules, and step back where something else was put in place."""
import copy
import functools
import pickle

import pytest
import torch


def _model(**kw):
    from transformers import LlamaConfig, LlamaForCausalLM
    torch.manual_seed(0)
    cfg = LlamaConfig(vocab_size=32, hidden_size=32, intermediate_size=48, num_hidden_layers=1,
                      num_attention_heads=2, num_key_value_heads=1, **kw)
    return LlamaForCausalLM(cfg).eval()


@pytest.fixture
def fused():
    from laprune_amd.llama import _fuse_decode_ops
    model = _model()
    _fuse_decode_ops(model)
    return model


def _parts(model):
    layer, x = model.model.layers[0], torch.randn(1, 1, 32)
    return [(layer.mlp, (x,)), (layer.input_layernorm, (x,)), (layer.self_attn.o_proj, (x,)),
            (model.model.rotary_emb, (x, torch.tensor([[3]])))]


@torch.no_grad()
def test_a_copied_or_pickled_module_runs_on_its_own_weights(fused):
    from laprune_amd.llama import _own_forward
    for mod, args in _parts(fused):
        assert "forward" in mod.__dict__
        for other in (copy.deepcopy(mod), pickle.loads(pickle.dumps(mod))):
            assert _own_forward(other)
            for t in (*other.parameters(), *other.buffers()):
                t.mul_(3.0)
            got, want = other(*args), type(mod).forward(other, *args)
            for a, b in zip(got, want):
                assert torch.equal(a, b)
            mine = mod(*args)
            assert not all(torch.equal(a, b) for a, b in zip(got, mine))


def test_a_replaced_forward_stays(fused):
    """Also one made with functools.wraps around the forward bound here, whose
    attributes it takes over."""
    from laprune_amd.llama import _fuse_decode_ops, _plain
    gate = fused.model.layers[0].mlp.gate_proj
    assert _plain(gate)
    calls, inner = [], gate.forward

    @functools.wraps(inner)
    def outer(x):
        calls.append(1)
        return inner(x)

    gate.forward = outer
    assert not _plain(gate)
    _fuse_decode_ops(fused)
    assert gate.forward is outer
    fused.model.layers[0].mlp(torch.randn(1, 1, 32))
    assert calls


def test_models_without_some_part_are_served():
    """Only the attention layers' projections are needed: another MLP, norms of
    other names, no rotary module and no head are left as they are."""
    from laprune_amd.llama import _fuse_decode_ops, _step_mask
    model = _model()
    assert _step_mask(model, 2, "cpu").shape == (2, 1, 1, 1)
    layer = model.model.layers[0]
    layer.mlp = torch.nn.Sequential(torch.nn.Linear(32, 48), torch.nn.Linear(48, 32))
    del model.model.rotary_emb, model.model.norm, layer.input_layernorm, model.lm_head
    _fuse_decode_ops(model)
    assert "forward" in layer.self_attn.o_proj.__dict__
    del layer.mlp, layer.self_attn.o_proj
    _fuse_decode_ops(model)

    class Other(type(model.model)):
        pass

    model.model.__class__ = Other
    assert _step_mask(model, 2, "cpu") is None
