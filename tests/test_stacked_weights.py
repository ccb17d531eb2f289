"""MLA.stack_a: wq_a over wkv_a in one buffer, on the host (no kernel runs)."""
import pytest
import torch
from torch import nn

FP8 = torch.float8_e4m3fn


@pytest.fixture
def layer(monkeypatch):
    from dsv3fp8 import model
    monkeypatch.setattr(model.Linear, "dtype", FP8)
    g = torch.Generator().manual_seed(1)
    mla = model.MLA(model.ModelArgs(dim=256, n_heads=1, q_lora_rank=128, max_batch_size=1, max_seq_len=8))
    with torch.no_grad():
        for lin in (mla.wq_a, mla.wkv_a):
            lin.weight.copy_(torch.randn(lin.weight.shape, generator=g))
            lin.scale.copy_(torch.rand(lin.scale.shape, generator=g))
    return mla


def _check(mla):
    assert mla.stack_a()
    for part, scale, lin in ((mla._wa[:128], mla._wa.scale[:1], mla.wq_a), (mla._wa[128:], mla._wa.scale[1:], mla.wkv_a)):
        assert torch.equal(part.view(torch.uint8), lin.weight.view(torch.uint8)) and torch.equal(scale, lin.scale)
        assert part.data_ptr() == lin.weight.data_ptr() and scale.data_ptr() == lin.scale.data_ptr()


def test_stack_is_kept(layer):
    _check(layer)
    buffer = layer._wa.data_ptr()
    with torch.no_grad():                                   # loading in place goes through the views
        layer.wkv_a.weight.copy_(torch.ones(layer.wkv_a.weight.shape))
    _check(layer)
    assert layer._wa.data_ptr() == buffer


@pytest.mark.parametrize("name", ["wq_a", "wkv_a"])
@pytest.mark.parametrize("what", ["weight", "scale", "layer", "data"])
def test_replaced_parameters_are_stacked_anew(layer, name, what):
    _check(layer)
    lin = getattr(layer, name)
    if what == "weight":
        scale = lin.weight.scale
        lin.weight = nn.Parameter(torch.full_like(lin.weight.float(), 2.0).to(FP8), requires_grad=False)
        lin.weight.scale = scale
    elif what == "scale":
        lin.weight.scale = lin.scale = nn.Parameter(lin.scale.detach() * 2)
    elif what == "layer":
        new = type(lin)(lin.in_features, lin.out_features)
        with torch.no_grad():
            new.weight.copy_(torch.ones(new.weight.shape))
            new.scale.fill_(0.5)
        setattr(layer, name, new)
    else:                                                   # what Module.to(device) does
        lin.weight.data = lin.weight.data.clone()
        lin.scale.data = lin.scale.data.clone()
    _check(layer)


@pytest.mark.parametrize("what", ["type", "hook", "pre_hook", "global_hook", "global_pre_hook", "forward"])
def test_only_plain_modules_are_passed_by(layer, what):
    from dsv3fp8 import model
    from torch.nn.modules import module as modules
    assert layer.stack_a() and model._plain(layer.wkv_a, model.Linear)
    lin = layer.wkv_a
    if what == "type":
        lin.__class__ = type("Other", (model.Linear,), {})
    elif what == "forward":
        lin.forward = lambda x: x
    else:
        handle = {"hook": lin.register_forward_hook, "pre_hook": lin.register_forward_pre_hook,
                  "global_hook": modules.register_module_forward_hook,
                  "global_pre_hook": modules.register_module_forward_pre_hook}[what](lambda *a: None)
    try:
        assert not model._plain(lin, model.Linear) and not layer.stack_a()
    finally:
        if what.endswith("hook"):
            handle.remove()
    assert layer.stack_a() == what.endswith("hook")


def test_layers_with_a_bias_are_not_stacked(layer):
    layer.wq_a.bias = nn.Parameter(torch.ones(128))
    assert not layer.stack_a()
