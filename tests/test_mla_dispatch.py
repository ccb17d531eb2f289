"""When MLA.forward may take its fused kernels: the conditions, on the host (no kernel runs)."""
import pytest
import torch
from torch import nn

FP8 = torch.float8_e4m3fn


@pytest.fixture
def layer(monkeypatch):
    from dsv3fp8 import model
    monkeypatch.setattr(model.Linear, "dtype", FP8)
    old = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    yield model.MLA(model.ModelArgs(dim=256, n_heads=2, q_lora_rank=128, max_batch_size=1, max_seq_len=8))
    torch.set_default_dtype(old)


@pytest.mark.parametrize("scale", [0.0, -0.1, 1e-40, float("inf"), float("nan"), torch.tensor(0.1)])
def test_scales_that_the_attention_kernels_refuse(layer, scale):
    q = torch.zeros(1, 2, 2, 192, dtype=torch.bfloat16)
    assert layer._attention_kernels_ok(q, 4, None)
    layer.softmax_scale = scale
    assert not layer._attention_kernels_ok(q, 4, None)


def _strided(n):
    return torch.ones(2 * n, dtype=torch.bfloat16)[::2]


@pytest.mark.parametrize("name", ["q_norm", "kv_norm"])
@pytest.mark.parametrize("what", ["eps", "strided", "expanded", "offset", "fp32"])
def test_norms_that_the_latent_kernel_does_not_take(layer, name, what):
    x = torch.zeros(1, 2, 256, dtype=torch.bfloat16)
    assert layer._latent_kernel_ok(x)
    norm = getattr(layer, name)
    if what == "eps":
        norm.eps = None
    else:
        n = norm.dim
        norm.weight = nn.Parameter({"strided": _strided(n), "expanded": torch.ones(1, dtype=torch.bfloat16).expand(n),
                                    "offset": torch.ones(n + 1, dtype=torch.bfloat16)[1:], "fp32": torch.ones(n, dtype=torch.float32)}[what])
    assert not layer._latent_kernel_ok(x)


@pytest.mark.parametrize("name", ["q_norm", "kv_norm", "wq_a", "wkv_a", "wq_b"])
def test_weights_that_are_not_parameters(layer, name):
    module = getattr(layer, name)
    weight = module.weight.detach()
    del module.weight
    module.register_buffer("weight", weight)
    assert not layer._latent_kernel_ok(torch.zeros(1, 2, 256, dtype=torch.bfloat16))


class _OnGpu(torch.Tensor):
    """A tensor of the host that says it is on the GPU."""
    is_cuda = True
    __torch_function__ = torch._C._disabled_torch_function_impl


class _Slots:
    __slots__ = ()

    def __call__(self, x):
        return x + 1


@pytest.mark.parametrize("what", ["buffers", "parameter", "attribute", "beside", "callable", "no dictionary"])
def test_parts_are_what_the_attributes_say(layer, monkeypatch, what):
    """The kernels get the very caches and modules that the conditions looked at, also where these are no buffers or registered
    modules of the layer: a Parameter, a view of a pool that the program owns, an attribute that hides a buffer; wo may be
    any callable.  (The operators are stand-ins that note their arguments; nothing runs on a GPU.)"""
    from dsv3fp8 import model
    monkeypatch.setattr(model, "gemm_impl", "fp8")
    layer.qk_nope_head_dim, layer.qk_rope_head_dim, layer.v_head_dim, layer.kv_lora_rank = 128, 64, 128, 512
    pool = torch.zeros(4, 8, 512, dtype=torch.bfloat16), torch.zeros(4, 8, 64, dtype=torch.bfloat16)
    for name, cache in zip(("kv_cache", "pe_cache"), pool):
        if what == "parameter":
            setattr(layer, name, nn.Parameter(cache[:1]))
        elif what == "attribute":
            delattr(layer, name)
            setattr(layer, name, cache[1:2])
        elif what == "beside":
            layer.__dict__[name] = cache[1:2]
    if what == "beside":
        for name in ("q_norm", "kv_norm", "wq_b", "wo"):
            layer.__dict__[name] = type(getattr(layer, name))(*{"q_norm": (128,), "kv_norm": (512,), "wq_b": (128, 384), "wo": (256, 256)}[name])
    if what in ("callable", "no dictionary"):
        del layer.wo
        layer.wo = (lambda x: x + 1) if what == "callable" else _Slots()
    q, out, calls = torch.zeros(1, 1, 2, 192, dtype=torch.bfloat16), torch.zeros(1, 1, 256, dtype=torch.bfloat16), []
    monkeypatch.setattr(model, "_mla_query", lambda *a: (calls.append(a), q)[1])
    monkeypatch.setattr(model, "_mla_output", lambda *a: (calls.append(a), out)[1])
    monkeypatch.setattr(torch.ops.dsv3fp8, "mla_decode", lambda *a: (calls.append(a), out)[1])
    x = torch.zeros(1, 1, 256, dtype=torch.bfloat16).as_subclass(_OnGpu)
    with torch.no_grad():
        y = layer(x, 3, torch.ones(1, 32, dtype=torch.complex64), None)
    query, attention = calls
    assert query[3] is layer.q_norm.weight and query[4] is layer.kv_norm.weight and query[11] is layer.wq_b.weight
    assert query[6] is layer.kv_cache and query[7] is layer.pe_cache
    assert attention[2] is layer.kv_cache and attention[3] is layer.pe_cache and attention[4] is layer.wkv_b.weight
    if what in ("callable", "no dictionary"):
        assert torch.equal(y, out + 1)
    else:
        assert y is out and attention[-2] is layer.wo.weight


def test_masks_that_the_attention_kernels_do_not_take(layer):
    q = torch.zeros(1, 2, 2, 192, dtype=torch.bfloat16)
    ones = torch.ones(2, 4)
    for mask in (ones, ones.bfloat16()):
        assert layer._attention_kernels_ok(q, 4, mask)
    for mask in (ones.half(), ones.bool(), ones[:1], torch.ones(4, 2).t(), ones[None], ones.to("meta")):
        assert not layer._attention_kernels_ok(q, 4, mask)
    assert not layer._attention_kernels_ok(q.float(), 4, None) and not layer._attention_kernels_ok(q[:, :, :, ::2], 4, None)


# (sequences, new tokens, positions, explicit form, absorbed form): the layer's microseconds at 128 heads, measured when the costs
# of the rule were fitted
MEASURED = [(1, 64, 64, 94, 107), (1, 96, 512, 124, 158), (1, 32, 2048, 188, 131), (1, 192, 2048, 255, 354), (1, 64, 4096, 309, 211),
            (1, 192, 4096, 382, 552), (1, 64, 16384, 977, 495), (1, 192, 16384, 1122, 1719), (8, 32, 64, 165, 200),
            (8, 32, 512, 340, 244), (8, 96, 512, 439, 577), (8, 64, 2048, 955, 720), (8, 128, 2048, 1085, 1376),
            (8, 64, 4096, 1740, 1150), (8, 128, 4096, 1890, 2207), (8, 32, 16384, 6578, 1771), (8, 96, 16384, 6837, 5068),
            (8, 192, 16384, 7591, 10028), (16, 128, 10000, 8707, 7301), (16, 224, 10000, 9888, 12643)]


def test_form_of_the_attention(layer):
    layer.n_local_heads = 128
    for b, s, t, explicit, absorbed in MEASURED:
        assert layer._explicit_pays(b, s, t) == (explicit < absorbed), (b, s, t)
    for s in range(1, 300):                             # nothing in the caches yet: from 32 tokens on, explicit
        for b in (1, 3, 8, 64):
            assert layer._explicit_pays(b, s, s) == (s >= layer.explicit_min_tokens)
    for heads in (1, 16, 127, 128, 200):                # other head counts
        layer.n_local_heads = heads
        for b, t in ((1, 500), (2, 3000), (8, 16384)):
            assert layer._explicit_pays(b, t, t) and not layer._explicit_pays(b, 31, t)
