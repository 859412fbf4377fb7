"""Which adapter modules take the native key-token attention: only those whose
layers a plain call would run as they are."""
from __future__ import annotations

import pytest
import torch
import torch.nn.utils.prune

import eccv26_tad_amd as sv


def _module():
    import eccv26_tad_amd as sv

    return sv.SparseConvAdapter(768, 0.25, use_attn=2, n_key_tokens=3)


def _lora(m):
    m.qkv.forward = lambda x: torch.nn.functional.linear(x, m.qkv.weight)


class _Scaled(torch.nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


def _subclass(m):
    m.down_attn = _Scaled(256, 128)


CHANGES = {
    "spectral_norm": lambda m: torch.nn.utils.spectral_norm(m.qkv),
    "forward_hook": lambda m: m.down_attn.register_forward_hook(lambda *a: None),
    "norm_hook": lambda m: m.attn_norm.register_forward_pre_hook(lambda *a: None),
    "backward_hook": lambda m: m.k_norm.register_full_backward_hook(lambda *a: None),
    "forward": _lora,
    "subclass": _subclass,
    "no_bias": lambda m: setattr(m, "down_attn", torch.nn.Linear(256, 128, bias=False)),
}


def test_plain_module_is_native():
    m = _module()
    assert m._key_attention_ok(2, 4) and m._key_attention_ok(65535, 9000)
    # no visual token, no sample, more samples than a grid dimension holds
    assert not m._key_attention_ok(2, 3) and not m._key_attention_ok(0, 4) and not m._key_attention_ok(65536, 4)


@pytest.mark.parametrize("change", sorted(CHANGES))
def test_changed_layers_are_called(change):
    m = _module()
    CHANGES[change](m)
    assert not m._key_attention_ok(2, 4)


def test_hook_on_all_modules():
    m = _module()
    handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    try:
        assert not m._key_attention_ok(2, 4)
    finally:
        handle.remove()
    assert m._key_attention_ok(2, 4)


class _Route(Exception):
    pass


def _route(m, monkeypatch):
    """Which route a 16-bit call takes: "one node" for AdapterRowsFunction,
    "chain" for the node of other widths, or "layers" when the modules' calls
    (sparse_conv among them) run."""
    from eccv26_tad_amd import adapter

    def take(name):
        def apply(*args):
            raise _Route(name)
        return apply

    monkeypatch.setattr(adapter.SparseConvAdapter, "_fused_dtype", lambda self, x: torch.bfloat16)
    monkeypatch.setattr(adapter.AdapterRowsFunction, "apply", take("one node"))
    monkeypatch.setattr(adapter.SparseConvAdapterFunction, "apply", take("chain"))
    monkeypatch.setattr(adapter.AdapterDownFunction, "apply", take("layers"))
    with pytest.raises(_Route) as route:
        m(torch.zeros(2, 8, 768), 1, 5, torch.arange(5).expand(2, -1), 5, torch.full((2, 5, 9), -1, dtype=torch.int32))
    return str(route.value)


class _ScaledConv(sv.SparseConv2d):
    def forward(self, *args, **kwargs):
        return 2 * super().forward(*args, **kwargs)


class _Wrapped(torch.nn.Module):
    def __init__(self, conv):
        super().__init__()
        self.conv = conv


CONV_CHANGES = {
    "wrapped": lambda m: setattr(m, "sparse_conv", _Wrapped(m.sparse_conv)),
    "spectral_norm": lambda m: torch.nn.utils.spectral_norm(m.sparse_conv),
    "weight_norm": lambda m: torch.nn.utils.parametrizations.weight_norm(m.sparse_conv),
    "pruned": lambda m: torch.nn.utils.prune.l1_unstructured(m.sparse_conv, "weight", 0.5),
    "forward_hook": lambda m: m.sparse_conv.register_forward_hook(lambda *a: None),
    "backward_hook": lambda m: m.sparse_conv.register_full_backward_hook(lambda *a: None),
    "forward": lambda m: setattr(m.sparse_conv, "forward", lambda *a, **k: None),
    "subclass": lambda m: setattr(m, "sparse_conv", _ScaledConv(256, 256)),
}


@pytest.mark.parametrize("change", ["plain"] + sorted(CONV_CHANGES))
def test_changed_sparse_conv_is_called(change, monkeypatch):
    m = _module()
    CONV_CHANGES.get(change, lambda m: None)(m)
    assert _route(m, monkeypatch) == ("one node" if change == "plain" else "layers")


@pytest.mark.parametrize("mode", ["no_grad", "inference_mode", "frozen", "grad"])
@pytest.mark.parametrize("attn", [0, 2])
def test_inference_prepares_no_backward(mode, attn, monkeypatch):
    """Parameters require gradients when a model is served under no_grad too."""
    from eccv26_tad_amd import adapter

    seen = []

    def forward(x, *args):
        seen.append(args[16])
        return x.clone(), x.new_empty(0), x.new_empty(0), *[x.new_empty(0)] * (26 if attn else 11)

    m = sv.SparseConvAdapter(768, 0.25, use_attn=attn, n_key_tokens=3)
    m.sparse_conv.packed_weight_cache = None  # keyed by the stream of a GPU
    m.requires_grad_(mode != "frozen")
    monkeypatch.setattr(adapter.SparseConvAdapter, "_fused_dtype", lambda self, x: torch.bfloat16)
    monkeypatch.setattr(adapter._ops, "adapter_forward", forward)
    with {"no_grad": torch.no_grad, "inference_mode": torch.inference_mode}.get(mode, torch.enable_grad)():
        y = m(torch.zeros(2, 8, 768), 1, 5, torch.arange(5).expand(2, -1), 5, torch.full((2, 5, 9), -1, dtype=torch.int32))
    assert seen == [mode == "grad"] and y.requires_grad == (mode == "grad")


def _strided(norm):
    norm.weight = torch.nn.Parameter(torch.ones(2 * norm.weight.numel())[::2])


SHAPES = {
    "qkv_in": lambda m: setattr(m, "qkv", torch.nn.Linear(64, 384)),
    "qkv_out": lambda m: setattr(m, "qkv", torch.nn.Linear(128, 256)),
    "down": lambda m: setattr(m, "down_attn", torch.nn.Linear(256, 64)),
    "down_in": lambda m: setattr(m, "down_attn", torch.nn.Linear(128, 128)),
    "proj": lambda m: setattr(m, "attn_proj", torch.nn.Linear(128, 128)),
    "proj_bias": lambda m: setattr(m, "attn_proj", torch.nn.Linear(128, 256, bias=False)),
    "norm": lambda m: setattr(m, "attn_norm", torch.nn.LayerNorm(128)),
    "no_affine": lambda m: setattr(m, "attn_norm", torch.nn.LayerNorm(256, elementwise_affine=False)),
    "head_norm": lambda m: setattr(m, "q_norm", torch.nn.LayerNorm(16)),
    "strided_norm": lambda m: _strided(m.attn_norm),
    "strided_head_norm": lambda m: _strided(m.k_norm),
    "norm_types": lambda m: m.k_norm.half(),
    "hidden": lambda m: setattr(m, "down_proj", torch.nn.Linear(768, 128)),
}


@pytest.mark.parametrize("change", sorted(SHAPES))
def test_layers_of_other_shapes_are_called(change):
    """The kernels read as many values as their widths give: layers of other
    shapes and strides stay with PyTorch, which takes or refuses them."""
    m = _module()
    SHAPES[change](m)
    assert not m._key_attention_ok(2, 4)


def test_exchanged_widths_take_their_own_route(monkeypatch):
    m = sv.SparseConvAdapter(768, 0.25)
    assert _route(m, monkeypatch) == "one node"
    m.down_proj, m.up_proj, m.sparse_conv = torch.nn.Linear(768, 64), torch.nn.Linear(64, 768), sv.SparseConv2d(64, 64)
    assert _route(m, monkeypatch) == "chain"
