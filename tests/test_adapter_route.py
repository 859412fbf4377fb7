"""Which adapter modules take the native key-token attention: only those whose
layers a plain call would run as they are."""
from __future__ import annotations

import pytest
import torch


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
