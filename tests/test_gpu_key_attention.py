"""The adapter's row LayerNorm and key-token attention kernels against float64
autograd, at row counts around their workgroups and every key-count variant."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
TYPES = [("f16", "f16"), ("bf16", "f32"), ("f16", "f32"), ("bf16", "bf16")]


def _types(cd, param):
    T = {"f16": torch.float16, "bf16": torch.bfloat16}[cd]
    return T, torch.float32 if param == "f32" else T


def _rel(got, exact):
    return float((got.double() - exact).norm() / exact.norm().clamp_min(1e-12))


@pytest.mark.parametrize("c", [128, 256])
@pytest.mark.parametrize("rows", [1, 3, 16, 17, 4099])
@pytest.mark.parametrize("cd,param", TYPES)
def test_layer_norm_rows(dev, c, rows, cd, param):
    import eccv26_tad_amd as sv

    T, PT = _types(cd, param)
    g = torch.Generator(device=dev).manual_seed(rows + c)
    x = (2 + 3 * torch.randn(rows, c, generator=g, device=dev)).to(T)
    w, b = ((k + 0.3 * torch.randn(c, generator=g, device=dev)).to(PT) for k in (1, 0))
    dy = torch.randn(rows, c, generator=g, device=dev).to(T)
    y, stats = sv.ops.layer_norm_rows(x, w, b, 1e-5)
    dx, dwb = sv.ops.layer_norm_rows_bwd(dy, x, stats, w)
    X, W, Bb = (t.double().requires_grad_(True) for t in (x, w, b))
    Y = F.layer_norm(X, (c,), W, Bb, 1e-5)
    gx, gw, gb = torch.autograd.grad(Y, (X, W, Bb), dy.double())
    # one rounding to T of an fp32 evaluation; the parameter sums stay fp32
    assert _rel(y, Y.detach()) <= ULP[T] and _rel(dx, gx) <= ULP[T]
    assert _rel(dwb[0], gw) <= 1e-5 and _rel(dwb[1], gb) <= 1e-5


@pytest.mark.parametrize("hd", [16, 32])
@pytest.mark.parametrize("B,N,nk", [(1, 2, 1), (2, 17, 1), (2, 35, 3), (3, 64, 4), (1, 50, 5), (2, 2000, 16)])
@pytest.mark.parametrize("cd,param", TYPES)
def test_key_attention(dev, hd, B, N, nk, cd, param):
    import eccv26_tad_amd as sv

    T, PT = _types(cd, param)
    a = 4 * hd
    assert sv.ops.key_attention_ok(4, hd, N, nk) and not sv.ops.key_attention_ok(4, hd, N, 17)
    g = torch.Generator(device=dev).manual_seed(N + nk)
    q, kv, dout = (torch.randn(*s, generator=g, device=dev).to(T) for s in ((B, N, a), (B, nk, 2 * a), (B, N, a)))
    P = [(k + 0.3 * torch.randn(hd, generator=g, device=dev)).to(PT) for k in (1, 0, 1, 0)]
    out = sv.ops.key_attention(q, kv, *P, 1e-5)
    dq, dkv, dn = sv.ops.key_attention_bwd(dout, q, kv, *P, 1e-5)
    Q, KV, *PD = (t.double().requires_grad_(True) for t in (q, kv, *P))
    qn = F.layer_norm(Q[:, nk:].view(B, -1, 4, hd), (hd,), PD[0], PD[1], 1e-5)
    kn = F.layer_norm(KV[:, :, :a].view(B, nk, 4, hd), (hd,), PD[2], PD[3], 1e-5)
    # the kernels' roundings to T, passed over by the gradient: queries and keys,
    # and with float32 parameters the scores, their scaling and the probabilities
    to_t = lambda v: v + (v.detach().to(T).double() - v.detach())  # noqa: E731
    amp = to_t if PT != T else lambda v: v
    qn, kn = to_t(qn), to_t(kn)
    p = amp(torch.softmax(amp(amp((qn.unsqueeze(2) * kn.unsqueeze(1)).sum(-1)) / hd ** 0.5), 2))
    att = (p.unsqueeze(-1) * KV[:, None, :, a:].view(B, 1, nk, 4, hd)).sum(2).reshape(B, N - nk, a)
    OUT = torch.cat([torch.zeros(B, nk, a, dtype=torch.float64, device=dev), att], 1)
    gq, gkv, *gp = torch.autograd.grad(OUT, (Q, KV, *PD), dout.double())
    assert torch.count_nonzero(out[:, :nk]) == 0 and torch.count_nonzero(dq[:, :nk]) == 0
    assert _rel(out, OUT.detach()) <= ULP[T]
    # with one key the softmax is constant: these gradients are zero
    if nk > 1:
        assert _rel(dq, gq) <= 2 * ULP[T] and _rel(dkv, gkv) <= 2 * ULP[T]
        for k in (0, 1, 2):
            # a float32 value beside the middle of two values of T rounds the other way: 1 ulp in a few of
            # the values that a sum over all rows of a head's channel takes
            assert _rel(dn[k], gp[k]) <= 1e-4 + ULP[T] / 8, k
    else:
        assert _rel(dkv[:, :, a:], gkv[:, :, a:]) <= 2 * ULP[T]
        assert float(dq.double().abs().max()) <= 1e-5 and float(dn[:3].abs().max()) <= 1e-3
    # the key bias moves every score of a query alike: zero but for rounding
    assert float(dn[3].abs().max()) <= 1e-4 * (1 + float(dn[2].abs().max())) * N ** 0.5


@pytest.mark.parametrize("hd", [16, 32])
@pytest.mark.parametrize("B,N,nk", [(8, 3, 1), (9, 3, 1), (3, 20, 6), (256, 5, 2), (257, 5, 2), (700, 19, 16)])
@pytest.mark.parametrize("cd,param", TYPES[:2])
def test_key_attention_of_many_samples(dev, hd, B, N, nk, cd, param):
    """Up to 8 keys in one workgroup, more in up to 256 of whole samples."""
    test_key_attention(dev, hd, B, N, nk, cd, param)
