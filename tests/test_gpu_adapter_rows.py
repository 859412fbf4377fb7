"""The adapter GEMMs over whole token tiles (adapter_prep, adapter_rows_*)
against float64, at row counts around their tiles and every type combination."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _near(name, got, exact, bound):
    err = (got.double() - exact).abs()
    assert got.shape == exact.shape, name
    assert bool((err <= bound).all()), (name, float((err / bound.clamp_min(1e-30)).max()))


@pytest.mark.parametrize("embed,hidden", [(384, 128), (768, 256), (1024, 256)])
@pytest.mark.parametrize("B,N,S", [(1, 1, 1), (2, 17, 0), (1, 33, 3), (3, 65, 2), (1, 4, 4), (2, 5000, 1)])
@pytest.mark.parametrize("cd,param", [("f16", "f16"), ("bf16", "f32"), ("bf16", "bf16"), ("f16", "f32")])
def test_rows_match_float64(dev, embed, hidden, B, N, S, cd, param):
    import eccv26_tad_amd as sv

    ops = sv.ops
    T = {"f16": torch.float16, "bf16": torch.bfloat16}[cd]
    PT = torch.float32 if param == "f32" else T
    g = torch.Generator(device=dev).manual_seed(embed + 7 * N + S)

    def rnd(*s, scale=1.0):
        return (torch.randn(*s, generator=g, device=dev) * scale).to(PT)

    E, h = embed, hidden
    w_d, b_d, w_u, b_u, w_c, b_c = (rnd(h, E, scale=0.05), rnd(h, scale=0.1), rnd(E, h, scale=0.05),
                                    rnd(E, scale=0.1), rnd(9, h, h, scale=0.05), rnd(h))
    gamma = rnd(1) + 1
    wd, bd, wu, bu, bc, wc, wuc, wdT, wuT, pf, pb = ops.adapter_prep(w_d, b_d, w_c, b_c, w_u, b_u, gamma, cd == "bf16",
                                                                     True, True)
    # the SparseConv2D layouts and the casts are those of the separate calls
    ref_pf, ref_pb = ops.pack_weight(w_c.to(T), True, True)
    assert torch.equal(pf, ref_pf) and torch.equal(pb[: pf.numel() + 4], ref_pb[: pf.numel() + 4])
    assert torch.equal(wc, w_c.to(T)) and torch.equal(wuc, w_u.to(T)) and torch.equal(bc, b_c.to(T))
    u, eps = ULP[T], 2.0 ** -24
    cast = [t.to(T).double() for t in (w_d, b_d, w_u, b_u)]
    n_pa = B * (N - S)

    def join(sp, pa, n):
        return torch.cat([sp, pa.view(B, N - S, n)], dim=1)

    x = rnd(B, N, E)
    xt = x.to(T).double()
    pre, sp, pa, copy = ops.adapter_rows_down(x, wd, bd, h, S, True)
    z = xt @ cast[0].t() + cast[1]
    acc = (E + 4) * eps * (xt.abs() @ cast[0].abs().t() + cast[1].abs())
    _near("pre", pre, z, u * z.abs() + acc + 1e-7)
    gz = F.gelu(pre.double())
    _near("gelu", join(sp, pa, h), gz, u * gz.abs() + 4e-7 * pre.double().abs() + 1e-7)
    assert pa.shape == (n_pa, h)
    assert torch.equal(copy, x.to(T)) if PT != T else copy.numel() == 0

    go = rnd(B, N, E)
    gt = go.to(T).double()
    sp2, pa2, copy = ops.adapter_rows_split(go, wuT, h, S, True)
    wg = (cast[2].float() * gamma.float()).to(T).double()  # w_u cast, times gamma, rounded
    dc = gt @ wg
    _near("split", join(sp2, pa2, h), dc, u * dc.abs() + (E + 4) * eps * (gt.abs() @ wg.abs()) + 1e-7)
    assert torch.equal(copy, go.to(T)) if PT != T else copy.numel() == 0

    a = join(sp, pa, h).double()
    z = a @ cast[2].t() + cast[3]
    acc = (h + 4) * eps * (a.abs() @ cast[2].abs().t() + cast[3].abs())
    gm = gamma.double()
    for res_t, out32 in {(PT, PT == torch.float32), (T, PT == torch.float32), (PT, False)}:
        res = x.to(res_t)
        y = z * gm + res.double()
        got = ops.adapter_rows_res(sp, pa, wu, bu, gamma, res, out32)
        assert got.dtype == (torch.float32 if out32 else T)
        _near("up", got, y, gm.abs() * (2.5 * u * z.abs() + acc) + (0 if out32 else u) * y.abs() + 1e-6)
    du = join(sp, pa, h)
    y = a @ cast[0] + x.double()
    acc = (h + 4) * eps * (a.abs() @ cast[0].abs() + x.double().abs())
    got = ops.adapter_rows_res(None, du, wdT, du.new_empty(0), None, x, PT == torch.float32)
    _near("gx", got, y, (0 if PT == torch.float32 else u) * y.abs() + acc + 1e-7)


@pytest.mark.parametrize("embed,attn,S,heat", [(384, 0, 2, False), (768, 2, 3, False), (384, 2, 1, False), (1024, 2, 5, False),
                                               (768, 2, 32, False), (384, 2, 32, False), (768, 2, 33, False),
                                               (768, 0, 31, True), (768, 0, 0, False)])
@pytest.mark.parametrize("amp", [True, False])
def test_module_gradients_match_float32(dev, embed, attn, S, heat, amp):
    """The native forward and backward of the module against the float32
    restatement of the reference adapter, every gradient."""
    from tests.adapter_ref import adapter_fp32, gain_scales
    import eccv26_tad_amd as sv

    B, T, H, W = 2, 3, 5, 6
    g = torch.Generator(device=dev).manual_seed(embed + S + attn)
    kw = dict(heatmap_grid_size=(H, W)) if heat else {}
    mod = sv.SparseConvAdapter(embed, 0.25, use_attn=attn, n_key_tokens=max(S, 1), **kw).to(dev)
    with torch.no_grad():
        for name, p in mod.named_parameters():
            if name.endswith("weight") and p.dim() > 1:
                p.copy_(torch.randn(p.shape, generator=g, device=dev) * p.shape[-1] ** -0.5)
            else:
                p.add_(0.2 * torch.randn(p.shape, generator=g, device=dev) + 0.1)
    cd = torch.bfloat16 if amp else torch.float16
    dt = torch.float32 if amp else cd
    mod = mod.to(dt)
    mask = torch.zeros(B, T * H * W, dtype=torch.uint8, device=dev)
    idx = torch.rand(B, T * H * W, generator=g, device=dev).topk(40, 1).indices.sort(1).values
    mask.scatter_(1, idx, 1)
    table = sv.build_neighbor_table(mask.view(B, T, H, W), batched=True, n=80)
    x = torch.randn(B, S + 40, embed, generator=g, device=dev).to(dt).requires_grad_(True)
    go = (torch.randn(B, S + 40, embed, generator=g, device=dev) + 0.5).to(dt)
    args = (H, W, idx, T * H * W)
    with torch.autocast("cuda", dtype=cd, enabled=amp):
        y = mod(x, *args, table)
    names = [n for n, _ in mod.named_parameters() if n != "k_norm.bias" and (heat or n != "heatmap_gate")]
    grads = torch.autograd.grad(y, [x] + [mod.get_parameter(n) for n in names], go)
    xr = x.detach().float().requires_grad_(True)
    gains = {}
    yr, P = adapter_fp32(mod, xr, *args, gains=gains)
    yr.backward(go.float())
    scales = gain_scales(gains)
    tol = 2.5e-2 if amp else 4e-3  # a few roundings of each chain in bf16 / f16
    assert float((y.float() - yr).norm() / yr.norm()) <= tol
    for name, got in zip(["x"] + names, grads):
        want = xr.grad if name == "x" else P[name].grad
        assert got.dtype == dt and got.shape == want.shape, name
        err = float((got.float() - want).norm())
        # a scalar gain's gradient against its sum of absolute terms
        bar = tol * scales[name] * 0.2 if name in scales else tol * float(want.norm())
        assert err <= bar, (name, err, bar)


@pytest.mark.parametrize("amp", [True, False])
@pytest.mark.parametrize("name", ["down_proj.weight", "sparse_conv.bias", "up_proj.weight", "down_attn.weight", "qkv.weight"])
def test_parameter_changed_before_backward(dev, amp, name):
    """A parameter changed in place between the two passes is refused when its
    own values were saved and has no effect when it had been cast."""
    import eccv26_tad_amd as sv

    g = torch.Generator(device=dev).manual_seed(5)
    dt = torch.float32 if amp else torch.float16
    mod = sv.SparseConvAdapter(384, 0.25, use_attn=2, n_key_tokens=2).to(dev, dt)
    with torch.no_grad():
        for p in mod.parameters():
            p.add_(0.1 * torch.randn(p.shape, generator=g, device=dev))
    idx = torch.arange(40, device=dev).expand(1, -1)
    table = sv.build_neighbor_table(torch.ones(1, 2, 4, 5, dtype=torch.uint8, device=dev), batched=True, n=40)
    x = torch.randn(1, 42, 384, generator=g, device=dev).to(dt).requires_grad_(True)

    def gradient(change):
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            y = mod(x, 4, 5, idx, 40, table)
        if change:
            with torch.no_grad():
                mod.get_parameter(name).add_(0.25)
        return torch.autograd.grad(y, x, torch.ones_like(y))[0]

    if amp:
        want = gradient(False)
        assert torch.equal(gradient(True), want)
    else:
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            gradient(True)


@pytest.mark.parametrize("embed,attn", [(384, 0), (768, 2), (512, 0)])
@pytest.mark.parametrize("amp", [True, False])
def test_no_grad_matches_grad_mode(dev, embed, attn, amp):
    """A forward without gradients gives the same bits, and packs and keeps the
    forward's layout of the convolution only."""
    import eccv26_tad_amd as sv

    g = torch.Generator(device=dev).manual_seed(embed)
    mod = sv.SparseConvAdapter(embed, 0.25, use_attn=attn, n_key_tokens=2).to(dev, torch.float32 if amp else torch.float16)
    with torch.no_grad():
        for p in mod.parameters():
            p.add_(0.05 * torch.randn(p.shape, generator=g, device=dev))
    idx = torch.arange(40, device=dev).expand(2, -1)
    table = sv.build_neighbor_table(torch.ones(2, 2, 4, 5, dtype=torch.uint8, device=dev), batched=True, n=80)
    x = torch.randn(2, 42, embed, generator=g, device=dev).to(mod.gamma.dtype)
    cache = mod.sparse_conv.packed_weight_cache

    def call(mode):
        with mode(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            return mod(x, 4, 5, idx, 40, table).detach()

    cold = call(torch.no_grad)
    kept = cache._packed
    assert kept[1] is None
    assert torch.equal(call(torch.no_grad), cold) and cache._packed is kept
    assert torch.equal(call(torch.enable_grad), cold) and cache._packed[1] is not None
    kept = cache._packed
    assert torch.equal(call(torch.no_grad), cold) and cache._packed is kept


@pytest.mark.parametrize("B,N,S", [(1, 1, 0), (1, 9, 1), (3, 7, 7), (2, 1025, 0), (3, 683, 4), (4, 513, 512)])
def test_patch_rows(dev, B, N, S):
    import eccv26_tad_amd as sv

    want = torch.arange(B * N, device=dev).view(B, N)[:, S:].reshape(-1)
    got = sv.ops.patch_rows(torch.empty(0, device=dev), B, N, S)
    assert got.dtype == torch.int32 and torch.equal(got.long(), want)


@pytest.mark.parametrize("embed", [384, 512])
def test_first_backward_of_a_shape_in_a_capture(dev, embed):
    """Nothing of a backward that ran only inside a graph capture, or on another
    stream, is read by a later one."""
    import eccv26_tad_amd as sv

    g = torch.Generator(device=dev).manual_seed(embed)
    mod = sv.SparseConvAdapter(embed, 0.25).to(dev, torch.float16)
    with torch.no_grad():
        for p in mod.parameters():
            p.add_(0.1 * torch.randn(p.shape, generator=g, device=dev))
    params = list(mod.parameters())

    def inputs(T):
        idx = torch.arange(20 * T, device=dev).expand(2, -1)
        table = sv.build_neighbor_table(torch.ones(2, T, 4, 5, dtype=torch.uint8, device=dev), batched=True, n=40 * T)
        x = torch.randn(2, 2 + 20 * T, embed, generator=g, device=dev).half().requires_grad_(True)
        return x, (4, 5, idx, 20 * T, table), torch.randn(2, 2 + 20 * T, embed, generator=g, device=dev).half()

    def step(x, args, go):
        return torch.autograd.grad(mod(x, *args), [x] + params, go)

    def same(a, b):
        return all(torch.equal(s, t) for s, t in zip(a, b))

    warm, case = inputs(3), inputs(5)
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        step(*warm)
    torch.cuda.current_stream(dev).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step(*case)
    eager = step(*case)  # before any replay
    with torch.cuda.stream(side):
        side.wait_stream(torch.cuda.current_stream(dev))
        other = step(*case)
    torch.cuda.current_stream(dev).wait_stream(side)
    assert same(eager, other)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize(dev)
        assert same(captured, eager) and same(step(*case), eager)


def test_patch_rows_of_2_gib(dev):
    """Inference where the convolution's operand reaches 2^31 bytes, beyond the
    32-bit offsets of its packed kernel: sampled rows against float32."""
    import eccv26_tad_amd as sv

    n, E, h, S = 2 ** 31 // 512, 768, 256, 1
    g = torch.Generator(device=dev).manual_seed(3)
    mod = sv.SparseConvAdapter(E, 0.25).to(dev, torch.float16)
    with torch.no_grad():
        mod.up_proj.weight.copy_(0.05 * torch.randn(E, h, generator=g, device=dev))
    x = torch.randn(1, S + n, E, generator=g, device=dev, dtype=torch.float16)
    step = torch.arange(9, device=dev, dtype=torch.int32) - 4
    table = torch.arange(n, device=dev, dtype=torch.int32).view(n, 1) + step
    table = torch.where((table >= 0) & (table < n), table, -1)
    idx = torch.arange(n, device=dev).view(1, n)
    with torch.no_grad():
        y = mod(x, 1, n, idx, n, table.view(1, n, 9))
    rows = torch.cat([torch.tensor([0, 1, 2, 3, n // 2, n - 4, n - 2, n - 1], device=dev),
                      torch.randint(0, n, (200,), generator=g, device=dev)])
    p = {k: v.detach().float() for k, v in mod.named_parameters()}
    near = table[rows].long()
    src = x[0, S + near.clamp_min(0)].float()
    u = F.gelu(F.linear(src, p["down_proj.weight"], p["down_proj.bias"])) * (near >= 0).unsqueeze(-1)
    conv = p["sparse_conv.bias"] + u.flatten(1) @ p["sparse_conv.weight"].reshape(9 * h, h)
    want = F.linear(conv, p["up_proj.weight"], p["up_proj.bias"]) * p["gamma"] + x[0, S + rows].float()
    got = y[0, S + rows].float()
    # the parts' roundings to float16 (hidden rows, convolution, z, output), each 2^-11 of its value
    assert float((got - want).norm() / want.norm()) <= 4 * 2.0 ** -11
    assert float((got - want).abs().max()) <= 8 * 2.0 ** -11 * float(want.abs().max())


@pytest.mark.parametrize("embed", [384, 768])
def test_hooked_sparse_conv_with_key_attention(dev, embed):
    """The layer is called, and the chain around it agrees with the one node
    within the roundings of either; a doubling hook changes the result."""
    import eccv26_tad_amd as sv

    g = torch.Generator(device=dev).manual_seed(embed)
    mod = sv.SparseConvAdapter(embed, 0.25, use_attn=2, n_key_tokens=2).to(dev, torch.float16)
    with torch.no_grad():
        for p in mod.parameters():
            p.add_(0.1 * torch.randn(p.shape, generator=g, device=dev))
    idx = torch.arange(40, device=dev).expand(2, -1)
    table = sv.build_neighbor_table(torch.ones(2, 2, 4, 5, dtype=torch.uint8, device=dev), batched=True, n=80)
    x = torch.randn(2, 42, embed, generator=g, device=dev).half().requires_grad_(True)
    go = torch.randn(2, 42, embed, generator=g, device=dev).half()
    wrt = [x] + [p for n, p in mod.named_parameters() if n != "k_norm.bias"]
    scale = [1]

    def step():
        y = mod(x, 4, 5, idx, 40, table)
        return [y.detach(), *torch.autograd.grad(y, wrt, go)]

    plain = step()
    mod.sparse_conv.register_forward_hook(lambda m, args, out: out * scale[0])
    for a, b in zip(plain, step()):
        # a few float16 roundings of each chain; single gains sum products that cancel
        assert float((a - b).float().norm()) <= (4e-3 if a.numel() > 1 else 5e-2) * float(a.float().norm())
    scale[0] = 2
    assert float((step()[0] - plain[0]).float().norm()) > 0.05 * float(plain[0].float().norm())
