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
