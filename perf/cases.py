"""Workloads that timing and output comparisons of this framework run over.

Five kinds of work, each through the package's public entry points:

* ``conv``: a SparseConv2d layer, as the extension's calls of one training step
  (weight pack, forward, combined backward; how the benchmark counts a step),
  as the module with autograd, or as the module's forward in inference;
* ``depthwise``: the training step of the depthwise layer;
* ``adapter``: the sparse-conv adapter of a ViT block, forward and backward or
  forward alone, under autocast or in one 16-bit type, with the heatmap
  injection or the key-token attention of the configurations that use them;
* ``prune``: the full-grid neighbor table and the token prunes of a forward
  pass over the backbone.

A case names its grid (``B`` samples of ``T`` slices of ``H x W`` cells), the
share of cells it keeps, its widths and its types. Inputs come from the seed
alone: keep sets are a per-sample top-k of a score (uniform, or two drifting
Gaussian blobs per frame), activations are N(0, 1), weights are drawn as the
layers' initialisation draws them.
"""
from __future__ import annotations

import math
import random

import torch

import eccv26_tad_amd as sv

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _conv(name, how, dtype, B, T, H, W, keep, C, masks="uniform"):
    return dict(name=name, kind="conv", how=how, dtype=dtype, B=B, T=T, H=H, W=W, keep=keep, C=C, masks=masks)


def _adapter(name, how, dtype, amp, B, T, H, W, keep, embed, special=1, attn=0, heatmap=False):
    return dict(name=name, kind="adapter", how=how, dtype=dtype, amp=amp, B=B, T=T, H=H, W=W, keep=keep,
                embed=embed, special=special, attn=attn, heatmap=heatmap)


def listed():
    return [
        # one short clip through a ViT-S adapter's layer at inference: launches and host time count
        _conv("conv_infer_c128_f16_clip", "infer", "f16", 1, 8, 14, 14, 0.6, 128),
        # the plumbing configuration: a small float32 layer trained without autocast
        _conv("conv_train_c48_f32", "module", "f32", 1, 8, 14, 14, 0.5, 48),
        # a ViT-S wide layer trained in float32 over whole windows
        _conv("conv_train_c128_f32", "module", "f32", 2, 80, 14, 14, 0.7, 128),
        # the headline layer (4x reduced ViT-B) at the lowest and at the headline keep rate
        _conv("conv_train_c192_f16_keep10", "ops", "f16", 2, 80, 14, 14, 0.10, 192),
        _conv("conv_train_c192_f16_keep55", "ops", "f16", 2, 80, 14, 14, 0.55, 192),
        # a ViT-L adapter's layer in bfloat16
        _conv("conv_train_c256_bf16_keep25", "ops", "bf16", 2, 96, 16, 16, 0.25, 256),
        # the widest layer: long windows, 5 to 15 % of each frame kept
        _conv("conv_train_c512_bf16_ragged", "ops", "bf16", 4, 128, 16, 16, 0.10, 512, masks="ragged"),
        # the depthwise layer on clustered keep sets
        dict(name="depthwise_train_c192_f16_keep55", kind="depthwise", dtype="f16", B=2, T=80, H=14, W=14, keep=0.55,
             C=192, masks="blobs"),
        # a ViT-S adapter serving one window under autocast(bf16), as the test loop runs it
        _adapter("adapter_infer_vits_amp", "infer", "f32", True, 1, 32, 14, 14, 0.6, 384),
        # a ViT-B adapter trained as the training loop does: float32 parameters under autocast(bf16)
        _adapter("adapter_train_vitb_amp", "train", "f32", True, 2, 80, 14, 14, 0.55, 768),
        # the same width with every token's attention to the key tokens (three of them)
        _adapter("adapter_train_vitb_attn2_amp", "train", "f32", True, 2, 80, 14, 14, 0.55, 768, special=3, attn=2),
        # the first two pruning blocks of a ViT-B: table, token gather, table remap
        dict(name="prune_vitb_f16", kind="prune", dtype="f16", B=2, T=80, H=14, W=14, keep=0.7, C=768, special=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["conv16", "conv16", "conv32", "depthwise", "adapter", "adapter", "prune"])
    while True:
        B = rng.randint(1, 4)
        T = _log_int(rng, 4, 128)
        H, W = rng.randint(7, 16), rng.randint(7, 16)
        keep = round(rng.uniform(0.08, 1.0), 3)
        grid = dict(B=B, T=T, H=H, W=W, keep=keep)
        n = B * T * H * W * keep
        if kind == "conv16":
            C = rng.choice([64, 96, 128, 192, 256, 384, 512])
            c = dict(kind="conv", how=rng.choice(["ops", "ops", "module", "infer"]), dtype=rng.choice(["f16", "bf16"]),
                     C=C, masks=rng.choice(["uniform", "ragged", "blobs"]), **grid)
            fits = n * C * C <= 13000 * 512 * 512
        elif kind == "conv32":
            C = rng.choice([32, 48, 64, 96, 128, 192, 256])
            c = dict(kind="conv", how=rng.choice(["ops", "module", "infer"]), dtype="f32", C=C,
                     masks=rng.choice(["uniform", "blobs"]), **grid)
            fits = n * C * C <= 21000 * 128 * 128
        elif kind == "depthwise":
            C = rng.choice([48, 96, 128, 192, 256, 384])
            c = dict(kind="depthwise", dtype=rng.choice(["f16", "bf16", "f32"]), C=C,
                     masks=rng.choice(["uniform", "blobs"]), **grid)
            fits = n * C <= 32000 * 256
        elif kind == "adapter":
            embed = rng.choice([384, 768, 1024])
            amp = rng.random() < 0.7
            heat = rng.random() < 0.25
            attn = 0 if heat else rng.choice([0, 0, 0, 2])
            special = 1 + H * W if heat else rng.randint(1, 4)
            c = dict(kind="adapter", how=rng.choice(["train", "train", "infer"]), amp=amp,
                     dtype="f32" if amp else rng.choice(["f16", "bf16"]), embed=embed, special=special, attn=attn,
                     heatmap=heat, **grid)
            fits = n * embed <= 17500 * 768
        else:
            c = dict(kind="prune", dtype=rng.choice(["f16", "bf16", "f32"]), C=rng.choice([384, 768, 1024]),
                     special=rng.randint(1, 4), **grid)
            fits = B * T * H * W * c["C"] <= 31360 * 768
        if fits and n >= 64:
            return c


# ---------------------------------------------------------------------------
# keep sets and tables in plain PyTorch
# ---------------------------------------------------------------------------

def _dev():
    return torch.device("cuda")


def _gen(seed, salt=0):
    g = torch.Generator(device=_dev())
    g.manual_seed(seed * 1009 + salt)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=_dev())


def _uniform(g, bound, *shape):
    return (torch.rand(*shape, generator=g, device=_dev()) * 2 - 1) * bound


def _frame_counts(c):
    """Kept cells of each frame of a ragged mask: evenly spread over half to
    one and a half times the keep rate."""
    frames, cells = c["B"] * c["T"], c["H"] * c["W"]
    return [min(cells, max(1, round(c["keep"] * cells * (0.5 + (f + 0.5) / frames)))) for f in range(frames)]


def _kept_per_sample(c):
    return math.ceil(c["keep"] * c["T"] * c["H"] * c["W"])


def _rows(c):
    if c.get("masks") == "ragged":
        return sum(_frame_counts(c))
    return c["B"] * _kept_per_sample(c)


def _mask(c, g):
    """uint8 keep mask [B, T, H, W] with _rows(c) kept cells."""
    B, T, H, W = c["B"], c["T"], c["H"], c["W"]
    if c.get("masks") == "ragged":
        counts = torch.tensor(_frame_counts(c), device=_dev())
        counts = counts[torch.randperm(B * T, generator=g, device=_dev())]
        order = torch.rand(B * T, H * W, generator=g, device=_dev()).argsort(1).argsort(1)
        return (order < counts[:, None]).to(torch.uint8).view(B, T, H, W)
    noise = torch.rand(B, T, H, W, generator=g, device=_dev())
    if c.get("masks") == "blobs":
        size = torch.tensor([H - 1.0, W - 1.0], device=_dev())
        walk = torch.cat([torch.rand(B, 1, 2, 2, generator=g, device=_dev()) * size, 0.7 * _randn(g, B, T - 1, 2, 2)], 1)
        centre = torch.remainder(walk.cumsum(1), 2 * size)
        centre = torch.minimum(centre, 2 * size - centre)  # reflected at the borders
        ys = torch.arange(H, device=_dev()).view(1, 1, 1, H, 1)
        xs = torch.arange(W, device=_dev()).view(1, 1, 1, 1, W)
        d2 = (ys - centre[..., 0, None, None]) ** 2 + (xs - centre[..., 1, None, None]) ** 2
        score = torch.exp(-d2 / (2 * 2.5 ** 2)).sum(2) + 1e-3 * noise
    else:
        score = noise
    top = score.view(B, -1).topk(_kept_per_sample(c), dim=1).indices
    return torch.zeros(B, T * H * W, dtype=torch.uint8, device=_dev()).scatter_(1, top, 1).view(B, T, H, W)


def _plain_table(mask):
    """Neighbor table [N, 9] (int64, -1 missing) of a keep mask."""
    B, T, H, W = mask.shape
    kept = mask.reshape(B * T, H, W).bool()
    rank = (kept.reshape(-1).long().cumsum(0) - 1).view(B * T, H, W)
    rank = torch.where(kept, rank, torch.full_like(rank, -1))
    pad = torch.nn.functional.pad(rank, (1, 1, 1, 1), value=-1)
    offs = [pad[:, 1 + dy:1 + dy + H, 1 + dx:1 + dx + W] for dy in (-1, 0, 1) for dx in (-1, 0, 1)]
    return torch.stack(offs, -1).reshape(-1, 9)[kept.reshape(-1)]


def _entries(c):
    """Expected valid table entries: the centre, and each in-frame neighbor
    with the probability that it is kept."""
    H, W, n = c["H"], c["W"], _rows(c)
    around = (3 * H - 2) * (3 * W - 2) / (H * W) - 1
    return n * (1 + around * min(1.0, n / (c["B"] * c["T"] * H * W)))


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------

def _conv_inputs(c, seed):
    g = _gen(seed)
    mask = _mask(c, g)
    n, C, dt = _rows(c), c["C"], DTYPES[c["dtype"]]
    bound = 1.0 / math.sqrt(9 * C)
    x = _randn(g, n, C).to(dt)
    w = _uniform(g, bound, 9, C, C).to(dt)
    b = _uniform(g, bound, C).to(dt)
    go = _randn(g, n, C).to(dt)
    return mask, x, w, b, go


def _depthwise_inputs(c, seed):
    g = _gen(seed)
    mask = _mask(c, g)
    n, C, dt = _rows(c), c["C"], DTYPES[c["dtype"]]
    x = _randn(g, n, C).to(dt)
    w = _uniform(g, 1 / 3, 9, C).to(dt)
    b = _uniform(g, 0.1, C).to(dt)
    go = _randn(g, n, C).to(dt)
    return mask, x, w, b, go


def _hidden(c):
    return 2 ** round(math.log2(c["embed"] // 4))


def _adapter_inputs(c, seed):
    """Mask, kept positions [B, N_kept], x and its output gradient [B, S + N_kept, embed], parameters by name."""
    g = _gen(seed)
    mask = _mask(c, g)
    B, E, h, dt = c["B"], c["embed"], _hidden(c), DTYPES[c["dtype"]]
    idx = mask.view(B, -1).nonzero()[:, 1].view(B, -1)
    N = c["special"] + idx.shape[1]
    x = _randn(g, B, N, E).to(dt)
    # a loss gradient has a mean per channel; without one the scalar gains' gradients cancel down to rounding noise
    go = (_randn(g, B, N, E) + _randn(g, E)).to(dt)
    bound = 1.0 / math.sqrt(9 * h)
    P = {"down_proj.weight": 0.02 * _randn(g, h, E), "down_proj.bias": 0.02 * _randn(g, h),
         "up_proj.weight": 0.02 * _randn(g, E, h), "up_proj.bias": 0.02 * _randn(g, E),
         "sparse_conv.weight": _uniform(g, bound, 9, h, h), "sparse_conv.bias": _uniform(g, bound, h),
         "gamma": 1 + 0.1 * _randn(g, 1)}
    if c["heatmap"]:
        P["heatmap_gate"] = 0.3 + 0.1 * _randn(g, 1)
    if c["attn"]:
        a = h // 2
        P.update({"attn_norm.weight": 1 + 0.1 * _randn(g, h), "attn_norm.bias": 0.1 * _randn(g, h),
                  "attn_gamma": 1 + 0.1 * _randn(g, 1),
                  "down_attn.weight": 0.05 * _randn(g, a, h), "down_attn.bias": 0.02 * _randn(g, a),
                  "qkv.weight": 0.05 * _randn(g, 3 * a, a), "qkv.bias": 0.02 * _randn(g, 3 * a),
                  "q_norm.weight": 1 + 0.1 * _randn(g, a // 4), "q_norm.bias": 0.1 * _randn(g, a // 4),
                  "k_norm.weight": 1 + 0.1 * _randn(g, a // 4), "k_norm.bias": 0.1 * _randn(g, a // 4),
                  "attn_proj.weight": 0.05 * _randn(g, h, a), "attn_proj.bias": 0.02 * _randn(g, h)})
    return mask, idx, x, go, {k: v.to(dt) for k, v in P.items()}


def prepare(case, seed):
    c = case
    if c["kind"] == "conv":
        mask, x, w, b, go = _conv_inputs(c, seed)
        table = sv.build_neighbor_table(mask, n=_rows(c))
        s = dict(c=c, table=table, x=x, w=w, b=b, go=go)
        if c["how"] != "ops":
            mod = sv.SparseConv2d(c["C"], c["C"]).to(_dev(), x.dtype)
            with torch.no_grad():
                mod.weight.copy_(w)
                mod.bias.copy_(b)
            s["mod"] = mod
            if c["how"] == "module":
                x.requires_grad_(True)
        return s
    if c["kind"] == "depthwise":
        mask, x, w, b, go = _depthwise_inputs(c, seed)
        return dict(c=c, table=sv.build_neighbor_table(mask, n=_rows(c)), x=x, w=w, b=b, go=go)
    if c["kind"] == "adapter":
        mask, idx, x, go, P = _adapter_inputs(c, seed)
        kw = dict(heatmap_grid_size=(c["H"], c["W"])) if c["heatmap"] else {}
        mod = sv.SparseConvAdapter(c["embed"], 0.25, use_attn=c["attn"], n_key_tokens=c["special"], **kw)
        mod = mod.to(_dev(), x.dtype)
        with torch.no_grad():
            for name, p in mod.named_parameters():
                if name in P:
                    p.copy_(P[name])
        table = sv.build_neighbor_table(mask, batched=True, n=_rows(c))
        # k_norm.bias adds the same score to every key of a query: its gradient is zero but for rounding noise
        names = [name for name, _ in mod.named_parameters() if name in P and name != "k_norm.bias"]
        if c["how"] == "train":
            x.requires_grad_(True)
        return dict(c=c, mod=mod, names=names, wrt=[x] + [mod.get_parameter(k) for k in names], x=x, go=go, idx=idx,
                    table=table)
    g = _gen(seed)
    B, T, H, W, dt = c["B"], c["T"], c["H"], c["W"], DTYPES[c["dtype"]]
    n0 = T * H * W
    n1 = math.ceil(c["keep"] * n0)
    n2 = math.ceil(c["keep"] * n1)
    keeps = [torch.rand(B, a, generator=g, device=_dev()).topk(b, dim=1).indices.sort(1).values
             for a, b in ((n0, n1), (n1, n2))]
    x = _randn(g, B, c["special"] + n0, c["C"]).to(dt)
    return dict(c=c, x=x, keeps=keeps, idx=torch.arange(n0, device=_dev()).expand(B, -1).contiguous())


# ---------------------------------------------------------------------------
# run
# ---------------------------------------------------------------------------

def run(state):
    s, c = state, state["c"]
    if c["kind"] == "conv":
        if c["how"] == "infer":
            with torch.no_grad():
                return s["mod"](s["x"], s["table"], tokens_per_batch=0)
        if c["how"] == "module":
            y = s["mod"](s["x"], s["table"], tokens_per_batch=0)
            gi, gw, gb = torch.autograd.grad(y, (s["x"], s["mod"].weight, s["mod"].bias), s["go"])
            return {"y": y, "gi": gi, "gw": gw, "gb": gb}
        # the extension's calls of SparseConv2dFunction; the bias rule is the layer's (fp32 add from 128 channels)
        ops, mode = sv.ops, 1 if c["C"] >= 128 else 2
        pf, pb = ops.pack_weight(s["w"], True, True)
        y = ops.fwd_packed(s["x"], s["table"], s["w"], pf, s["b"], 0, mode)
        gi, gw, gb = ops.bwd_packed(s["go"], s["x"], s["table"], s["w"], pb, c["C"], 0, True,
                                    symmetric=sv.is_symmetric_table(s["table"]))
        return {"y": y, "gi": gi, "gw": gw, "gb": gb}
    if c["kind"] == "depthwise":
        y = sv.ops.dw_fwd(s["x"], s["table"], s["w"], s["b"], 0)
        gi, gw, gb = sv.ops.dw_bwd(s["go"], s["x"], s["table"], s["w"], 0, True,
                                   symmetric=sv.is_symmetric_table(s["table"]))
        return {"y": y, "gi": gi, "gw": gw, "gb": gb}
    if c["kind"] == "adapter":
        args = (c["H"], c["W"], s["idx"], c["T"] * c["H"] * c["W"], s["table"])
        amp = torch.autocast("cuda", dtype=torch.bfloat16, enabled=c["amp"])
        if c["how"] == "infer":
            with torch.no_grad(), amp:
                return s["mod"](s["x"], *args)
        with amp:
            y = s["mod"](s["x"], *args)
        grads = torch.autograd.grad(y, s["wrt"], s["go"].to(y.dtype))
        return {"y": y, **dict(zip(["x"] + s["names"], grads))}
    table = sv.get_initial_neighbor_indices(c["H"], c["W"], c["T"], s["x"].device, c["B"])
    x, idx = s["x"], s["idx"]
    for keep in s["keeps"]:
        x, idx, table = sv.prune_tokens(x, keep, idx, table, c["special"])
    return {"x": x, "idx": idx, "table": table}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------

def work(case):
    c = case
    size = {"f16": 2, "bf16": 2, "f32": 4}[c["dtype"]]
    train = c.get("how") != "infer"
    if c["kind"] == "prune":
        n0 = c["T"] * c["H"] * c["W"]
        n1 = math.ceil(c["keep"] * n0)
        n2 = math.ceil(c["keep"] * n1)
        rows = 2 * (2 * c["special"] + n1 + n2)  # each prune reads and writes the rows it keeps
        index = 36 * (n0 + 2 * n1 + n2) + 24 * (n1 + n2)
        return {"bytes": c["B"] * (rows * c["C"] * size + index), "flops": 0}
    n, E = _rows(c), _entries(c)
    if c["kind"] == "depthwise":
        return {"bytes": 4 * n * c["C"] * size + 36 * n + 21 * c["C"] * size, "flops": 3 * 2 * E * c["C"]}
    if c["kind"] == "conv":
        C, passes = c["C"], 3 if train else 1
        acts = 4 if train else 2
        return {"bytes": acts * n * C * size + 36 * n + (2 if train else 1) * (9 * C * C + C) * size,
                "flops": passes * 2 * E * C * C}
    e, h = c["embed"], _hidden(c)
    m = c["B"] * c["special"] + n
    params = (2 * e * h + 9 * h * h) * size
    attn = (h * h // 2 + 3 * h * h // 4 + h * h // 2) if c["attn"] else 0
    return {"bytes": (4 if train else 2) * m * e * size + 36 * n + (2 if train else 1) * params,
            "flops": (3 if train else 1) * 2 * (2 * m * e * h + E * h * h + m * attn)}


def tolerance(case):
    c = case
    if c["kind"] == "prune":
        return "exact"
    if c["kind"] == "adapter":
        # the few key tokens collect every query's rounding in their gradients: single values are off by more there
        return {"rel": 3e-2 if c["amp"] or c["dtype"] == "bf16" else 6e-3, "max": 0.99 if c["attn"] else 0.2}
    # one rounding of an fp32 sum
    return {"rel": {"f16": 1e-3, "bf16": 8e-3, "f32": 1e-5}[c["dtype"]]}


# ---------------------------------------------------------------------------
# the same in plain PyTorch, 64 bits
# ---------------------------------------------------------------------------

def _sparse_conv64(x, table, w, b):
    pad = torch.cat([x, x.new_zeros(1, x.shape[1])])
    y = b.expand(x.shape[0], -1)
    for k in range(9):
        rows = pad.index_select(0, torch.where(table[:, k] < 0, x.shape[0], table[:, k]))
        y = y + (torch.matmul(rows, w[k]) if w.dim() == 3 else rows * w[k])
    return y


def _conv64(c, seed):
    mask, x, w, b, go = (_depthwise_inputs if c["kind"] == "depthwise" else _conv_inputs)(c, seed)
    x, w, b = (t.double().requires_grad_(True) for t in (x, w, b))
    y = _sparse_conv64(x, _plain_table(mask), w, b)
    if c.get("how") == "infer":
        return y.detach()
    gi, gw, gb = torch.autograd.grad(y, (x, w, b), go.double())
    return {"y": y.detach(), "gi": gi, "gw": gw, "gb": gb}


def _adapter64(c, seed):
    F = torch.nn.functional
    mask, idx, x, go, P = _adapter_inputs(c, seed)
    B, S, h = c["B"], c["special"], _hidden(c)
    x = x.double().requires_grad_(True)
    P = {k: v.double().requires_grad_(True) for k, v in P.items()}
    u = F.gelu(F.linear(x, P["down_proj.weight"], P["down_proj.bias"]))
    special, patches = u[:, :S], u[:, S:]
    if c["heatmap"]:
        cells = (idx % (c["H"] * c["W"])).unsqueeze(-1).expand(-1, -1, h)
        patches = patches + torch.gather(special[:, 1:], 1, cells) * P["heatmap_gate"]
    conv = _sparse_conv64(patches.reshape(-1, h), _plain_table(mask), P["sparse_conv.weight"], P["sparse_conv.bias"])
    z = torch.cat([special, conv.view(B, -1, h)], dim=1)
    if c["attn"]:
        a = h // 2
        t = F.linear(F.layer_norm(z, (h,), P["attn_norm.weight"], P["attn_norm.bias"]),
                     P["down_attn.weight"], P["down_attn.bias"])
        q, k, v = F.linear(t, P["qkv.weight"], P["qkv.bias"]).view(B, -1, 3, 4, a // 4).permute(2, 0, 1, 3, 4)
        q = F.layer_norm(q, (a // 4,), P["q_norm.weight"], P["q_norm.bias"])[:, S:]
        k = F.layer_norm(k, (a // 4,), P["k_norm.weight"], P["k_norm.bias"])[:, :S]
        score = (q.unsqueeze(2) * k.unsqueeze(1)).sum(-1) / math.sqrt(a // 4)  # [B, queries, keys, heads]
        att = (torch.softmax(score, 2).unsqueeze(-1) * v[:, None, :S]).sum(2)
        att = torch.cat([torch.zeros_like(v[:, :S]), att], dim=1).reshape(B, -1, a)
        z = z + F.linear(att, P["attn_proj.weight"], P["attn_proj.bias"]) * P["attn_gamma"]
    y = F.linear(z, P["up_proj.weight"], P["up_proj.bias"]) * P["gamma"] + x
    if c["how"] == "infer":
        return y.detach()
    names = [k for k in P if k != "k_norm.bias"]
    grads = torch.autograd.grad(y, [x] + [P[k] for k in names], go.double())
    return {"y": y.detach(), **dict(zip(["x"] + names, grads))}


def exact(case, seed):
    if case["kind"] == "prune":
        return None  # copies and indices: nothing is rounded
    if case["kind"] == "adapter":
        return _adapter64(case, seed)
    return _conv64(case, seed)
