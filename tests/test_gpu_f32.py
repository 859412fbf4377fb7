"""The float32 layer's kernels against a float64 scatter over the table's
entries, at row counts and widths around the kernels' blocks and tiles."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.helpers import random_mask

pytestmark = pytest.mark.gpu


@pytest.fixture
def sv():
    import eccv26_tad_amd as sv

    return sv


def _table(rng, n, one_way):
    """Symmetric table [n, 9] (int32) of a random mask cut to n rows, with
    ``one_way`` entries whose partner is removed."""
    import eccv26_tad_amd as sv

    side = 1 + int(np.ceil(np.sqrt(n / 0.5 / 4)))
    mask = np.zeros((1, 4, side, side), dtype=np.uint8)
    while mask.sum() < n:
        mask = random_mask(rng, 1, 4, side, side, min(1.0, 0.6))
        side += 1
    t = sv.build_neighbor_table(torch.from_numpy(mask).cuda()).cpu().numpy()[:n]
    t[t >= n] = -1
    pairs = np.argwhere((t >= 0) & (np.arange(9) != 4))
    for i, k in pairs[rng.permutation(len(pairs))[:one_way]]:
        t[t[i, k], 8 - k] = -1
    if one_way:  # the last row too: the last, partly filled block
        t[n - 1, 0], t[0, 8] = 0, -1
    return t


def _exact(t, x, w, b, go):
    """(y, gi, gw, gb, and the same sums of absolute terms) in float64."""
    n = len(x)
    out = []
    for f in (lambda v: v, np.abs):
        x_, w_, go_, b_ = f(x), f(w), f(go), f(b)
        y = np.tile(b_, (n, 1))
        gi = np.zeros_like(x_)
        gw = np.zeros_like(w_)
        for k in range(9):
            i = np.nonzero(t[:, k] >= 0)[0]
            j = t[i, k]
            y[i] += x_[j] @ w_[k]
            np.add.at(gi, j, go_[i] @ w_[k].T)
            gw[k] = x_[j].T @ go_[i]
        out.append((y, gi, gw, go_.sum(0)))
    return out


def _check(name, got, exact, mag, terms):
    # an fp32 sum of `terms` products in any order: each addition rounds by at
    # most 2^-24 of the sum of absolute terms
    err = np.abs(got.double().cpu().numpy() - exact)
    bar = 2.0 ** -24 * (terms + 2) * mag + 1e-30
    assert (err <= bar).all(), (name, float((err / bar).max()))


@pytest.mark.parametrize("n", [1, 255, 256, 257, 1000])
@pytest.mark.parametrize("one_way", [0, 3])
@pytest.mark.parametrize("dname", ["f32", "f64"])
def test_backward_input_finds_one_way_entries(sv, n, one_way, dname):
    rng = np.random.default_rng(n + one_way)
    t = _table(rng, n, one_way)
    ci, co = 8, 12
    dt = {"f32": torch.float32, "f64": torch.float64}[dname]
    x, w, go, b = (rng.standard_normal(s).astype(np.float32).astype(np.float64)
                   for s in ((n, ci), (9, ci, co), (n, co), (co,)))
    (_, gi, _, _), (_, mag, _, _) = _exact(t, x, w, b, go)
    dev = [torch.from_numpy(v).to("cuda", dt) for v in (go, w)]
    tab = torch.from_numpy(t).cuda()
    got = sv.ops.bwd_in(dev[0], tab, dev[1], n, ci, 0)
    _check("gi", got, gi, mag, 9 * co)
    if not one_way:
        empty = torch.empty(0, dtype=torch.uint8, device="cuda")
        same = sv.ops.bwd_in_packed(dev[0], tab, dev[1], empty, n, ci, 0, symmetric=True)
        assert torch.equal(same, got)


@pytest.mark.parametrize("n,ci,co", [(1, 4, 4), (15, 16, 32), (33, 48, 48), (129, 20, 36), (200, 64, 40),
                                     (257, 100, 128), (300, 128, 96), (1500, 36, 200), (4099, 64, 64)])
@pytest.mark.parametrize("one_way", [0, 2])
def test_layer_matches_float64(sv, n, ci, co, one_way):
    """Forward with bias, backward-input and backward-weight in float32."""
    rng = np.random.default_rng(n + ci + one_way)
    t = _table(rng, n, one_way)
    x, w, go, b = (rng.standard_normal(s).astype(np.float32).astype(np.float64)
                   for s in ((n, ci), (9, ci, co), (n, co), (co,)))
    (y, gi, gw, gb), (my, mgi, mgw, mgb) = _exact(t, x, w, b, go)
    X, W, GO, B = (torch.from_numpy(v).to("cuda", torch.float32) for v in (x, w, go, b))
    tab = torch.from_numpy(t).cuda()
    for mode in (1, 2):
        _check("y", sv.ops.fwd_bias(X, tab, W, B, 0, mode), y, my, 9 * ci + 1)
    _check("y - b", sv.ops.fwd(X, tab, W, co, 0), y - b, my, 9 * ci + 1)
    _check("gi", sv.ops.bwd_in(GO, tab, W, n, ci, 0), gi, mgi, 9 * co)
    for bias in (True, False):
        got_w, got_b = sv.ops.bwd_w_bias(GO, X, tab, ci, 0, bias)
        _check("gw", got_w, gw, mgw, n)
        if bias:
            _check("gb", got_b, gb, mgb, n)
    if not one_way:
        empty = torch.empty(0, dtype=torch.uint8, device="cuda")
        _check("gi", sv.ops.bwd_in_packed(GO, tab, W, empty, n, ci, 0, symmetric=True), gi, mgi, 9 * co)


@pytest.mark.parametrize("n,ci,co", [(3601, 512, 512), (15001, 256, 256)])
def test_backward_weight_of_long_splits(sv, n, ci, co):
    """Splits of more rows than the kernel lists at once (1024), the last one
    and its last list uneven; the workspace holds one partial per split."""
    import ctypes
    import os

    lib = ctypes.CDLL(os.path.join(os.path.dirname(sv.__file__), "libsvtad_sparse.so"))
    lib.svtad_bwd_w_workspace_bytes.restype = ctypes.c_size_t
    lib.svtad_bwd_w_workspace_bytes.argtypes = [ctypes.c_int64] + [ctypes.c_int] * 3
    splits = lib.svtad_bwd_w_workspace_bytes(n, ci, co, 0) // ((9 * ci * co + co) * 4)
    assert 1 <= splits and -(-n // splits) > 1024
    terms = -(-n // splits) + 32 + splits  # a split's rows one after another, then the splits
    rng = np.random.default_rng(n)
    t = torch.from_numpy(_table(rng, n, 2)).cuda()
    x, go = (torch.from_numpy(rng.standard_normal((n, c)).astype(np.float32)).cuda() for c in (ci, co))
    got_w, got_b = sv.ops.bwd_w_bias(go, x, t, ci, 0, True)
    for k in range(9):
        i = (t[:, k] >= 0).nonzero()[:, 0]
        xs, gs = x[t[i, k].long()].double(), go[i].double()
        _check("gw", got_w[k], (xs.t() @ gs).cpu().numpy(), (xs.abs().t() @ gs.abs()).cpu().numpy(), terms)
    g = go.double()
    _check("gb", got_b, g.sum(0).cpu().numpy(), g.abs().sum(0).cpu().numpy(), terms)
