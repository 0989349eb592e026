"""The tile and union kernels (pfa_tile_attn.h, pfa_cand_attn.h) against the row
kernel (pfa_attn.hip) by their distance from 64-bit results: P and its sums at
no less than the row kernel's f32 precision."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _distance(got, want):
    """f32 results: relative 2-norm error; 16-bit results: the share that is not
    the 64-bit result rounded once (the rounding itself hides the sums' error
    from a norm, but not the results that it makes fall on the other side)."""
    if got.dtype == torch.float32:
        return float((got.double() - want).norm() / want.norm())
    return float((got != want.to(got.dtype)).double().mean())


def _inputs(dt, BH, T, D, g):
    """q, k, v on the device and the int8 scales by their argument names."""
    q, k, v = (torch.randn(BH, T, D, generator=g) for _ in range(3))
    if dt != "int8":
        td = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dt]
        return [t.to(td).cuda() for t in (q, k, v)], {}
    s = [t.abs().amax(dim=(1, 2)) / 127.0 for t in (q, k, v)]
    q, k, v = ((t / c.view(-1, 1, 1)).round().to(torch.int8).cuda() for t, c in zip((q, k, v), s))
    return [q, k, v], {n: c.cuda() for n, c in zip(("q_scale", "k_scale", "v_scale"), s)}


def _exact(q, k, v, cm, scales):
    """Causal or masked attention of every row in 64 bits."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    sc = [scales.get(n) for n in ("q_scale", "k_scale", "v_scale")]
    future = torch.ones(q.size(1), q.size(1), dtype=torch.bool, device=q.device).triu(1)
    for h in range(q.size(0)):
        a, b, c = (t[h].double() * (1.0 if x is None else x[h].double()) for t, x in zip((q, k, v), sc))
        s = (a @ b.t()) / q.size(2) ** 0.5
        s = s.masked_fill(future, float("-inf")) if cm is None else s + cm.double()
        out[h] = torch.softmax(s, dim=-1) @ c
    return out


# 64-row blocks: 120 (keys split four or two ways), 525 (two ways, f32 and 128
# dims whole) and 850 (whole)
@pytest.mark.parametrize("form,BH,T", [("causal", 24, 320), ("masked", 24, 320), ("union", 24, 320),
                                       ("causal", 48, 700), ("masked", 48, 700),
                                       ("causal", 64, 850), ("masked", 64, 850)])
@pytest.mark.parametrize("dt", ["f32", "int8", "bf16", "f16"])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
def test_no_further_from_64_bits_than_the_row_kernel(form, BH, T, dt, D, monkeypatch):
    from proteus_attention.kernels import sparse_attn as sa

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(21)
    (q, k, v), kw = _inputs(dt, BH, T, D, g)
    t, cm = torch.arange(T), None
    if form == "masked":
        cm = torch.where(t[:, None] >= t[None, :], -0.02 * (t[:, None] - t[None, :]).float(), float("-inf"))
        cm = cm.to({"f16": torch.float16, "bf16": torch.bfloat16}.get(dt, torch.float32)).to(dev)
    want = _exact(q, k, v, cm, kw)
    # the row kernel: the same keys as candidate lists, no neighbours' lists shared
    rows = BH * T
    lists = t.to(torch.int32).to(dev).expand(rows, T).contiguous()
    lens = (torch.full((rows,), T) if form == "masked" else (t + 1).repeat(BH)).to(dev)
    with monkeypatch.context() as mp:
        mp.setattr(sa, "_union_rows", lambda *a: False)
        row = sa.aspa_sparse_attention(q, k, v, shortlist_candidates=lists, shortlist_lengths=lens, causal_mask=cm, **kw)
    if form == "union":
        wide = torch.zeros(rows, (3 << 20) // rows + 1, dtype=torch.int32, device=dev)
        wide[:, :T] = lists
        got = sa.aspa_sparse_attention(q, k, v, shortlist_candidates=wide, shortlist_lengths=lens, **kw)
    else:
        monkeypatch.setattr(sa, "_CAUSAL_TILE_BLOCKS", {D: None})  # bf16 on the tiles at any size
        got = sa.aspa_sparse_attention(q, k, v, causal_mask=cm, **kw)
    assert not torch.equal(got, row)  # (another kernel)
    near, far = _distance(row, want), _distance(got, want)
    # f32: 7,680 rows and more with an error of their own each put the ratio of
    # two equal kernels within 1 / sqrt(2 * 7680) = 0.8% of 1 (one sigma).  16
    # bits: n results on the other side of a rounding scatter by sqrt(n) in
    # each kernel
    n = near * want.numel()
    bound = near * 1.03 if got.dtype == torch.float32 else (n + 4 * (2 * n) ** 0.5 + 8) / want.numel()
    assert far <= bound, (near, far)
