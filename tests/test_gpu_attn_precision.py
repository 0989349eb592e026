"""The tile and union kernels (pfa_tile_attn.h, pfa_cand_attn.h) against the row
kernel (pfa_attn.hip) by their distance from 64-bit results: P and its sums at
no less than the row kernel's f32 precision."""
from __future__ import annotations

import pytest
import torch

from oracle import aspa_oracle as O

pytestmark = pytest.mark.gpu


def _distance(got, want):
    """f32 results: relative 2-norm error; 16-bit results: the share that is not
    the 64-bit result rounded once (the rounding itself hides the sums' error
    from a norm, but not the results that it makes fall on the other side)."""
    if got.dtype == torch.float32:
        return float((got.double() - want).norm() / want.norm())
    return float((got != want.to(got.dtype)).double().mean())


@pytest.mark.parametrize("form", ["causal", "masked", "union"])
@pytest.mark.parametrize("dt", ["f32", "int8", "bf16", "f16"])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
def test_no_further_from_64_bits_than_the_row_kernel(form, dt, D):
    from proteus_attention.kernels.sparse_attn import aspa_sparse_attention

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(21)
    BH, T = 24, 320
    q, k, v = (torch.randn(BH, T, D, generator=g) for _ in range(3))
    kw = {}
    if dt == "int8":
        s = [t.abs().amax(dim=(1, 2)) / 127.0 for t in (q, k, v)]
        q, k, v = ((t / c.view(-1, 1, 1)).round().to(torch.int8) for t, c in zip((q, k, v), s))
        kw = dict(q_scale=s[0].to(dev), k_scale=s[1].to(dev), v_scale=s[2].to(dev))
    else:
        q, k, v = (t.to({"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[dt]) for t in (q, k, v))
    t = torch.arange(T)
    cm = None
    if form == "masked":
        cm = torch.where(t[:, None] >= t[None, :], -0.02 * (t[:, None] - t[None, :]).float(), float("-inf"))
        cm = cm.to({"f16": torch.float16, "bf16": torch.bfloat16}.get(dt, torch.float32))
    want = O.sparse_attention(q, k, v, causal_mask=cm, compute_dtype=torch.float64, out_dtype=torch.float64,
                              **{n: c.cpu() for n, c in kw.items()})
    # the row kernel: the same keys as candidate lists, too few entries for the
    # union kernel (3 << 20, reached by a wide list stride)
    rows = BH * T
    lists = t.to(torch.int32).expand(rows, T).contiguous().to(dev)
    lens = (torch.full((rows,), T) if form == "masked" else (t + 1).repeat(BH)).to(dev)
    assert rows * T < 3 << 20
    args = (q.to(dev), k.to(dev), v.to(dev))
    mask = {} if cm is None else {"causal_mask": cm.to(dev)}
    row = aspa_sparse_attention(*args, shortlist_candidates=lists, shortlist_lengths=lens, **mask, **kw).cpu()
    if form == "union":
        wide = torch.zeros(rows, (3 << 20) // rows + 1, dtype=torch.int32, device=dev)
        wide[:, :T] = lists
        got = aspa_sparse_attention(*args, shortlist_candidates=wide, shortlist_lengths=lens, **kw).cpu()
    else:
        got = aspa_sparse_attention(*args, **mask, **kw).cpu()
    assert not torch.equal(got, row)  # (another kernel)
    near, far = _distance(row, want), _distance(got, want)
    # f32: 7,680 rows with an error of their own each put the ratio of two
    # equal kernels within 1 / sqrt(2 * 7680) = 0.8% of 1 (one sigma).  16
    # bits: n results on the other side of a rounding scatter by sqrt(n) in
    # each kernel
    n = near * want.numel()
    bound = near * 1.03 if got.dtype == torch.float32 else (n + 4 * (2 * n) ** 0.5 + 8) / want.numel()
    print(form, dt, D, near, far)
    assert far <= bound, (near, far)
