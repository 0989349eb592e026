"""Sequence lengths around the first strided anchor that a row can reach below
its window, where the anchor pass starts to run, against the materialised
candidates."""
from __future__ import annotations

import pytest
import torch

import configs

pytestmark = pytest.mark.gpu


# (window, stride): the first strided anchor below the window lies 256, 300 or 100 tokens back
@pytest.mark.parametrize("w,s,first", [(256, 128, 256), (256, 100, 300), (97, 50, 100)])
@pytest.mark.parametrize("over", [-1, 0, 1, 2, 40])
@pytest.mark.parametrize("H", [16, 4, 2])  # heads of 16, 64 and 128 dims
def test_lengths_around_the_first_anchor(w, s, first, over, H, monkeypatch):
    from proteus_attention.models.aspa import AdaptiveSparseAttention, ModelConfig

    B, C, T = 2, 256, first + over + 1  # over = 0: the last row reaches the anchor at token 0
    m = AdaptiveSparseAttention(ModelConfig(**configs.shortlist_cfg(T, C, H, 1024, w, s)))
    m = m.to(device="cuda", dtype=torch.bfloat16).eval()
    m.record_shortlist_lengths = True
    x = torch.randn(B, T, C, generator=torch.Generator().manual_seed(T)).to(device="cuda", dtype=torch.bfloat16)
    snap = {n: b.detach().clone() for n, b in m.named_buffers() if n.startswith("routing_")}
    out = []
    with torch.no_grad():
        for generic in (False, True):
            if generic:
                monkeypatch.setenv("PFA_FORCE_GENERIC", "1")
            for n, b in snap.items():
                getattr(m, n).copy_(b)
            m(x)
            st = m._last_sparse_state
            # (a window over the whole sequence is attended causally, without the anchor pass)
            assert st["linear_shortlist_structured"] is (not generic and T > w)
            n = int(st["row_offsets"].max())
            out.append((m._last_shortlist_lengths[:n].cpu().long(), m.last_head_consensus.double(), m.qkv(x)))
    (len_s, got, qkv), (len_g, want, _) = out
    assert torch.equal(len_s, len_g)
    # the structured kernel rounds P to bf16 (2^-9 relative each, on v), and both results are bf16
    v = qkv.view(B, T, 3, -1)[:, :, 2].abs().max().double()
    assert float((got - want).abs().max()) <= float(v) * (2.0 ** -9 + 2.0 ** -8)
