"""pfa_pack_mask on both sides of its folded-scan rule, against the mask's own
nonzero positions."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,T", [(1, 1), (8, 8192), (5, 2049), (4096, 7), (4097, 7), (3, 100)])
def test_pack_mask_both_sides_of_the_scan_rule(P, T):
    from proteus_attention.kernels.sparse_attn import _pack_mask_i32

    m = torch.rand(P, T, generator=torch.Generator().manual_seed(P)) < 0.3
    m[P // 2] = False
    tok, head, offs, n, mx = _pack_mask_i32(m.cuda())
    want = m.nonzero()
    counts = m.sum(1)
    assert n == want.shape[0] and mx == int(counts.max())
    assert torch.equal(tok.cpu().long(), want[:, 1]) and torch.equal(head.cpu().long(), want[:, 0])
    assert torch.equal(offs.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)]))
