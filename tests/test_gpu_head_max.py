"""Masked rows whose head's last key does not lie in the sequence: keys are read
inside it, as by the row kernel."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 64, 128])
def test_last_key_outside_the_sequence(dtype, D):
    from proteus_attention import _hip
    from proteus_attention.kernels import sparse_attn as sa

    dev, BH, T = torch.device("cuda:0"), 3, 100
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(BH, T, D, generator=g).to(dtype).to(dev) for _ in range(3))
    heads, toks = (t.to(torch.int32).to(dev) for t in torch.ones(BH, T).nonzero(as_tuple=True))
    mask = torch.randn(T, T, generator=g).to(dtype).to(dev)
    t4 = [_hip.tensor4(t, BH) for t in (q, k, v)]

    def run(last):
        out = torch.zeros_like(q)
        sa._attn_launch(*t4, dtype, _hip.tensor4(out, BH), dtype, BH, T, D, toks, heads, None, None, None, mask,
                        torch.tensor(last, dtype=torch.int32, device=dev), D ** -0.5, (None, None, None), dev)
        return out.cpu()

    want = run([T - 1] * 3)
    got = run([T + 700, -1, T - 1])
    assert torch.isfinite(want).all()
    assert torch.equal(got[0], want[0]) and torch.equal(got[2], want[2]) and torch.isnan(got[1]).all()


def test_prepacked_offsets_without_a_heads_rows():
    """A head that the offsets give no rows has no last key: NaN rows, no read
    outside k and v."""
    from proteus_attention.kernels.sparse_attn import aspa_sparse_attention

    dev, T = torch.device("cuda:0"), 70
    q, k, v = (torch.randn(2, T, 64, device=dev) for _ in range(3))
    heads, toks = (t.to(dev) for t in torch.ones(2, T).nonzero(as_tuple=True))
    pre = (heads, toks, torch.tensor([0, 0, 2 * T], dtype=torch.int32, device=dev), T)
    got = aspa_sparse_attention(q, k, v, prepacked=pre, causal_mask=torch.zeros(T, T, device=dev))
    assert torch.isnan(got[0]).all() and torch.isfinite(got[1]).all()
