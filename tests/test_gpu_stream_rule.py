"""The eager forward on one stream and on two: the same bits."""
from __future__ import annotations

import pytest
import torch

import configs

pytestmark = pytest.mark.gpu

CASES = [("shortlist", torch.bfloat16, {}), ("shortlist", torch.float32, {}), ("shortlist", torch.float16, {}),
         ("shortlist", torch.bfloat16, dict(attn_quantize_int8=True)), ("sparse", torch.bfloat16, {}),
         ("sparse", torch.float32, {}), ("dense", torch.bfloat16, dict(attn_mode="subquad"))]


@pytest.mark.parametrize("form,dtype,extra", CASES)
def test_one_stream_and_two_give_the_same(form, dtype, extra, monkeypatch):
    from proteus_attention.models import aspa

    B, T, C, H = 2, 700, 256, 4
    base = configs.sparse_cfg(T, C, H) if form == "sparse" else configs.shortlist_cfg(T, C, H, 256, window=96, stride=32)
    g = torch.Generator().manual_seed(6)
    xs = [torch.randn(B, T, C, generator=g).to(device="cuda", dtype=dtype) for _ in range(3)]
    seen = []
    for most in (0, 1 << 40):
        monkeypatch.setattr(aspa, "_ONE_STREAM_ELEMS", {dtype: most})
        torch.manual_seed(1)
        m = aspa.AdaptiveSparseAttention(aspa.ModelConfig(**dict(base, **extra))).to(device="cuda", dtype=dtype).eval()
        forks, real = [], m._fork_stream
        m.__dict__["_fork_stream"] = lambda d: (forks.append(1), real(d))[1]
        with torch.no_grad():
            ys = [m(x) for x in xs]  # (the prototypes move with each forward)
        assert bool(forks) == (most == 0)
        seen.append(ys + [m.routing_prototypes, m.routing_usage_ema, m.routing_confidence, m._last_gate_probs])
    for a, b in zip(*seen):
        assert torch.equal(a, b)
