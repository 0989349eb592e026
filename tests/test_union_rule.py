"""The rule that lets candidate rows share their neighbours' lists: the spacing
of a head's rows within one batch row."""
from __future__ import annotations

import types

import pytest
import torch

from proteus_attention import _hip
from proteus_attention.kernels import sparse_attn as sa


@pytest.mark.parametrize("dtype,limit", [(torch.float32, 16), (torch.bfloat16, 32), (torch.float16, 32), (torch.int8, 32)])
def test_spacing_counts_one_batch_row(dtype, limit, monkeypatch):
    seen = []

    def fwd(*args):
        seen.append(args[-3])  # the workspace
        return 0

    monkeypatch.setattr(_hip, "lib", lambda: types.SimpleNamespace(pfa_sparse_attn_fwd_ws=fwd))
    monkeypatch.setattr(_hip, "stream_ptr", lambda device: None)
    T, dev, t4 = 960, torch.device("cpu"), _hip.Tensor4()

    def shared(B, H, spacing):
        n = B * H * (T // spacing)
        rows, cand = torch.zeros(n, dtype=torch.int32), torch.zeros(n, 4, dtype=torch.int32)
        sa._attn_launch(t4, t4, t4, dtype, t4, torch.float32, H, T, 64, rows, rows, None, cand, rows, None, None, 1.0,
                        (None, None, None), dev, batch=B)
        return seen[-1] is not None

    for B, H in ((1, 8), (4, 8), (8, 1)):
        assert shared(B, H, limit) and shared(B, H, 1)
        assert not shared(B, H, limit + limit // 4)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_layer_names_its_batch_rows(dtype, monkeypatch):
    from proteus_attention.models.aspa import AdaptiveSparseAttention, ModelConfig

    import configs

    T, B = 256, 3
    m = AdaptiveSparseAttention(ModelConfig(**configs.shortlist_cfg(T, 64, 4, 64, window=32, stride=16)))
    m = m.to(device="cuda", dtype=dtype).eval()
    got, real = [], sa._attn_launch

    def launch(*a, **k):
        got.append((a[6], k.get("batch", 1)))
        return real(*a, **k)

    monkeypatch.setattr(sa, "_attn_launch", launch)
    with torch.no_grad():
        m(torch.randn(B, T, 64, device="cuda", dtype=dtype))
    assert got == [(4, B)]
