"""A shortlist layer whose window covers the sequence: attended causally without
candidate lists, with the lists' telemetry."""
from __future__ import annotations

import pytest
import torch

import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,int8", [(torch.float32, False), (torch.float16, False), (torch.float32, True)])
@pytest.mark.parametrize("graph", [False, True])
def test_full_window_reports_its_rows_candidate_counts(dtype, int8, graph):
    from proteus_attention.models.aspa import AdaptiveSparseAttention, ModelConfig

    T = 300
    cfg = dict(configs.sparse_cfg(T, 64, 4, keep=0.3), attn_quantize_int8=int8)
    m = AdaptiveSparseAttention(ModelConfig(**cfg)).to(device="cuda", dtype=dtype).eval()
    g = torch.Generator().manual_seed(2)
    with torch.no_grad():
        if graph and not int8:
            m.enable_hip_graph(True)
        for _ in range(3):  # (another input each time: a replay's rows are its own)
            m(torch.randn(2, T, 64, generator=g).to(device="cuda", dtype=dtype))
            st = m._last_sparse_state
            n = int(st["row_offsets"].max())
            tokens = st["token_idx"][:n]
            assert n and torch.equal(m._last_shortlist_lengths[:n].long(), tokens.long() + 1)
            assert st["linear_shortlist_candidates"] is False and st["linear_shortlist_structured"] is False
