"""A graph capture where the memory that it needs sits in the allocator's cache:
a capture cannot release cached blocks itself."""
from __future__ import annotations

import gc

import pytest
import torch

import configs

pytestmark = pytest.mark.gpu


def test_capture_when_its_memory_is_cached():
    from proteus_attention.models.aspa import AdaptiveSparseAttention, ModelConfig

    dev, T = torch.device("cuda:0"), 32768
    m = AdaptiveSparseAttention(ModelConfig(**configs.shortlist_cfg(T, 512, 8, 1024, window=256, stride=128)))
    m = m.to(device=dev, dtype=torch.bfloat16).eval()
    x = torch.randn(1, T, 512, device=dev).to(torch.bfloat16)
    with torch.no_grad():
        want = m(x).clone()
        m.enable_hip_graph(True, static_output=True)
        m.hip_graph_input(x)  # the warm-up's blocks stay cached for its stream
        m.reset_hip_graphs()
        gc.collect()
        torch.cuda.synchronize(dev)
        # room for little beyond what is reserved; the cache holds more than the capture takes
        reserved, total = torch.cuda.memory_reserved(dev), torch.cuda.mem_get_info(dev)[1]
        assert reserved - torch.cuda.memory_allocated(dev) > 256 << 20
        torch.cuda.set_per_process_memory_fraction((reserved + (8 << 20)) / total, dev)
        try:
            y = m(m.hip_graph_input(x))
            assert torch.isfinite(y).all() and y.shape == want.shape
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0, dev)
