"""pfa_router_tail against the entry points it joins, bit for bit."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_parts", [0, 1, 15, 16, 17, 129, 1100])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_router_tail_bitwise(n_parts, dtype):
    from proteus_attention import _hip

    dev = torch.device("cuda:0")
    lib, st = _hip.lib(), _hip.stream_ptr(dev)
    g = torch.Generator().manual_seed(5)
    for G, C in ((1, 8), (8, 256), (16, 130)):
        part = torch.rand(max(1, n_parts), G, C + 1, generator=g)
        part[:, 0, C] *= 1e-9 if G > 1 else 1.0  # a gate without tokens is left as it is
        bufs = [torch.randn(s, generator=g).to(dtype).to(dev) for s in ((G, C), (G,), (G,))]
        stats = torch.rand(max(1, n_parts), 8, generator=g).to(dev)
        heads = torch.randint(0, 99, (n_parts % 7,), generator=g, dtype=torch.int32).to(dev)
        tag = _hip.dtype_tag(dtype)
        want_p, want_b = part.to(dev), [b.clone() for b in bufs]
        want_s = torch.empty(G, C + 1, device=dev)
        want_o, got_o = (torch.zeros(8, dtype=torch.float64, device=dev) for _ in range(2))
        _hip.check(lib.pfa_router_stats_reduce(_hip.ptr(stats), stats.size(0), _hip.ptr(want_o), st), "stats")
        if n_parts:
            _hip.check(lib.pfa_proto_partial_reduce(_hip.ptr(want_p), n_parts, G, C, _hip.ptr(want_s), st), "reduce")
            _hip.check(lib.pfa_proto_ema_update(_hip.ptr(want_s), G, C, 0.97, *(_hip.ptr(b) for b in want_b), tag, st),
                       "ema")
        got_p, got_s = part.to(dev), torch.empty(G, C + 1, device=dev)
        h64 = torch.empty(heads.numel(), dtype=torch.int64, device=dev)
        _hip.check(lib.pfa_router_tail(_hip.ptr(got_p), n_parts, G, C, 0.97, _hip.ptr(got_s),
                                       *(_hip.ptr(b) for b in bufs), tag, _hip.ptr(stats), stats.size(0),
                                       _hip.ptr(got_o), _hip.ptr(heads), heads.numel(), _hip.ptr(h64), st), "tail")
        assert torch.equal(got_o, want_o) and torch.equal(h64, heads.long())
        assert all(torch.equal(a, b) for a, b in zip(bufs, want_b))
        if n_parts:
            assert torch.equal(got_s, want_s)
