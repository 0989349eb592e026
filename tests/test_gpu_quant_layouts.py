"""Per-head int8 over row widths and strides with and without 8-element
accesses, and q, k and v in one call, bit for bit against the oracle."""
from __future__ import annotations

import pytest
import torch

from oracle import aspa_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,D", [(1, 8), (37, 7), (37, 12), (300, 16), (2049, 64), (5, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("mode", ["max", "percentile", "ema_percentile"])
def test_quantize_layouts(T, D, dtype, mode):
    from proteus_attention import _hip
    from proteus_attention.kernels import sparse_attn as sa

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(3)
    for gap in (0, 3, 8):  # elements between rows: 3 breaks the 8-element alignment
        x = torch.randn(3, 4, T, D + gap, generator=g).to(dtype)[..., :D]
        xd = [torch.empty(4, T, D + gap, dtype=dtype, device=dev)[..., :D].copy_(x[i]) for i in range(3)]
        out = [torch.empty(4, T, D, dtype=torch.int8, device=dev) for _ in range(3)]
        scales = torch.empty(3, 4, dtype=torch.float32, device=dev)
        ema0 = torch.rand(3, 4, generator=g) + 1.0
        emas = [ema0[i].to(dev) if mode == "ema_percentile" else None for i in range(3)]
        valid = (True, False, True) if mode == "ema_percentile" else (False,) * 3
        sa.quantize_qkv_int8(tuple(_hip.tensor4(t, 4) for t in xd), dtype, 4, T, D, None, 4, mode, 0.97, 0.9,
                             tuple(emas), valid, tuple(_hip.tensor4(t, 4) for t in out), torch.int8, scales, dev)
        for i in range(3):
            q, s, e = O.quantize_per_head_int8(x[i], mode, 0.97, ema0[i] if valid[i] else None, 0.9)
            got = scales[i].cpu()
            # exact, but for the interpolation of two order statistics, lo +
            # w (hi - lo): torch's CPU lerp may fuse the product into the sum,
            # one rounding of a term below the result (1 ulp), and the EMA and
            # the division by 127 round once more each
            tol = 0.0 if mode == "max" else 3 * 2.0 ** -23
            assert torch.allclose(got, s, rtol=tol, atol=0.0), (gap, i)
            ref = (x[i].float().reshape(4, -1) / got[:, None]).round().clamp(-127, 127).to(torch.int8).view_as(q)
            assert torch.equal(out[i].cpu(), ref), (gap, i)
            if e is not None:
                assert torch.allclose(emas[i].cpu(), e, rtol=tol, atol=0.0)
