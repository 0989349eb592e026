"""Paths of the causal and masked branches that depend on values, strides and
size: rows computed again because their result is not finite, 64-bit key
addresses, and the structured kernel as a causal tile above the tile kernel's
lines."""
from __future__ import annotations

import pytest
import torch

from test_gpu_attn_precision import _exact, _inputs

pytestmark = pytest.mark.gpu

# twice the relative 2-norm of one rounding of the result (2^-8 and 2^-11 at
# most), in f32 of sums of up to 900 products
TOL = {"f32": 2e-6, "int8": 2e-6, "f16": 1e-3, "bf16": 8e-3}


def _err(got, want):
    return float((got.double() - want).norm() / want.norm())


def _by_rows(sa, monkeypatch, q, k, v, cm, kw):
    BH, T = q.shape[:2]
    lists = torch.arange(T, dtype=torch.int32, device=q.device).expand(BH * T, T).contiguous()
    lens = torch.full((BH * T,), T, device=q.device) if cm is not None else (torch.arange(T, device=q.device) + 1).repeat(BH)
    with monkeypatch.context() as mp:
        mp.setattr(sa, "_union_rows", lambda *a: False)
        return sa.aspa_sparse_attention(q, k, v, shortlist_candidates=lists, shortlist_lengths=lens, causal_mask=cm, **kw)


# rows for each key split: blocks of 64 rows <= 256, <= 768, above
@pytest.mark.parametrize("BH,T", [(3, 100), (90, 200), (300, 180)])
@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "int8"])
@pytest.mark.parametrize("masked", [False, True])
def test_nonfinite_rows_as_by_the_row_kernel(BH, T, D, dt, masked, monkeypatch):
    from proteus_attention.kernels import sparse_attn as sa

    g = torch.Generator().manual_seed(9)
    (q, k, v), kw = _inputs(dt, BH, T, D, g)
    cm = None
    if masked:
        cm = torch.randn(T, T, generator=g)
        cm[torch.rand(T, T, generator=g) < 0.3] = float("-inf")
        cm[:, 0] = 0.5
        cm[5] = float("-inf")  # a row without a key
        cm = cm.to({"f16": torch.float16, "bf16": torch.bfloat16}.get(dt, torch.float32)).cuda()
    if dt == "int8":
        kw["v_scale"][0], kw["k_scale"][BH - 1] = float("inf"), float("nan")
    else:
        v[0, 60, D // 2], k[BH - 1, 50, 3] = float("inf"), float("nan")
        q[1, 70, 1] = float("-inf")
    monkeypatch.setattr(sa, "_CAUSAL_TILE_BLOCKS", {D: None})
    got = sa.aspa_sparse_attention(q, k, v, causal_mask=cm, **kw)
    want = _by_rows(sa, monkeypatch, q, k, v, cm, kw)
    assert not torch.isfinite(want).all() and torch.isfinite(want).any()
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(got), kind(want))
    ok = torch.isfinite(want)
    assert _err(got[ok], want[ok].double()) <= TOL[dt]


@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "int8"])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("one", ["k", "v"])
def test_rows_that_share_one_key_row(D, dt, masked, one):
    """k or v without a step between its rows (expanded): addresses in 64 bits."""
    from proteus_attention.kernels.sparse_attn import aspa_sparse_attention

    BH, T = 5, 150
    g = torch.Generator().manual_seed(10)
    (q, k, v), kw = _inputs(dt, BH, T, D, g)
    if one == "k":
        k = k[:, :1].expand(-1, T, -1)
    else:
        v = v[:, :1].expand(-1, T, -1)
    cm = torch.randn(T, T, generator=g).to({"f16": torch.float16, "bf16": torch.bfloat16}.get(dt, torch.float32)).cuda()
    cm = cm if masked else None
    got = aspa_sparse_attention(q, k, v, causal_mask=cm, **kw)
    assert _err(got, _exact(q, k, v, cm, kw)) <= TOL[dt]


@pytest.mark.parametrize("BH,T,D", [(17, 3900, 64), (9, 1900, 128)])
def test_operator_causal_above_the_tiles_line(BH, T, D, monkeypatch):
    """1,036 blocks of 64 rows at 64 dims, 268 at 128: the structured kernel."""
    from proteus_attention.kernels import sparse_attn as sa

    g = torch.Generator().manual_seed(12)
    (q, k, v), _ = _inputs("bf16", BH, T, D, g)
    calls, real = [], sa._causal_attn_mfma
    monkeypatch.setattr(sa, "_causal_attn_mfma", lambda *a: (calls.append(1), real(*a))[1])
    monkeypatch.setattr(sa, "_attn_launch", None)
    got = sa.aspa_sparse_attention(q, k, v)
    assert calls and sa.get_last_backend_info()["details"]["mfma"] is True
    assert _err(got, _exact(q, k, v, None, {})) <= TOL["bf16"]


def test_module_force_dense_above_the_tiles_line(monkeypatch):
    from configs import COMMON
    from oracle import aspa_oracle as O

    from proteus_attention.kernels import sparse_attn as sa
    from proteus_attention.models.aspa import AdaptiveSparseAttention, ModelConfig

    dev, T, C, H = torch.device("cuda:0"), 8300, 512, 8  # 1,038 blocks
    torch.manual_seed(0)
    m = AdaptiveSparseAttention(ModelConfig(**dict(COMMON, d_model=C, n_head=H, attn_h_total=H, attn_gates=H,
                                                   attn_mode="subquad", attn_token_sparse=False)))
    m = m.to(dev, torch.bfloat16).eval()
    x = torch.randn(1, T, C, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(dev)
    calls, real = [], sa._causal_attn_mfma
    monkeypatch.setattr(sa, "_causal_attn_mfma", lambda *a: (calls.append(1), real(*a))[1])
    with torch.no_grad():
        m(x)
        qkv = m.qkv(x).view(1, T, 3, H, 64)
    assert calls and m._last_sparse_state["mode"].startswith("dense")
    cos, sin = m._rope_factors(T, dev, torch.bfloat16)
    q, k = (O.apply_rope(qkv[:, :, i].cpu(), cos.cpu(), sin.cpu()).to(dev) for i in range(2))
    q, k, v = (t[0].permute(1, 0, 2).contiguous() for t in (q, k, qkv[:, :, 2]))
    want = _exact(q, k, v, None, {}).permute(1, 0, 2).reshape(1, T, C)
    assert _err(m.last_head_consensus, want) <= TOL["bf16"]
