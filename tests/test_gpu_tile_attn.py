"""The tile kernel of the causal and masked branches (pfa_tile_attn.h) at the
edges of its tiles, key splits and row blocks, against the oracle in 64 bits."""
from __future__ import annotations

import pytest
import torch

from oracle import aspa_oracle as O

pytestmark = pytest.mark.gpu

# relative 2-norm error of one rounding of the result (f16: 2^-11, bf16: 2^-8
# at most) and, in f32, of sums of up to 800 f32 products; twice each
TOL = {"f32": 2e-6, "int8": 2e-6, "f16": 1e-3, "bf16": 8e-3}


def _inputs(dt, BH, T, D, g):
    q, k, v = (torch.randn(BH, T, D, generator=g) for _ in range(3))
    if dt != "int8":
        td = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[dt]
        return [t.to(td) for t in (q, k, v)], {}
    s = [t.abs().amax(dim=(1, 2)) / 127.0 for t in (q, k, v)]
    q, k, v = ((t / c.view(-1, 1, 1)).round().to(torch.int8) for t, c in zip((q, k, v), s))
    return [q, k, v], dict(q_scale=s[0], k_scale=s[1], v_scale=s[2])


def _mask(T, dt, g):
    cm = torch.randn(T, T, generator=g)
    cm[torch.rand(T, T, generator=g) < 0.3] = float("-inf")
    cm[:, 0] = 0.5
    return cm.to({"f16": torch.float16, "bf16": torch.bfloat16}.get(dt, torch.float32))


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "int8"])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("masked", [False, True])
def test_tile_attention_edges(dt, D, masked):
    """Lengths around a tile, heads that share a row block, one row, and at 32
    and 64 dims enough rows for each key split (blocks of 64 rows <= 256, <= 768,
    above; every width, over many tiles: test_gpu_attn_precision.py)."""
    from proteus_attention.kernels.sparse_attn import aspa_sparse_attention

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(7)
    sizes = [(1, 1, 1.0), (3, 7, 0.6), (2, 65, 1.0), (5, 130, 0.4), (2, 777, 0.5)]
    if D in (32, 64):
        sizes += [(200, 120, 0.9), (700, 80, 0.9)]  # 338 and 788 row blocks
    for BH, T, frac in sizes:
        (q, k, v), kw = _inputs(dt, BH, T, D, g)
        act = torch.rand(BH, T, generator=g) < frac
        act[0, 0] = True
        cm = _mask(T, dt, g) if masked else None
        want = O.sparse_attention(q, k, v, active_mask=act, causal_mask=cm, compute_dtype=torch.float64,
                                  out_dtype=torch.float64, **kw)
        dkw = {n: t.to(dev) for n, t in kw.items()}
        got = aspa_sparse_attention(q.to(dev), k.to(dev), v.to(dev), active_mask=act.to(dev),
                                    causal_mask=None if cm is None else cm.to(dev), **dkw).cpu()
        err = float((got.double() - want).norm() / want.norm())
        assert err <= TOL[dt], (BH, T, err)
        assert torch.equal(got[~act], torch.zeros_like(got[~act]))


@pytest.mark.parametrize("dt", ["f32", "f16"])
def test_tile_attention_strided_and_nonfinite(dt):
    """Views with gaps between rows and heads, rows given in any order, and
    infinities and NaN in keys that a row does not reach."""
    from proteus_attention.kernels.sparse_attn import aspa_sparse_attention

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(8)
    (q, k, v), _ = _inputs(dt, 2, 100, 64, g)
    wide = torch.stack((q, k, v), dim=2).to(dev)  # (BH, T, 3, D): row stride 3D
    heads, toks = torch.ones(2, 100).nonzero(as_tuple=True)
    perm = torch.cat([torch.randperm(100, generator=g), 100 + torch.randperm(100, generator=g)])
    pre = (heads[perm].to(dev), toks[perm].to(dev), torch.tensor([0, 100, 200], dtype=torch.int32, device=dev), 100)
    want = O.sparse_attention(q, k, v, compute_dtype=torch.float64, out_dtype=torch.float64)
    got = aspa_sparse_attention(wide[:, :, 0], wide[:, :, 1], wide[:, :, 2], prepacked=pre).cpu()
    assert float((got.double() - want).norm() / want.norm()) <= TOL[dt]
    v[0, 60], k[1, 50] = float("inf"), float("nan")
    got = aspa_sparse_attention(q.to(dev), k.to(dev), v.to(dev)).cpu()
    assert torch.isfinite(got[0, :60]).all() and torch.isfinite(got[1, :50]).all()
    assert float((got[0, :60].double() - want[0, :60]).norm() / want[0, :60].norm()) <= TOL[dt]
    assert not torch.isfinite(got[0, 60:]).any() and torch.isnan(got[1, 50:]).all()
