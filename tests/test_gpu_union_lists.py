"""The union kernel's key list (pfa_cand_attn.h): more keys than it holds at a
time, in one range of the table and over several, and a key named twice after
some were attended."""
from __future__ import annotations

import pytest
import torch

from test_gpu_attn_precision import _inputs

pytestmark = pytest.mark.gpu

TOL = {"f32": 2e-6, "int8": 2e-6, "f16": 1e-3, "bf16": 8e-3}


def _lists(kind, T, rows, g):
    """Per row, nine tenths of the keys common to all rows, in any order."""
    def some(lo, hi, n):
        return lo + torch.randperm(hi - lo, generator=g)[:n]

    common = {"split": lambda: some(0, 8192, 5300),            # more than the list in one range
              "full_half": lambda: torch.cat([torch.arange(4096), some(4096, 8192, 300)]),
              "ranges": lambda: torch.cat([some(0, 8192, 3000), some(8192, 16384, 3000)]),
              "late_twice": lambda: torch.cat([some(0, 8192, 3000), some(8192, 16384, 3000)]),
              "ranges_split": lambda: torch.cat([some(0, 8192, 3000), some(8192, 16384, 200), some(16384, T, 5000)]),
              }[kind]()
    out = []
    for r in range(rows):
        c = common[torch.randperm(common.numel(), generator=g)]
        if kind != "full_half" or r % 16:  # (one row of each sixteen lists them all)
            c = c[: common.numel() * 9 // 10]
        if kind == "late_twice" and r % 16 == 7:
            c[3] = c[c > 8192][5]
        out.append(c)
    return out


@pytest.mark.parametrize("kind,T", [("split", 9000), ("full_half", 8192), ("ranges", 16384), ("late_twice", 16384),
                                    ("ranges_split", 24000)])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "int8"])
def test_more_keys_than_the_list_holds(kind, T, D, dt, monkeypatch):
    from proteus_attention.kernels import sparse_attn as sa

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(31)
    (q, k, v), kw = _inputs(dt, 2, T, D, g)
    act = torch.zeros(2, T, dtype=torch.bool)
    act[0, torch.randperm(T, generator=g)[:37]] = True  # the third block of sixteen holds rows of both heads
    act[1, torch.randperm(T, generator=g)[:27]] = True
    heads, toks = act.nonzero(as_tuple=True)
    lists = _lists(kind, T, 64, g)
    wide = torch.zeros(64, (3 << 20) // 64, dtype=torch.int32)
    for r, c in enumerate(lists):
        wide[r, : c.numel()] = c
    lens = torch.tensor([c.numel() for c in lists])
    spaces, real = [], sa._workspace

    def workspace(nbytes, device):
        spaces.append(real(nbytes, device).fill_(0xAA))
        return spaces[-1]

    monkeypatch.setattr(sa, "_union_rows", lambda *a: True)
    monkeypatch.setattr(sa, "_workspace", workspace)
    got = sa.aspa_sparse_attention(q, k, v, active_mask=act.to(dev), shortlist_candidates=wide.to(dev),
                                   shortlist_lengths=lens.to(dev), **kw)
    # (a block is left to the row kernel only where a list names a key twice)
    assert spaces[-1][:4].tolist() == [1 if kind == "late_twice" else 0] * 4
    sc = [kw[n].double() if kw else torch.ones(2, dtype=torch.float64, device=dev) for n in ("q_scale", "k_scale", "v_scale")]
    want = torch.zeros(q.shape, dtype=torch.float64, device=dev)
    for r in range(64):
        h, t, c = int(heads[r]), int(toks[r]), lists[r].to(dev)
        s = (k[h, c].double() * sc[1][h]) @ (q[h, t].double() * sc[0][h]) / D ** 0.5
        want[h, t] = torch.softmax(s, 0) @ (v[h, c].double() * sc[2][h])
    assert float((got.double() - want).norm() / want.norm()) <= TOL[dt]
    assert int(torch.count_nonzero(got[~act.to(dev)])) == 0
