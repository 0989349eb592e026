"""Candidate attention over the union of sixteen lists (pfa_cand_attn.h): lists
of several ranges, shared and unshared, unsorted, repeated or out of range, some
attended by the union kernel and some left by it to the row kernel, against the
oracle in 64 bits.  (More keys than the kernel lists at a time:
test_gpu_union_lists.py.)"""
from __future__ import annotations

import pytest
import torch

from oracle import aspa_oracle as O

pytestmark = pytest.mark.gpu

# twice the relative 2-norm of one rounding of the result, in f32 of its sums
TOL = {"f32": 2e-6, "int8": 2e-6, "f16": 1e-3, "bf16": 8e-3}


def _lists(kind, n, T, L, toks, g):
    if kind == "shared":  # a window that neighbours share, then lone keys
        w = L // 2
        win = (toks[:, None] - torch.arange(w)).clamp(min=0)
        lone = (toks[:, None] - w - 7 * torch.arange(L - w)).clamp(min=0)
        cand = torch.cat([win, lone], 1)
        keep = torch.zeros(n, T, dtype=torch.bool).scatter_(1, cand, True)  # each key once
        lens = keep.sum(1)
        order = torch.argsort(keep.to(torch.int8), dim=1, descending=True, stable=True)[:, :L]
        return order, lens
    cand = torch.stack([torch.randperm(T, generator=g)[:L] for _ in range(n)])  # unsorted, little shared
    lens = torch.randint(1, L + 1, (n,), generator=g)
    if kind == "twice":
        cand[::5, 1] = cand[::5, 0]
        lens.clamp_(min=2)
    if kind == "outside":  # clamped to the first and the last key
        cand[::3, 0], cand[::3, 1] = -4, T + 3
    return cand, lens


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16", "int8"])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("kind", ["shared", "random", "twice", "outside"])
def test_candidate_union_vs_oracle(dt, D, kind):
    from proteus_attention.kernels.sparse_attn import aspa_sparse_attention

    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(11)
    # one range of the key table; several, with a list read again (over 512
    # entries); rows of many heads in one block of sixteen
    for BH, T, L, frac in ((3, 700, 600, 0.6), (1, 9000, 900, 0.08), (400, 9, 9, 0.5)):
        q, k, v = (torch.randn(BH, T, D, generator=g) for _ in range(3))
        kw = {}
        if dt == "int8":
            s = [t.abs().amax(dim=(1, 2)) / 127.0 for t in (q, k, v)]
            q, k, v = ((t / c.view(-1, 1, 1)).round().to(torch.int8) for t, c in zip((q, k, v), s))
            kw = dict(q_scale=s[0], k_scale=s[1], v_scale=s[2])
        else:
            td = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[dt]
            q, k, v = q.to(td), k.to(td), v.to(td)
        act = torch.rand(BH, T, generator=g) < frac
        act[0, 0] = True
        toks = act.nonzero()[:, 1]
        n = int(toks.numel())
        cand, lens = _lists(kind, n, T, L, toks, g)
        want = O.sparse_attention(q, k, v, active_mask=act, shortlist_candidates=cand, shortlist_lengths=lens,
                                  compute_dtype=torch.float64, out_dtype=torch.float64, **kw)
        # the union kernel whatever the size of the call: the rule's lower
        # bound on N * L is met by a wide list stride
        wide = torch.zeros(n, max(L, (3 << 20) // n + 1), dtype=torch.int32, device=dev)
        wide[:, :L] = cand.to(dev)
        args = dict(active_mask=act.to(dev), shortlist_candidates=wide, shortlist_lengths=lens.to(dev),
                    **{m: t.to(dev) for m, t in kw.items()})
        qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
        got = aspa_sparse_attention(qd, kd, vd, **args).cpu()
        err = float((got.double() - want).norm() / want.norm())
        assert err <= TOL[dt], (BH, T, kind, err)
        assert torch.equal(got[~act], torch.zeros_like(got[~act]))
        if dt == "f32":  # an infinite value reaches the rows that list its key, and no other
            vd[0, T // 2] = float("inf")
            got = aspa_sparse_attention(qd, kd, vd, **args).cpu()
            c = cand.clamp(0, T - 1)
            listed = ((c == T // 2) & (torch.arange(L) < lens[:, None])).any(1)
            heads = act.nonzero()[:, 0]
            rows = got[heads, toks]
            hit = listed & (heads == 0)
            assert torch.isfinite(rows[~hit]).all() and not torch.isfinite(rows[hit]).any()
