"""Performance cases: the calls a user of this framework makes, over the sizes,
types and options they are made at.

Four kinds of call:

* ``layer``   -- ``AdaptiveSparseAttention.forward``, the attention layer, in its
  shortlist form (local window + strided anchors + prototype tokens) and its
  token-sparse causal form, launched eagerly or replayed from its HIP graph;
* ``mha``     -- ``CausalASPAMultiheadAttention``, the ``nn.MultiheadAttention``
  drop-in at its default settings;
* ``op``      -- ``aspa_sparse_attention`` on (B*H, T, D) tensors: with
  shortlist candidates from ``build_packed_shortlist_candidates``, implicitly
  causal, or with an additive (T, T) mask;
* ``chunked`` -- ``ChunkedShortlistRunner.run``, the long-context pipeline.

Inputs are N(0, 1) with 1% of the positions scaled by 4 (salient tokens);
weights are Xavier-normal.  Everything is made from the seed on the GPU.
"""
from __future__ import annotations

import heapq
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "proteus-flux-attention_amd"))

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
ESIZE = {"bf16": 2, "f16": 2, "f32": 4, "int8": 1}
DEVICE = "cuda"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _layer(name, **kw):
    case = dict(kind="layer", form="shortlist", dtype="bf16", B=1, T=4096, C=512, H=8, gates=8, L=2048, window=512,
                stride=256, keep=1.0, int8=False, graph=False)
    case.update(kw)
    return dict(case, name=name) if name else case


def _op(name, **kw):
    case = dict(kind="op", form="causal", dtype="bf16", B=1, H=8, T=2048, D=64, active=0.5, L=0, window=0, stride=0)
    case.update(kw)
    return dict(case, name=name) if name else case


def listed():
    return [
        # The smallest layer call: a short f32 sequence with a quarter of its
        # tokens kept, as in a unit test or an interactive prompt.  Launches
        # and latency decide.
        _layer("layer_sparse_1k_f32", form="sparse", dtype="f32", T=1024, C=256, keep=0.25),
        # Token-sparse causal attention over a small batch of 8K prompts.
        _layer("layer_sparse_8k_bf16", form="sparse", B=2, T=8192, keep=0.25),
        # The headline: a 64K-token shortlist forward replayed from its graph,
        # as a serving loop runs it.
        _layer("layer_64k_bf16_graph", T=65536, graph=True),
        # The longest single-pass sequence, launched eagerly.
        _layer("layer_512k_bf16", T=524288, L=4096),
        # Many narrow heads and gates (32 x 16 dims, 64 gates) at 64K.
        _layer("layer_64k_heads16_bf16", T=65536, H=32, gates=64),
        # The layer in torch's default type, at a ragged length: research code
        # that never casts its module.
        _layer("layer_10k_f32", dtype="f32", T=10007, L=1024, window=256, stride=128),
        # Per-head int8 q/k/v inside the layer, batched.
        _layer("layer_8k_int8_bf16", B=2, T=8192, L=1024, window=256, stride=128, int8=True),
        # The nn.MultiheadAttention drop-in at its defaults on short prompts of
        # a ragged length.
        dict(kind="mha", name="mha_500_bf16", dtype="bf16", B=4, T=500, C=512, H=8),
        # The operator with shortlist candidates built for the packed rows: an
        # integration that brings its own projections and router.
        _op("op_shortlist_8k_bf16", form="shortlist", T=8192, L=512, window=256, stride=128, active=0.25),
        # The operator's implicit causal branch on half-active heads, f16.
        _op("op_causal_4k_f16", B=2, T=4096, dtype="f16"),
        # The operator with an explicit additive mask at a ragged length, f32.
        _op("op_masked_1k_f32", form="masked", B=2, T=1500, dtype="f32", active=0.5),
        # A million tokens through the chunked pipeline, with the int8
        # all-query final pass.
        dict(kind="chunked", name="chunked_1m_bf16", T=1 << 20, C=512, H=8, chunk=65536, budget=512, buffer=8192),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "mha", "op", "op", "op", "chunked"])
    if kind == "layer":
        C, H, gates = rng.choice([(512, 8, 8), (512, 8, 8), (512, 8, 16), (256, 8, 8), (512, 32, 64), (512, 4, 8)])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32", "f16"])
        if rng.random() < 0.3:
            T = _log_int(rng, 256, 16384 if dtype == "bf16" else 4096)
            return _layer(None, form="sparse", dtype=dtype, B=rng.randint(1, 3), T=T, C=C, H=H, gates=gates,
                          keep=round(rng.uniform(0.1, 0.6), 2), graph=rng.random() < 0.3)
        int8 = dtype == "bf16" and rng.random() < 0.2
        T = _log_int(rng, 256, 131072 if dtype == "bf16" and not int8 else 16384)
        window = rng.choice([128, 256, 512])
        return _layer(None, dtype=dtype, B=rng.randint(1, 2), T=T, C=C, H=H, gates=gates,
                      L=rng.choice([2, 4]) * window, window=window, stride=rng.choice([64, 100, 128, 256]), int8=int8,
                      graph=not int8 and rng.random() < 0.3)
    if kind == "mha":
        C, H = rng.choice([(512, 8), (256, 8), (512, 4), (768, 12)])
        return dict(kind="mha", dtype=rng.choice(["bf16", "bf16", "f32", "f16"]), B=rng.randint(1, 8),
                    T=_log_int(rng, 80, 2048), C=C, H=H)
    if kind == "op":
        form = rng.choice(["shortlist", "causal", "masked"])
        window = rng.choice([64, 128, 256])
        return _op(None, form=form, dtype=rng.choice(["bf16", "bf16", "f32", "f16", "int8"]), B=rng.randint(1, 3),
                   H=rng.choice([4, 8, 16]), T=_log_int(rng, 128, 8192 if form == "shortlist" else 4096),
                   D=rng.choice([32, 64, 64, 128]), active=round(rng.uniform(0.1, 1.0), 2),
                   L=2 * window if form == "shortlist" else 0, window=window if form == "shortlist" else 0,
                   stride=rng.choice([64, 100, 128]) if form == "shortlist" else 0)
    chunk = rng.choice([8192, 16384, 32768])
    return dict(kind="chunked", T=_log_int(rng, 2 * chunk, 1 << 19), C=512, H=8, chunk=chunk,
                budget=rng.choice([256, 512]), buffer=rng.choice([1024, 2048, 4096]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _sequence(B, T, C, dtype, g):
    x = torch.randn(B, T, C, generator=g, device=DEVICE)
    salient = torch.rand(T, generator=g, device=DEVICE) < 0.01
    x[:, salient] *= 4.0
    return x.to(dtype)


def _xavier(rows, cols, dtype, g):
    return (torch.randn(rows, cols, generator=g, device=DEVICE) * math.sqrt(2.0 / (rows + cols))).to(dtype)


def _layer_config(case):
    """The module's options.  Two heads per token, prototype routing on."""
    T = case["T"]
    cfg = dict(n_layer=1, p_dropout=0.0, bias=False, attn_variant="aspa", attn_h_active=2, attn_h_active_min=2,
               attn_h_active_max=2, attn_router_top_p=0.0, attn_linear_head_k=2, attn_router_noise_std=0.0,
               attn_force_dense_threshold=None, attn_small_seq_dense=0, attn_proto_enable=True, vocab_size=0,
               n_ctx=T, n_head=case["H"], d_model=case["C"], attn_h_total=case["H"], attn_gates=case["gates"],
               attn_mode="linear", attn_quantize_int8=case["int8"])
    if case["form"] == "sparse":
        L, window, stride, policy = T, T, 0, "local"
        cfg.update(attn_token_sparse=True, attn_token_keep_ratio=case["keep"],
                   attn_linear_token_keep_schedule="fixed")
    else:
        L, window, stride, policy = case["L"], case["window"], case["stride"], "local+anchors+proto"
        cfg.update(attn_token_sparse=False, attn_linear_L_schedule="fixed")
    cfg.update(attn_linear_L=L, attn_linear_L_base=L, attn_linear_L_min=L, attn_linear_L_max=L,
               attn_linear_window=window, attn_linear_anchor_stride=stride, attn_linear_policy=policy)
    return cfg


def _layer_inputs(case, seed):
    g, dt, C, G = _gen(seed), DTYPES[case["dtype"]], case["C"], case["gates"]
    return dict(x=_sequence(case["B"], case["T"], C, dt, g), router=_xavier(G, C, dt, g),
                protos=_xavier(G, C, dt, g), qkv=_xavier(3 * C, C, dt, g), proj=_xavier(C, C, dt, g))


def _mha_inputs(case, seed):
    g, dt, C = _gen(seed), DTYPES[case["dtype"]], case["C"]
    return dict(x=_sequence(case["B"], case["T"], C, dt, g), qkv=_xavier(3 * C, C, dt, g),
                qkv_bias=_xavier(1, 3 * C, dt, g)[0], proj=_xavier(C, C, dt, g), proj_bias=_xavier(1, C, dt, g)[0],
                router=_xavier(2 * case["H"], C, dt, g), protos=_xavier(2 * case["H"], C, dt, g))


def _op_inputs(case, seed):
    g, BH, T, D = _gen(seed), case["B"] * case["H"], case["T"], case["D"]
    s = {}
    for n in "qkv":
        t = torch.randn(BH, T, D, generator=g, device=DEVICE)
        if case["dtype"] == "int8":
            scale = t.abs().amax(dim=(1, 2)) / 127.0
            s[n + "_scale"] = scale
            t = (t / scale.view(-1, 1, 1)).round().clamp(-127, 127).to(torch.int8)
        else:
            t = t.to(DTYPES[case["dtype"]])
        s[n] = t
    # the same number of active rows in every head, the first token among them
    order = torch.rand(BH, T, generator=g, device=DEVICE)
    order[:, 0] = -1.0
    best = order.argsort(dim=1)[:, :max(1, round(case["active"] * T))]
    s["mask"] = torch.zeros(BH, T, dtype=torch.bool, device=DEVICE).scatter_(1, best, True)
    if case["form"] == "masked":
        # a banded causal bias: a distance penalty, and -inf ahead of the row
        t = torch.arange(T, device=DEVICE)
        dist = (t[:, None] - t[None, :]).to(torch.float32)
        bias = torch.where(dist >= 0, -0.01 * dist, torch.full_like(dist, float("-inf")))
        s["bias"] = bias.to(DTYPES.get(case["dtype"], torch.float32))
    if case["form"] == "shortlist":
        s["scores"] = torch.rand(case["B"], T, generator=g, device=DEVICE)
        heads, rows = s["mask"].nonzero(as_tuple=True)
        s["rows"], s["row_batch"] = rows, heads // case["H"]
    return s


def _set(param, value):
    with torch.no_grad():
        param.copy_(value)


def prepare(case, seed):
    if case["kind"] == "layer":
        from proteus_attention.models.aspa import AdaptiveSparseAttention, ModelConfig

        w, dt = _layer_inputs(case, seed), DTYPES[case["dtype"]]
        m = AdaptiveSparseAttention(ModelConfig(**_layer_config(case))).to(device=DEVICE, dtype=dt).eval()
        for p, n in ((m.head_router.linear.weight, "router"), (m.routing_prototypes, "protos"),
                     (m.qkv.weight, "qkv"), (m.proj.weight, "proj")):
            _set(p, w[n])
        x = w["x"]
        if case["graph"]:
            # a serving loop's set-up: the graph captured once, the input in
            # the graph's own buffer (where the forward can be captured)
            m.enable_hip_graph(True, static_output=True)
            with torch.no_grad():
                try:
                    x = m.hip_graph_input(x)
                except RuntimeError:
                    m.enable_hip_graph(False)
        return dict(case=case, m=m, x=x)
    if case["kind"] == "mha":
        from proteus_attention import CausalASPAMultiheadAttention

        w, dt = _mha_inputs(case, seed), DTYPES[case["dtype"]]
        m = CausalASPAMultiheadAttention(case["C"], case["H"]).to(device=DEVICE, dtype=dt).eval()
        a = m.attention
        for p, n in ((a.head_router.linear.weight, "router"), (a.routing_prototypes, "protos"), (a.qkv.weight, "qkv"),
                     (a.qkv.bias, "qkv_bias"), (a.proj.weight, "proj"), (a.proj.bias, "proj_bias")):
            _set(p, w[n])
        return dict(case=case, m=m, x=w["x"])
    if case["kind"] == "op":
        return dict(_op_inputs(case, seed), case=case)
    from proteus_attention.tools.chunked_shortlist import ChunkedShortlistConfig

    cfg = ChunkedShortlistConfig(seq_len=case["T"], d_model=case["C"], chunk_len=case["chunk"],
                                 buffer_tokens=case["buffer"], per_chunk_budget=case["budget"],
                                 device=torch.device("cuda:0"), heads=case["H"], nucleus_top_p=1.0,
                                 final_mode="all_queries")
    return dict(case=case, cfg=cfg, x=_sequence(1, case["T"], case["C"], torch.bfloat16, _gen(seed)))


def run(state):
    case = state["case"]
    if case["kind"] == "layer":
        m = state["m"]
        with torch.no_grad():
            y = m(state["x"])
        return dict(y=y, protos=m.routing_prototypes, usage=m.routing_usage_ema, confidence=m.routing_confidence)
    if case["kind"] == "mha":
        with torch.no_grad():
            return state["m"](state["x"], need_weights=False, is_causal=True)[0]
    if case["kind"] == "op":
        from proteus_attention.kernels.sparse_attn import aspa_sparse_attention, build_packed_shortlist_candidates

        kw = dict(active_mask=state["mask"])
        if case["dtype"] == "int8":
            kw.update(q_scale=state["q_scale"], k_scale=state["k_scale"], v_scale=state["v_scale"])
        if case["form"] == "masked":
            kw.update(causal_mask=state["bias"])
        if case["form"] != "shortlist":
            return aspa_sparse_attention(state["q"], state["k"], state["v"], **kw)
        cand, lens = build_packed_shortlist_candidates(
            state["rows"], state["row_batch"], case["T"], max_candidates=case["L"], linear_window=case["window"],
            anchor_stride=case["stride"], use_local=True, use_anchors=True, proto_scores=state["scores"],
            **_op_caps(case))
        out = aspa_sparse_attention(state["q"], state["k"], state["v"], shortlist_candidates=cand,
                                    shortlist_lengths=lens, **kw)
        return dict(out=out, cand=cand, lens=lens)
    from proteus_attention.tools.chunked_shortlist import ChunkedShortlistRunner

    torch.manual_seed(7)  # the runner draws its models' weights
    res = ChunkedShortlistRunner(state["cfg"]).run(state["x"])
    return dict(keep=res.keep_indices, scores=res.keep_scores, out=res.final_output)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _op_caps(case):
    L = case["L"]
    return dict(local_cap=case["window"], anchor_cap=L // 4, proto_cap=L // 4)


def _layer_caps(case):
    """(window, anchor slots, prototype tokens) of the shortlist form: L split
    60/30/10 over the three pieces, the remainder handed out in that order."""
    L = case["L"]
    caps = [int(round(L * f)) for f in (0.6, 0.3, 1.0 - 0.6 - 0.3)]
    if sum(caps) > L:
        caps = [int(math.floor(c * (L / sum(caps)))) for c in caps]
    left = L - sum(caps)
    for i in range(3):
        if left > 0:
            caps[i] += 1
            left -= 1
    caps[0] += max(0, left)
    return min(caps[0], case["window"], L), min(caps[1], L, case["T"]), min(L, caps[2], case["T"])


def _mean_keys(T, w, stride, slots, K):
    """Mean candidates of a row: window, anchors below it, prototypes."""
    step = max(1, T // 4096)
    tot = n = 0
    for t in range(0, T, step):
        win = min(t + 1, w)
        anchors = max(0, min(slots, t // stride) - (win - 1) // stride) if stride else 0
        tot += win + anchors + min(K, max(0, t + 1 - win))
        n += 1
    return tot / n


def work(case):
    if case["kind"] == "chunked":
        T, C, H, S = case["T"], case["C"], case["H"], min(case["buffer"], case["budget"] * -(-case["T"] // case["chunk"]))
        # chunk router + query projection, causal attention of every query to
        # the shortlist (half of the pairs visible), output projection
        flops = 4.0 * T * C * C + 4.0 * T * C * 2 * H + 4.0 * C * T * S / 2
        return dict(bytes=2.0 * T * C * 2, flops=flops)
    e = ESIZE[case["dtype"]]
    if case["kind"] == "mha":
        n, T, C = case["B"] * case["T"], case["T"], case["C"]
        D, heads = C // case["H"], _mha_heads(case)
        return dict(bytes=e * (2.0 * n * C + 4 * C * C),
                    flops=8.0 * n * C * C + 4.0 * heads * D * n * min((T + 1) / 2, 512))
    if case["kind"] == "layer":
        B, T, C, H, G = case["B"], case["T"], case["C"], case["H"], case["gates"]
        if case["form"] == "sparse":
            rows, keys = 2 * B * T * case["keep"], (T + 1) / 2
        else:
            w, slots, K = _layer_caps(case)
            rows, keys = 2 * B * T, _mean_keys(T, w, case["stride"], slots, K)
        # projections of every token, router and prototype statistics, attention
        flops = 8.0 * B * T * C * C + 6.0 * B * T * C * G + 4.0 * rows * keys * (C // H)
        return dict(bytes=e * (2.0 * B * T * C + 4 * C * C + 3 * G * C), flops=flops)
    BH, T, D = case["B"] * case["H"], case["T"], case["D"]
    rows, out_e = BH * T * case["active"], 4 if case["dtype"] == "int8" else e
    nbytes = BH * T * D * (3.0 * e + out_e) + BH * T
    if case["form"] == "shortlist":
        c = _op_caps(case)
        keys = _mean_keys(T, c["local_cap"], case["stride"], c["anchor_cap"], c["proto_cap"])
        nbytes += rows * (case["L"] * 8 + 8)  # the candidate lists it returns
    elif case["form"] == "masked":
        keys = (T + 1) / 2
        nbytes += T * T * out_e
    else:
        keys = (T + 1) / 2
    return dict(bytes=nbytes, flops=4.0 * rows * keys * D)


def tolerance(case):
    if case["kind"] == "chunked":
        return {"rel": 1e-2, "max": 0.9, "differ": 1e-3}
    if case["kind"] == "op":
        # int8 inputs are exact: products and sums are f32
        rel = {"f32": 2e-6, "int8": 2e-6, "f16": 1e-3, "bf16": 8e-3}[case["dtype"]]
        return {"rel": rel, "max": 40 * rel}
    # a token whose two best heads nearly tie may take the other head, and a
    # token whose importance nearly ties may be kept or not
    return {"f32": {"rel": 1e-5, "max": 1e-3}, "f16": {"rel": 4e-3, "max": 0.9},
            "bf16": {"rel": 1e-2, "max": 0.9}}[case["dtype"]]


# ---------------------------------------------------------------------------
# the results in 64 bits
# ---------------------------------------------------------------------------

def _evict(scores, K):
    """Per position p, the first token at which p is no longer among the K best
    of the positions up to that token (equal scores: the lower position)."""
    vals = scores.tolist()
    out, heap, never = [0] * len(vals), [], 1 << 40
    for t, v in enumerate(vals):
        heapq.heappush(heap, (v, -t))
        out[t] = never
        if len(heap) > K:
            out[-heapq.heappop(heap)[1]] = t
    return torch.tensor(out, device=DEVICE)


def _allowed(t, p, evict, w, stride, slots):
    """Which of the keys p are candidates of the tokens t (anchors included)."""
    d = t[:, None] - p[None, :]
    ok = (d >= 0) & (d < max(w, 1))
    if stride and slots:
        ok |= (d > 0) & (d % stride == 0) & (d <= stride * slots)
        ok |= (p[None, :] == 0) & (stride * slots >= t[:, None])  # anchors below 0 are 0
    if evict is not None:
        ok |= (d >= 0) & (t[:, None] < evict[p][None, :])
    return ok


def _attend(q, k, v, active, allowed):
    """q, k, v (H, T, D) f64, active (H, T): softmax attention of the active rows
    over allowed(t) keys, 0 elsewhere."""
    H, T, D = q.shape
    out = torch.zeros_like(q)
    keys = torch.arange(T, device=DEVICE)
    for t0 in range(0, T, 256):
        t = keys[t0:t0 + 256]
        p, bias = allowed(t)
        s = q[:, t0:t0 + 256] @ k[:, p].transpose(1, 2).contiguous() / math.sqrt(D) + bias
        o = torch.softmax(s, dim=-1) @ v[:, p]
        out[:, t0:t0 + 256] = torch.where(active[:, t0:t0 + 256, None], o, 0.0)
    return out


def _attend_shortlist(q, k, v, active, evict, w, stride, slots):
    """The same with the window and the prototype tokens of 256 tokens as one
    key list and each row's anchors gathered."""
    H, T, D = q.shape
    out, every = torch.zeros_like(q), torch.arange(T, device=DEVICE)
    for t0 in range(0, T, 256):
        t = every[t0:t0 + 256]
        t1 = int(t[-1])
        lo = max(0, t0 - w + 1)
        p = every[lo:t1 + 1]
        if evict is not None:
            old = every[:lo]
            p = torch.cat([old[evict[:lo] > t0], p])
        d = t[:, None] - p[None, :]
        in_window = (d >= 0) & (d < max(w, 1))
        ok = in_window.clone()
        if evict is not None:
            ok |= (d >= 0) & (t[:, None] < evict[p][None, :])
        h, r = active[:, t0:t0 + 256].nonzero(as_tuple=True)
        if not h.numel():
            continue
        qs = q[h, t0 + r]
        s = (q[:, t0:t0 + 256] @ k[:, p].transpose(1, 2).contiguous())[h, r]
        n = min(slots, t1 // stride + 1) if stride else 0
        if n > 0:
            tr = t[r]
            a = (tr[:, None] - stride * torch.arange(1, n + 1, device=DEVICE)[None, :])
            reach = (stride * slots >= tr)[:, None] & (tr[:, None] > 0)
            first = (a <= 0) & (a > -stride) & reach          # the one anchor that stands for 0
            a_ok = ((a > 0) | first) & (a.clamp(min=0) < (tr - max(w, 1) + 1)[:, None])
            a = a.clamp(min=0)
            # a prototype that is an anchor too counts once
            dup = (d > 0) & (d % stride == 0) & (d <= stride * slots)
            dup |= (p[None, :] == 0) & (stride * slots >= t[:, None])
            ok &= in_window | ~dup
            sa = torch.bmm(k[h[:, None], a], qs[:, :, None])[:, :, 0]
            s = torch.cat([s, sa], dim=1)
            ok_r = torch.cat([ok[r], a_ok], dim=1)
        else:
            ok_r = ok[r]
        pr = torch.softmax((s / math.sqrt(D)).masked_fill(~ok_r, float("-inf")), dim=-1)
        dense = torch.zeros(H, t.numel(), p.numel(), dtype=q.dtype, device=DEVICE)
        dense[h, r] = pr[:, :p.numel()]
        o = (dense @ v[:, p])[h, r]
        if n > 0:
            o = o + torch.bmm(pr[:, None, p.numel():], v[h[:, None], a])[:, 0]
        out[h, t0 + r] = o
    return out


def _rope(t, base_dtype):
    """(B, T, H, D) rotated; the angle tables are the model's, made in its type."""
    T, D = t.shape[1], t.shape[3]
    inv = (1.0 / (10000.0 ** (torch.arange(0, D, 2, dtype=torch.float32) / D))).to(DEVICE, base_dtype)
    ang = torch.outer(torch.arange(T, device=DEVICE, dtype=base_dtype), inv)
    c = ang.cos().repeat_interleave(2, dim=-1).double().view(1, T, 1, D)
    s = ang.sin().repeat_interleave(2, dim=-1).double().view(1, T, 1, D)
    rot = torch.stack((-t[..., 1::2], t[..., ::2]), dim=-1).reshape_as(t)
    return t * c + rot * s


def _route(case, w, gates):
    """Gate probabilities, per-head sums of them, prototype similarity and
    token importance.  Gate probabilities are held in the model's type and
    blended with the prototype prior (temperature 0.2, threshold 0.25, blend
    0.6, no confidence yet)."""
    dt, H = DTYPES[case["dtype"]], case["H"]

    def rd(t):  # a value the model holds in its own type
        return t.to(dt).double()

    x, protos = w["x"].double(), w["protos"].double()
    gate = rd(torch.softmax(rd(x @ w["router"].double().t()), dim=-1))
    unit = x / x.norm(dim=-1, keepdim=True).clamp_min(1e-6)
    sims = unit @ (protos / protos.norm(dim=-1, keepdim=True).clamp_min(1e-6)).t()
    sim = sims.amax(dim=-1)
    prior = torch.softmax(sims / 0.2, dim=-1) * rd(torch.tensor(1e-6, device=DEVICE))
    prior = prior / prior.sum(-1, keepdim=True).clamp_min(1e-6)
    blend = ((sim - 0.25) / 0.75).clamp(0.0, 1.0)
    bl = 0.6 * blend[..., None]
    gate = (gate * (1.0 - bl) + prior * bl).clamp_min(0.0)
    gate = gate / gate.sum(-1, keepdim=True).clamp_min(1e-6)
    importance = (gate.amax(-1) * (1.0 - blend) + sim * blend).float()
    to_head = (torch.arange(gates, device=DEVICE) * H) // gates
    head = torch.zeros(*sim.shape, H, dtype=torch.float64, device=DEVICE).index_add_(2, to_head, gate).float()
    return gate, head, sim, importance


def _top_heads(head, k):
    top = head.sort(dim=-1, descending=True, stable=True).indices[..., :k]
    return torch.zeros(head.shape, dtype=torch.bool, device=DEVICE).scatter_(2, top, True)


def _qkv(case, w, bias=0.0):
    """Rotated q, k and v, (B, H, T, D)."""
    B, T, C, H, dt = case["B"], case["T"], case["C"], case["H"], DTYPES[case["dtype"]]
    qkv = (w["x"].double().view(-1, C) @ w["qkv"].double().t() + bias).view(B, T, 3, H, C // H)
    q, k, v = _rope(qkv[:, :, 0], dt), _rope(qkv[:, :, 1], dt), qkv[:, :, 2]
    return [t.permute(0, 2, 1, 3).contiguous() for t in (q, k, v)]


def _exact_layer(case, seed):
    w = _layer_inputs(case, seed)
    B, T, C, H, G = case["B"], case["T"], case["C"], case["H"], case["gates"]
    gate, head, sim, importance = _route(case, w, G)
    active = _top_heads(head, 2)
    if case["form"] == "sparse":
        keep = int(torch.tensor(case["keep"] * T, dtype=torch.float32).round())
        kept = importance.sort(dim=-1, descending=True, stable=True).indices[:, :max(1, keep)]
        tok = torch.zeros(B, T, dtype=torch.bool, device=DEVICE).scatter_(1, kept, True)
        tok[:, 0] = True
        active &= tok[..., None]
    q, k, v = _qkv(case, w)
    if case["int8"]:
        for t in (q, k, v):
            s = (t.abs().amax(dim=(2, 3), keepdim=True) / 127.0).clamp_min(1e-6)
            t.copy_((t / s).round().clamp(-127, 127) * s)
    attn = torch.empty_like(q)
    for b in range(B):
        win, slots, K = (T, 0, 0) if case["form"] == "sparse" else _layer_caps(case)
        evict = _evict(sim[b].float(), K) if K else None
        stride = case["stride"] if slots else 0
        attn[b] = _attend_shortlist(q[b], k[b], v[b], active[b].t(), evict, win, stride, slots)
    y = attn.permute(0, 2, 1, 3).reshape(B, T, C) @ w["proj"].double().t()
    # prototype statistics of the pass (decay 0.97)
    gf, xf = gate.view(-1, G), w["x"].double().view(-1, C)
    cnt = gf.sum(0)
    mean = (gf.t() @ xf) / cnt[:, None]
    return dict(y=y, protos=w["protos"].double() * 0.97 + mean * 0.03, usage=cnt * 0.03,
                confidence=torch.full_like(cnt, 0.03))


def _mha_low(case):
    return max(64, case["C"] // case["H"])


def _mha_heads(case, head=None):
    """Heads per token of the drop-in: all of them up to `low` tokens, two from
    four times that, a fourth-root curve between; capped by the nucleus (0.9 of
    the mean head probability) and drawn towards two with the length."""
    T, H, low = case["T"], case["H"], _mha_low(case)
    ratio = min(1.0, max(0.0, (T - low) / (3.0 * low))) ** 0.25
    k = max(2, min(H, int(math.floor(H - ratio * (H - 2) + 1e-6))))
    if k > 2 and head is not None:
        mean = head.mean(dim=(0, 1)).sort(descending=True).values.cumsum(0).cpu()
        k = max(2, min(k, int((mean < float(mean[-1]) * 0.9).sum()) + 1))
    alpha = max(0.0, (T - low) / (20000.0 - low))
    return max(1, min(k, int(round((1.0 - alpha) * k + alpha * 2))))


def _mha_caps(case):
    """(window, anchor slots) of the drop-in: its dense sizes at short lengths
    blended into its shortlist sizes (L 512, window 512) with the length."""
    T, low = case["T"], _mha_low(case)
    a = max(0.0, (T - low) / (20000.0 - low))
    cap = max(64, min(512, T, max(64, 512 + T // 32)))
    L = max(64, min(512, int(a * 512 + (1.0 - a) * cap)))
    window = max(1, min(L, int(a * 512 + (1.0 - a) * max(1, min(T, max(512, T // 8))))))
    lw, aw = (1.0 - a) * 0.85 + a * (2.0 / 3.0), (1.0 - a) * 0.10 + a / 3.0
    lw = lw / (lw + aw)
    caps = [int(round(L * lw)), int(round(L * (1.0 - lw)))]
    if sum(caps) > L:
        caps = [int(math.floor(c * (L / sum(caps)))) for c in caps]
    for i in range(2):
        if sum(caps) < L:
            caps[i] += 1
    caps[0] += max(0, L - sum(caps))
    return min(caps[0], window), min(caps[1], L, T)


def _exact_mha(case, seed):
    w = _mha_inputs(case, seed)
    B, T, C, H = case["B"], case["T"], case["C"], case["H"]
    _, head, _, _ = _route(case, w, 2 * H)
    active = _top_heads(head, _mha_heads(case, head))
    dense = T <= _mha_low(case) or float(active.sum(1).max()) / T >= 0.6  # then every head, causally
    q, k, v = _qkv(case, w, w["qkv_bias"].double())
    win, slots = (T, 0) if dense else _mha_caps(case)
    attn = torch.empty_like(q)
    for b in range(B):
        act = torch.ones_like(active[b]) if dense else active[b]
        attn[b] = _attend_shortlist(q[b], k[b], v[b], act.t(), None, win, 256 if slots else 0, slots)
    o = attn.permute(0, 2, 1, 3).reshape(B, T, C)
    return o @ w["proj"].double().t() + w["proj_bias"].double()


def _causal_bias(t):
    p = torch.arange(int(t[-1]) + 1, device=DEVICE)
    return p, torch.where(p[None, :] <= t[:, None], 0.0, float("-inf")).double()


def _exact_op(case, seed):
    s, T, H = _op_inputs(case, seed), case["T"], case["H"]
    q, k, v = (s[n].double() * (s[n + "_scale"].double().view(-1, 1, 1) if case["dtype"] == "int8" else 1.0)
               for n in "qkv")
    if case["form"] == "causal":
        return _attend(q, k, v, s["mask"], _causal_bias)
    every = torch.arange(T, device=DEVICE)
    if case["form"] == "masked":
        return _attend(q, k, v, s["mask"], lambda t: (every, s["bias"][t].double()))
    c, out = _op_caps(case), torch.empty_like(q)
    for b in range(case["B"]):
        evict = _evict(s["scores"][b], min(c["proto_cap"], T))

        def allowed(t):
            ok = _allowed(t, every, evict, c["local_cap"], case["stride"], c["anchor_cap"])
            return every, torch.where(ok, 0.0, float("-inf")).double()

        h = slice(b * H, (b + 1) * H)
        out[h] = _attend(q[h], k[h], v[h], s["mask"][h], allowed)
    return dict(out=out, cand=None, lens=None)


def exact(case, seed):
    if case["kind"] == "layer":
        return _exact_layer(case, seed)
    if case["kind"] == "mha":
        return _exact_mha(case, seed)
    if case["kind"] == "op":
        return _exact_op(case, seed)
    return None  # the runner draws its own models' weights
