"""The timed workloads of the DSA hot path.

Each case is one call, or one training step, through the package's public entry
points, at the shapes the benchmark configurations and tests use (cfg1 to cfg5
of ``cppmega_amd.synthetic`` and ``bench.py``) or at odd sizes of the same
ranges.  A case is a plain dict; ``kind`` names the path:

  attn_train    SparseMLA (or SparseMLA_FP8) autograd step: forward, then the
                gradients of q and kv for an upstream gradient (training)
  attn_fwd      sparse_mla_fwd_interface of S query tokens, the last of S_kv
                (S = S_kv / n: a prefill chunk; S = 1: a decode step)
  index_select  fused_qk_topk_naive with Megatron's causal float mask, without
                autograd: the scores and the selected columns
  index_topk    indexer_topk: causal prefill, or one query token per sequence
                against its cached keys
  index_train   FusedDSAIndexerLoss step: top-k, KL loss, and the gradients of
                the indexer's q, weights and k
  layer         one DSA layer step: indexer_topk, then SparseMLA forward and
                backward on the columns it chose
"""
from __future__ import annotations

import math

import torch

import cppmega_amd as ca
from cppmega_amd import sparse_mla_ops as ops

# (d_qk, d_v): 64 latent + 64 rope (NAM56R), the 192/128 and 128/128 head dims
# of un-absorbed MLA, and the 512 latent + 64 rope row of absorbed MLA.
_NARROW = ((128, 64), (192, 128), (128, 128))
_WIDE = (576, 512)


def _attn(name, kind, B, S, S_kv, H, d_qk, d_v, topk, dtype="bf16"):
    return dict(name=name, kind=kind, B=B, S=S, S_kv=S_kv, H=H, d_qk=d_qk, d_v=d_v, topk=topk, dtype=dtype)


def _index(name, kind, B, S, S_kv, h, d, topk, dtype="bf16", np=0, hn=0):
    return dict(name=name, kind=kind, B=B, S=S, S_kv=S_kv, h=h, d=d, topk=topk, dtype=dtype, np=np, hn=hn)


def listed():
    return [
        # the smallest training call (cfg1's shape): a unit test, a debug run, the last short micro-batch
        _attn("attn_train_small", "attn_train", 1, 512, 512, 16, 128, 64, 64),
        # the production attention layer in training (cfg2, NAM56R)
        _attn("attn_train", "attn_train", 2, 4096, 4096, 32, 128, 64, 256),
        # a packed batch with no round size: sequence, heads and top-k that fill no tile
        _attn("attn_train_ragged", "attn_train", 3, 1531, 1531, 28, 192, 128, 200),
        # the production layer with tensorwise e4m3 (cfg4: 1% outliers x20), quantised in the step
        _attn("attn_train_fp8", "attn_train", 2, 4096, 4096, 32, 128, 64, 256, "fp8"),
        # training the long-context model: 4096 tokens at cfg5's heads, row and top-k
        _attn("attn_train_wide", "attn_train", 1, 4096, 4096, 128, 576, 512, 2048),
        # long-context evaluation: the last 4096-token prefill chunk of a 16384-token prompt (cfg5)
        _attn("attn_prefill_wide", "attn_fwd", 1, 4096, 16384, 128, 576, 512, 2048),
        # generation: one new token for each of 16 sequences against 16384 cached rows (cfg5)
        _attn("attn_decode_wide", "attn_fwd", 16, 1, 16384, 128, 576, 512, 2048),
        # what DSAttention calls for its indices (cfg3), causal float mask
        _index("index_select", "index_select", 2, 4096, 4096, 16, 64, 256),
        # the long-context indexer (cfg5): e4m3, top-2048 of a 16384-token prompt
        _index("index_topk_long", "index_topk", 1, 16384, 16384, 64, 128, 2048, "fp8"),
        # generation: the indexer of 16 new tokens against 16384 cached keys each
        _index("index_topk_decode", "index_topk", 16, 1, 16384, 64, 128, 2048, "fp8"),
        # training the indexer against the attention it stands for (NAM56R: 32 heads of 128)
        _index("index_train", "index_train", 2, 4096, 4096, 16, 64, 256, np=32, hn=128),
        # one whole DSA layer step (cfg3's indexer feeding cfg2's attention)
        dict(name="layer_step", kind="layer", B=2, S=4096, S_kv=4096, H=32, d_qk=128, d_v=64, topk=256, dtype="bf16",
             h=16, d=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(("attn_train", "attn_train", "attn_train_wide", "attn_fwd", "attn_fwd", "index_select",
                       "index_topk", "index_train", "layer"))
    if kind == "attn_train":
        d_qk, d_v = rng.choice(_NARROW)
        S = _log(rng, 200, 4096)
        c = _attn("", kind, rng.randint(1, 3), S, S, rng.choice((8, 16, 28, 32, 40, 64)), d_qk, d_v,
                  _log(rng, 33, 512), rng.choice(("bf16", "bf16", "fp8")))
    elif kind == "attn_train_wide":
        S = _log(rng, 128, 4096)
        c = _attn("", "attn_train", 1, S, S, rng.choice((16, 32, 64, 96, 128)), *_WIDE, _log(rng, 64, 2048))
    elif kind == "attn_fwd":
        S = rng.choice((1, 1, _log(rng, 2, 4096)))
        S_kv = max(S, _log(rng, 512, 16384))
        d_qk, d_v = rng.choice((*_NARROW, _WIDE, _WIDE))
        c = _attn("", kind, rng.randint(1, 32) if S == 1 else rng.randint(1, 2), S, S_kv,
                  rng.choice((16, 32, 64, 128)), d_qk, d_v, _log(rng, 64, 2048))
    elif kind == "index_select":
        S = _log(rng, 200, 4096)
        c = _index("", kind, rng.randint(1, 3), S, S, rng.choice((16, 32, 64)), rng.choice((64, 128)),
                   min(S, _log(rng, 33, 1024)))
    elif kind == "index_topk":
        S_kv = _log(rng, 512, 16384)
        one = rng.random() < 0.4
        h, d = rng.choice(((16, 64), (32, 64), (64, 128)))
        c = _index("", kind, rng.randint(1, 32) if one else rng.randint(1, 2), 1 if one else S_kv, S_kv, h, d,
                   _log(rng, 64, 2048), rng.choice(("bf16", "fp8")))
    elif kind == "index_train":
        S = _log(rng, 200, 4096)
        c = _index("", kind, rng.randint(1, 2), S, S, rng.choice((16, 32, 64)), rng.choice((64, 128)),
                   min(S, _log(rng, 33, 1024)), np=rng.choice((16, 28, 32)), hn=rng.choice((64, 128, 192)))
    else:
        S = _log(rng, 200, 4096)
        d_qk, d_v = rng.choice(_NARROW)
        c = dict(name="", kind="layer", B=rng.randint(1, 2), S=S, S_kv=S, H=rng.choice((16, 32, 64)), d_qk=d_qk,
                 d_v=d_v, topk=_log(rng, 33, 512), dtype="bf16", h=rng.choice((16, 32)), d=64)
    del c["name"]
    return c


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        c = _draw_once(rng)
        if work(c)["flops"] <= most:
            return c


# ---------------------------------------------------------------- inputs


def _causal_indices(g, B, S, S_kv, topk):
    """int32 [B, S, 1, topk]: per query token (position S_kv - S + t) up to topk distinct
    uniform picks of the positions before and at it, ascending, -1 padded."""
    out = torch.full((B, S, 1, topk), -1, dtype=torch.int32, device="cuda")
    cols = torch.arange(S_kv, device="cuda")
    k = min(topk, S_kv)
    step = max(1, (1 << 25) // S_kv)
    for b in range(B):
        for t0 in range(0, S, step):
            t1 = min(S, t0 + step)
            pos = torch.arange(S_kv - S + t0, S_kv - S + t1, device="cuda")[:, None]
            keys = torch.rand((t1 - t0, S_kv), generator=g, device="cuda").masked_fill_(cols[None] > pos, -1.0)
            val, ix = keys.topk(k, dim=-1)
            ix = ix.masked_fill_(val < 0, S_kv).sort(dim=-1).values
            out[b, t0:t1, 0, :k] = ix.masked_fill_(ix == S_kv, -1).to(torch.int32)
    return out


def _normal(g, shape, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(torch.bfloat16)


def _outliers(g, shape):
    x = torch.randn(shape, generator=g, device="cuda")
    return torch.where(torch.rand(shape, generator=g, device="cuda") < 0.01, x * 20, x).to(torch.bfloat16)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    c, kind = case, case["kind"]
    B, S, S_kv = c["B"], c["S"], c["S_kv"]
    s = dict(case=c)
    if kind in ("attn_train", "attn_fwd", "layer"):
        fp8 = c["dtype"] == "fp8"
        make = (lambda shape: _outliers(g, shape)) if fp8 else (lambda shape: _normal(g, shape, 0.5))
        s["q"], s["kv"] = make((B, S, c["H"], c["d_qk"])), make((B, S_kv, 1, c["d_qk"]))
        s["scale"] = c["d_qk"] ** -0.5
        if kind != "layer":
            s["indices"] = _causal_indices(g, B, S, S_kv, c["topk"])
        if kind != "attn_fwd":
            s["do"] = _normal(g, (B, S, c["H"], c["d_v"]))
            s["q"].requires_grad_()
            s["kv"].requires_grad_()
    if kind in ("index_select", "index_topk", "index_train", "layer"):
        h, d = c["h"], c["d"]
        iq, ik = _normal(g, (S, B, h, d)), _normal(g, (S_kv, B, d))
        s["iw"] = torch.randn((S, B, h), generator=g, device="cuda") / h ** 0.5
        if c["dtype"] == "fp8":
            iq, s["iq_scale"] = ops.tensorwise_quantize(iq)
            ik, s["ik_scale"] = ops.tensorwise_quantize(ik)
        s["iq"], s["ik"] = iq, ik
    if kind in ("index_select", "index_train"):
        s["mask"] = torch.full((S, S_kv), float("-inf"), device="cuda").triu_(1)
    if kind == "index_train":
        s["query"], s["key"] = (_normal(g, (n, B, c["np"], c["hn"])) for n in (S, S_kv))
        for n in ("iq", "iw", "ik"):
            s[n].requires_grad_()
    return s


# ---------------------------------------------------------------- one pass


def _attention_step(s, indices):
    c = s["case"]
    fn = ops.SparseMLA_FP8 if c["dtype"] == "fp8" else ops.SparseMLA
    out, lse = fn.apply(s["q"], s["kv"], indices, s["scale"], c["d_v"])
    dq, dkv = torch.autograd.grad(out, (s["q"], s["kv"]), s["do"])
    return dict(out=out.detach(), lse=lse.detach(), dq=dq, dkv=dkv)


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "attn_train":
        return _attention_step(s, s["indices"])
    if kind == "attn_fwd":
        out, lse = ops.sparse_mla_fwd_interface(s["q"], s["kv"], s["indices"], sm_scale=s["scale"], d_v=c["d_v"])
        return dict(out=out, lse=lse)
    if kind == "index_select":
        with torch.no_grad():
            scores, idx = ca.fused_qk_topk_naive(s["iq"], s["ik"], s["iw"], c["topk"], mask=s["mask"])
        return dict(scores=scores, idx=idx)
    if kind == "index_topk":
        idx = ca.indexer_topk(s["iq"], s["ik"], s["iw"], c["topk"], causal=c["S"] == c["S_kv"],
                              q_scale=s.get("iq_scale"), k_scale=s.get("ik_scale"))
        return dict(idx=idx)
    if kind == "index_train":
        idx, loss = ca.FusedDSAIndexerLoss.apply(s["iq"], s["iw"], s["ik"], s["query"], s["key"], c["hn"] ** -0.5,
                                                 c["topk"], 1.0, s["mask"], True, None)
        dq, dw, dk = torch.autograd.grad(loss, (s["iq"], s["iw"], s["ik"]))
        return dict(idx=idx, loss=loss.detach(), dq=dq, dw=dw, dk=dk)
    idx = ca.indexer_topk(s["iq"], s["ik"], s["iw"], c["topk"])
    return dict(idx=idx, **_attention_step(s, idx.unsqueeze(2)))


# ---------------------------------------------------------------- what a pass cannot do without


def _picks(c):
    """Filled (token, slot) pairs: token at position p has min(p + 1, topk)."""
    lo, n, k = c["S_kv"] - c["S"], c["S"], min(c["topk"], c["S_kv"])
    ramp = max(0, min(n, k - lo))                      # tokens with fewer than k positions
    return c["B"] * (ramp * lo + ramp * (ramp + 1) // 2 + (n - ramp) * k)


def work(case):
    c, kind = case, case["kind"]
    B, S, S_kv = c["B"], c["S"], c["S_kv"]
    nbytes = flops = 0
    if kind in ("attn_train", "attn_fwd", "layer"):
        H, D, V = c["H"], c["d_qk"], c["d_v"]
        nbytes += 2 * B * S * H * (D + V) + 2 * B * min(S_kv, S * c["topk"]) * D + 4 * B * S * H
        nbytes += 4 * B * S * c["topk"]                                          # indices: read, or the layer's output
        flops += 2 * H * _picks(c) * (D + V)
        if kind != "attn_fwd":
            nbytes += 2 * B * S * H * (D + V) + 2 * B * S_kv * D                 # dO, dq, dkv
            flops += 2 * H * _picks(c) * (3 * D + 2 * V)
    if kind in ("index_select", "index_topk", "index_train", "layer"):
        h, d, el = c["h"], c["d"], 1 if c["dtype"] == "fp8" else 2
        pairs = B * (S * (S + 1) // 2 if S == S_kv else S * S_kv)                # causal, or every cached key
        inputs = el * B * d * (S * h + S_kv) + 4 * B * S * h
        nbytes += inputs
        flops += 2 * h * d * pairs
        if kind == "index_topk":
            nbytes += 4 * B * S * c["topk"]
        if kind in ("index_select", "index_train"):
            nbytes += 8 * B * S * c["topk"] + 4 * S * S_kv                       # int64 picks, mask
        if kind == "index_select":
            nbytes += 4 * B * S * S_kv
        if kind == "index_train":
            nbytes += inputs + 2 * B * c["np"] * c["hn"] * (S + S_kv)            # dq, dw, dk; query, key
            flops += 4 * h * d * pairs + 2 * c["np"] * c["hn"] * pairs
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    """About four times the error seen against ``exact`` over the ranges: bf16 outputs and gradients are off by 2.0e-3
    to 2.4e-3 (rel) and up to 0.14 (one dq element, max), the e4m3 path by up to 5.9e-3 and 1.07 (an element of a
    nearly empty dq row), f32 scores by 6.6e-8 and 8.3e-7.  ``differ``: two scores that round across each other swap
    a pick, which moves up to a row's top-k slots."""
    kind = case["kind"]
    if kind == "index_select":
        return dict(rel=5e-7, max=5e-6, differ=0.002)
    if kind == "index_topk":
        return dict(rel=0.0, differ=0.002)
    if kind == "index_train":
        return dict(rel=0.01, max=0.1, differ=0.002)
    if case["dtype"] == "fp8":
        return dict(rel=0.024, max=0.99)
    return dict(rel=0.01, max=0.5, differ=0.002)


# ---------------------------------------------------------------- the same in 64 bits


def _e4m3(x):
    """The values that tensorwise e4m3 stands for: one scale 448 / amax, codes rounded to nearest even."""
    scale = 448.0 / x.float().abs().max()
    return (x.float() * scale).clamp(-448, 448).to(torch.float8_e4m3fn).double() / scale.double()


def _attention_exact(s):
    c = s["case"]
    q, kv = s["q"].detach(), s["kv"].detach()
    q, kv = (_e4m3(q), _e4m3(kv)) if c["dtype"] == "fp8" else (q, kv.double())
    B, S, H, D = q.shape
    V, train = c["d_v"], "do" in s
    out = torch.empty((B, S, H, V), dtype=torch.float64, device="cuda")
    lse = torch.empty((B, S, H), dtype=torch.float64, device="cuda")
    dq = torch.empty((B, S, H, D), dtype=torch.float64, device="cuda") if train else None
    dkv = torch.zeros_like(kv) if train else None
    step = max(1, (1 << 28) // (c["topk"] * max(D, H) * 8))
    for b in range(B):
        for t0 in range(0, S, step):
            sl = slice(t0, min(S, t0 + step))
            ix = s["indices"][b, sl, 0].long()
            off = (ix < 0)[:, None]
            rows = kv[b, ix.clamp(min=0), 0]                                     # [n, topk, D]
            qt = q[b, sl].double()
            z = (qt @ rows.transpose(1, 2) * s["scale"]).masked_fill_(off, -math.inf)
            z2 = torch.logsumexp(z, dim=-1)
            p = torch.exp(z - z2[..., None])
            o = p @ rows[..., :V]
            out[b, sl], lse[b, sl] = o, z2 / math.log(2)
            if train:
                do = s["do"][b, sl].double()
                ds = p * (do @ rows[..., :V].transpose(1, 2) - (o * do).sum(-1, keepdim=True)) * s["scale"]
                dq[b, sl] = ds @ rows
                drow = ds.transpose(1, 2) @ qt
                drow[..., :V] += p.transpose(1, 2) @ do
                dkv[b, :, 0].index_add_(0, ix.clamp(min=0).reshape(-1), drow.masked_fill_((ix < 0)[..., None], 0.0).reshape(-1, D))
    return dict(out=out, lse=lse, dq=dq, dkv=dkv) if train else dict(out=out, lse=lse)


def _scores_exact(s, b, sl):
    """[n, S_kv] scores of query tokens ``sl`` of batch b, -inf above the diagonal."""
    z = torch.zeros((sl.stop - sl.start, s["ik"].shape[0]), dtype=torch.float64, device="cuda")
    k = s["ik"][:, b].detach().double()
    for h in range(s["iq"].shape[2]):
        z += s["iw"][sl, b, h, None].detach().double() * (s["iq"][sl, b, h].detach().double() @ k.T).clamp_(min=0)
    return z + s["mask"][sl].double()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("index_topk", "layer"):
        return None                                                              # follows from the picks, which ties decide
    s = prepare(case, seed)
    if kind in ("attn_train", "attn_fwd"):
        return _attention_exact(s)
    B, S = c["B"], c["S"]
    if kind == "index_select":
        return dict(scores=torch.stack([_scores_exact(s, b, slice(0, S)) for b in range(B)]), idx=None)
    iq, iw, ik = (s[n].detach().double() for n in ("iq", "iw", "ik"))
    dq, dw, dk = torch.zeros_like(iq), torch.zeros_like(iw), torch.zeros_like(ik)
    total = torch.zeros((), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // S)
    for b in range(B):
        for t0 in range(0, S, step):
            sl = slice(t0, min(S, t0 + step))
            z = _scores_exact(s, b, sl)
            keep = torch.zeros_like(z, dtype=torch.bool).scatter_(1, z.topk(min(c["topk"], S), dim=-1).indices, True)
            keep &= z > -math.inf
            lq = torch.log_softmax(z.masked_fill(~keep, -math.inf), dim=-1)
            Q = lq.exp()
            P = torch.zeros_like(z)
            for n in range(c["np"]):
                a = s["query"][sl, b, n].double() @ s["key"][:, b, n].double().T * c["hn"] ** -0.5
                P += torch.softmax(a.masked_fill_(~keep, -math.inf), dim=-1) / c["np"]
            total += (P * ((P + 1e-10).log() - (Q + 1e-10).log())).sum()
            R = P * Q / (Q + 1e-10)
            G = (Q * R.sum(-1, keepdim=True) - R) / (B * S)
            for h in range(c["h"]):
                logits = iq[sl, b, h] @ ik[:, b].T
                dw[sl, b, h] = (G * logits.clamp(min=0)).sum(-1)
                M = G * (logits > 0) * iw[sl, b, h, None]
                dq[sl, b, h] = M @ ik[:, b]
                dk[:, b] += M.T @ iq[sl, b, h]
    return dict(idx=None, loss=total / (B * S), dq=dq, dw=dw, dk=dk)
