"""A NaN in q, kv or dO of the wide (d_qk = 576) kernels reaches every result that depends
on it and no other: the results without it elsewhere, bit for bit.  The forward's kernels
(unpipelined, pipelined, split slots) and the backward's, whose fp16 rows take their scale
from a maximum that drops NaN."""
import pytest
import torch

from cppmega_amd.sparse_mla_ops import sparse_mla_bwd, sparse_mla_fwd_interface

pytestmark = pytest.mark.gpu

D = 576


@pytest.mark.parametrize("where", ["q", "kv", "do"])
@pytest.mark.parametrize("S,S_kv,H,DV,topk,fp32_rows", [
    (5, 400, 128, 512, 300, False),    # forward: split slots
    (40, 300, 96, 512, 64, False),     # unpipelined
    (70, 300, 128, 512, 200, True),    # pipelined, two tiles
    (200, 500, 128, 512, 40, False),   # pipelined, four tiles
    (20, 200, 160, 576, 50, False),    # two partial rows per slot
])
def test_nan_stays_with_its_dependants(dev, S, S_kv, H, DV, topk, fp32_rows, where):
    g = torch.Generator(device=dev).manual_seed(S + H)
    make = lambda *shape: (torch.randn(shape, generator=g, device=dev) * 0.5).to(torch.bfloat16)
    q, kv, do = make(1, S, H, D), make(1, S_kv, 1, D), make(1, S, H, DV)
    idx = torch.rand((1, S, 1, S_kv), generator=g, device=dev).argsort(dim=-1)[..., :topk].to(torch.int32)
    idx[0, :, 0, 5:7] = -1
    idx = idx.contiguous()
    scale = D ** -0.5

    def run():
        out, lse = sparse_mla_fwd_interface(q, kv, idx, sm_scale=scale, d_v=DV)
        return (out, *sparse_mla_bwd(q, kv, out, do, idx, lse, sm_scale=scale, fp32_partials=fp32_rows))

    clean = run()
    t, h, r = S // 2, H - 3, int(idx[0, S // 2, 0, 11])
    bad = torch.zeros((S, H), dtype=torch.bool, device=dev)     # (token, head) pairs whose dq is NaN
    if where == "kv":
        kv[0, r, 0, 100] = torch.nan
        bad[(idx[0, :, 0] == r).any(-1)] = True
    else:
        bad[t, h] = True
        (q if where == "q" else do)[0, t, h, 7] = torch.nan
    dirty = run()
    rows = torch.zeros(S_kv, dtype=torch.bool, device=dev)      # kv rows that such a pair contributes to
    picks = idx[0, bad.any(-1), 0].long()
    rows[picks[picks >= 0]] = True
    none = torch.zeros_like(bad)
    for name, c, d, mask in zip(("out", "dq", "dkv"), clean, dirty, (none if where == "do" else bad, bad, rows[:, None])):
        assert not bool(c.isnan().any())
        nan = mask[..., None].expand_as(d[0])
        assert bool(d[0][nan].isnan().all()), name
        assert torch.equal(d[0][~nan], c[0][~nan]), name
