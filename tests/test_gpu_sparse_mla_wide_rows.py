"""The wide backward's two kernels at the edges of their splits: head groups of
one partial row (128 heads), 32-head tiles per workgroup (one, two, an odd
count), kv groups, 32-slot blocks, and both partial-row formats, against the
oracle at the usual bar (2e-2 relative / 1e-2 absolute)."""
import pytest
import torch

from cppmega_amd import synthetic
from cppmega_amd.sparse_mla_ops import sparse_mla_bwd, sparse_mla_bwd_fp8, sparse_mla_fwd_fp8_interface, \
    sparse_mla_fwd_interface
from oracle import fp8 as ofp8
from oracle import sparse_mla as orc
from tests._util import assert_close

pytestmark = pytest.mark.gpu

D = 576


@pytest.mark.parametrize("S,S_kv,H,G,DV,topk,fp32_rows", [
    (24, 24, 8, 1, 512, 32, False),      # one partial head tile
    (20, 90, 160, 1, 512, 33, False),    # two rows per entry, the second of one tile; ragged last block
    (20, 90, 288, 1, 512, 31, True),     # three rows per entry, fp32
    (18, 70, 192, 2, 512, 65, False),    # two kv groups of three head tiles
    (24, 40, 40, 1, 576, 96, False),     # V the whole row, a ragged second tile
    (1, 300, 128, 1, 512, 257, False),   # one token
])
def test_wide_rows_splits(dev, S, S_kv, H, G, DV, topk, fp32_rows):
    g = torch.Generator().manual_seed(H + topk)
    q = (torch.randn((1, S, H, D), generator=g) * 0.5).to(torch.bfloat16)
    kv = (torch.randn((1, S_kv, G, D), generator=g) * 0.5).to(torch.bfloat16)
    do = torch.randn((1, S, H, DV), generator=g).to(torch.bfloat16)
    idx = torch.rand((1, S, G, max(S_kv, topk)), generator=g).argsort(dim=-1)[..., :topk].to(torch.int32)
    idx[idx >= S_kv] = -1
    idx[0, 0, 0, ::3] = -1                                  # unsorted, masked slots throughout
    idx = idx.contiguous()
    scale = D ** -0.5
    qd, kd, dod, idd = q.to(dev), kv.to(dev), do.to(dev), idx.to(dev)
    out, lse = sparse_mla_fwd_interface(qd, kd, idd, sm_scale=scale, d_v=DV)
    dq, dkv = sparse_mla_bwd(qd, kd, out, dod, idd, lse, sm_scale=scale, fp32_partials=fp32_rows)
    rdq, rdkv = orc.sparse_mla_bwd(q, kv, out.cpu(), do, idx, lse.cpu(), scale, DV)
    assert_close(dq, rdq, what="dq")
    assert_close(dkv, rdkv, what="dkv")
    dq2, dkv2 = sparse_mla_bwd(qd, kd, out, dod, idd, lse, sm_scale=scale, fp32_partials=fp32_rows)
    assert torch.equal(dq, dq2) and torch.equal(dkv, dkv2)


def test_wide_rows_e4m3_two_rows_per_entry(dev):
    S, H, DV, topk = 40, 160, 512, 40
    q = (torch.randn((1, S, H, D), generator=torch.Generator().manual_seed(1)) * 0.5).to(torch.bfloat16)
    kv = (torch.randn((1, S, 1, D), generator=torch.Generator().manual_seed(2)) * 0.5).to(torch.bfloat16)
    do = torch.randn((1, S, H, DV), generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    idx = synthetic.causal_indices(1, S, topk, seed=4)
    q8, qs = ofp8.tensorwise_quantize(q)
    k8, ks = ofp8.tensorwise_quantize(kv)
    qsv, ksv = qs.expand(1, S).contiguous(), ks.expand(1, S).contiguous()
    args = [t.to(dev) for t in (q8, k8, qsv, ksv)]
    out, lse = sparse_mla_fwd_fp8_interface(args[0], args[1], idx.to(dev), q_scale=args[2], kv_scale=args[3],
                                            sm_scale=D ** -0.5, d_v=DV)
    dq, dkv = sparse_mla_bwd_fp8(*args, out, do.to(dev), idx.to(dev), lse, sm_scale=D ** -0.5)
    rdq, rdkv = orc.sparse_mla_bwd(q8, k8, out.cpu(), do, idx, lse.cpu(), D ** -0.5, DV, q_scale=qsv, kv_scale=ksv)
    assert_close(dq, rdq, what="dq")
    assert_close(dkv, rdkv, what="dkv")


@pytest.mark.parametrize("B,S,S_kv,H,G,DV,topk", [
    # the kernel, head tiles per workgroup x splits that the plan picks
    (2, 1, 3000, 128, 1, 512, 2048),     # pipelined, 1 x 16
    (20, 1, 600, 128, 1, 512, 513),      # pipelined, 1 x 3 of uneven blocks
    (3, 7, 500, 96, 1, 512, 300),        # unpipelined, one tile of three
    (1, 40, 700, 128, 1, 512, 600),      # pipelined, 2 x 3
    (1, 2, 600, 64, 2, 576, 290),        # kv groups, V the whole row: pipelined, 1 x 2
    (1, 70, 300, 128, 1, 512, 200),      # pipelined, two tiles, no split
    (1, 40, 300, 100, 1, 576, 100),      # unpipelined, one tile of four, the last ragged
    (1, 100, 300, 96, 1, 512, 70),       # unpipelined, two tiles of three (the last workgroup's second is empty)
    (1, 50, 300, 200, 2, 576, 70),       # the same with kv groups, V the whole row
    (1, 200, 300, 128, 1, 512, 40),      # pipelined, four tiles, no split
    (4, 15, 2100, 100, 1, 512, 2048),    # pipelined, 4 x 4, the last tile ragged
])
def test_wide_forward_splits(dev, B, S, S_kv, H, G, DV, topk):
    """Few tokens against a long kv: the slots of a token split over workgroups.
    One token's slots all masked, one's valid slots in its first block only."""
    g = torch.Generator().manual_seed(S_kv + topk)
    q = (torch.randn((B, S, H, D), generator=g) * 0.5).to(torch.bfloat16)
    kv = (torch.randn((B, S_kv, G, D), generator=g) * 0.5).to(torch.bfloat16)
    idx = torch.rand((B, S, G, max(S_kv, topk)), generator=g).argsort(dim=-1)[..., :topk].to(torch.int32)
    idx[idx >= S_kv] = -1
    idx[0, -1, 0] = -1
    idx[0, 0, -1, 9:] = -1
    if B > 1:
        idx[1, -1, 0, ::2] = -1
    idx = idx.contiguous()
    scale = D ** -0.5
    out, lse = sparse_mla_fwd_interface(q.to(dev), kv.to(dev), idx.to(dev), sm_scale=scale, d_v=DV)
    ro, rl = orc.sparse_mla_fwd(q, kv, idx, scale, DV)
    assert_close(out, ro, what="out")
    assert_close(lse, rl, what="lse2")


def test_wide_forward_split_matches_unsplit(dev):
    """A call given no workspace runs unsplit: the same result within rounding (bf16 out: 2^-8 of an element)."""
    from cppmega_amd import _lib
    B, S, S_kv, H, topk, DV = 4, 1, 2000, 128, 1024, 512
    g = torch.Generator().manual_seed(3)
    q = (torch.randn((B, S, H, D), generator=g) * 0.5).to(torch.bfloat16).to(dev)
    kv = (torch.randn((B, S_kv, 1, D), generator=g) * 0.5).to(torch.bfloat16).to(dev)
    idx = torch.rand((B, S, 1, S_kv), generator=g).argsort(dim=-1)[..., :topk].to(torch.int32).contiguous().to(dev)
    L = _lib.load()
    assert int(L.dsa_sparse_mla_fwd_call_workspace_size(B, S, S_kv, H, 1, D, DV, topk, _lib.DTYPE_BF16)) > 0
    out, lse = sparse_mla_fwd_interface(q, kv, idx, sm_scale=D ** -0.5, d_v=DV)
    out1, lse1 = torch.empty_like(out), torch.empty_like(lse)
    _lib.check(L.dsa_sparse_mla_fwd(q.data_ptr(), kv.data_ptr(), idx.data_ptr(), out1.data_ptr(), lse1.data_ptr(), B, S,
                                    S_kv, H, 1, D, DV, topk, D ** -0.5, _lib.DTYPE_BF16, None, None,
                                    torch.cuda.current_stream().cuda_stream), "dsa_sparse_mla_fwd")
    torch.testing.assert_close(out.float(), out1.float(), rtol=2 ** -7, atol=2 ** -7)
    torch.testing.assert_close(lse, lse1, rtol=1e-5, atol=1e-4)


def test_bf16_workspace_is_used_only_where_offered_for_splits(dev):
    """dsa_sparse_mla_fwd_ws neither reads nor writes a bf16 caller's workspace (one buffer
    may serve several streams); dsa_sparse_mla_fwd_call splits with a large enough one only,
    and refuses a misaligned one."""
    from cppmega_amd import _lib
    B, S, S_kv, H, topk, DV = 4, 1, 700, 128, 512, 512
    g = torch.Generator().manual_seed(4)
    q = (torch.randn((B, S, H, D), generator=g) * 0.5).to(torch.bfloat16).to(dev)
    kv = (torch.randn((B, S_kv, 1, D), generator=g) * 0.5).to(torch.bfloat16).to(dev)
    idx = torch.rand((B, S, 1, S_kv), generator=g).argsort(dim=-1)[..., :topk].to(torch.int32).contiguous().to(dev)
    L, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    n = int(L.dsa_sparse_mla_fwd_call_workspace_size(B, S, S_kv, H, 1, D, DV, topk, _lib.DTYPE_BF16))
    assert n > 0

    def call(fn, ws, nbytes):
        out = torch.empty((B, S, H, DV), dtype=torch.bfloat16, device=dev)
        lse = torch.empty((B, S, H), device=dev)
        rc = fn(q.data_ptr(), kv.data_ptr(), idx.data_ptr(), out.data_ptr(), lse.data_ptr(), B, S, S_kv, H, 1, D, DV, topk,
                D ** -0.5, _lib.DTYPE_BF16, None, None, ws, nbytes, st)
        return rc, out, lse

    ws = torch.full((n + 16,), 0x5a, dtype=torch.uint8, device=dev)
    rc, out, lse = call(L.dsa_sparse_mla_fwd_ws, ws.data_ptr(), n)
    assert rc == _lib.DSA_OK and bool((ws == 0x5a).all())
    for p, nbytes in ((ws.data_ptr(), n - 1), (None, 0)):           # too small, none: unsplit
        rc, o, l = call(L.dsa_sparse_mla_fwd_call, p, nbytes)
        assert rc == _lib.DSA_OK and torch.equal(o, out) and torch.equal(l, lse)
    assert bool((ws == 0x5a).all())
    assert call(L.dsa_sparse_mla_fwd_call, ws.data_ptr() + 4, n)[0] == _lib.DSA_ERR_INVALID_ARG
    rc, o, l = call(L.dsa_sparse_mla_fwd_call, ws.data_ptr(), n)
    assert rc == _lib.DSA_OK and not bool((ws[:n] == 0x5a).all()) and bool((ws[n:] == 0x5a).all())
    torch.testing.assert_close(o.float(), out.float(), rtol=2 ** -7, atol=2 ** -7)
