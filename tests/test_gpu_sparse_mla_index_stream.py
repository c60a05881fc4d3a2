"""The inverse index built ahead on a second stream behind an ``after`` event keeps off
memory that work queued since that event still uses."""
import pytest
import torch

from cppmega_amd import synthetic
from cppmega_amd.sparse_mla_ops import build_inverse_index, side_stream, sparse_mla_bwd, sparse_mla_fwd_interface

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,topk", [(1, 96, 33), (2, 1024, 64)])
def test_index_takes_no_block_freed_since_the_event(dev, B, S, topk):
    H, D, DV = 32, 128, 64
    inp = synthetic.sparse_mla_inputs(B, S, H, D, DV, topk, std=0.5, seed=S)
    q, kv, idx, do = (inp[k].to(dev) for k in ("q", "kv", "indices", "do"))
    out, lse = sparse_mla_fwd_interface(q, kv, idx, sm_scale=inp["scale"], d_v=DV)
    ref = sparse_mla_bwd(q, kv, out, do, idx, lse, sm_scale=inp["scale"])
    n = build_inverse_index(q, kv, idx, DV).buf.numel()
    torch.cuda.synchronize()
    after = torch.cuda.Event()
    after.record()
    work = torch.zeros(n, dtype=torch.uint8, device=dev)   # queued since the event, freed before it has run
    ptr = work.data_ptr()
    del work
    ix = build_inverse_index(q, kv, idx, DV, stream=side_stream(dev), after=after)
    assert ix.buf.data_ptr() != ptr
    got = sparse_mla_bwd(q, kv, out, do, idx, lse, sm_scale=inp["scale"], inverse_index=ix)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])


def test_two_builds_in_a_graph_keep_apart(dev):
    """Two backwards captured in one graph, each with an index built on the second stream
    behind an event recorded before either: the second build is not ordered after the first
    backward, so it must not take the first index's block, freed by then.  Every replay
    equals the eager results."""
    B, S, H, D, DV, topk = 1, 512, 32, 128, 64, 64
    inp = synthetic.sparse_mla_inputs(B, S, H, D, DV, topk, std=0.5, seed=3)
    q, kv, idx, do = (inp[k].to(dev) for k in ("q", "kv", "indices", "do"))
    idx2 = idx.flip(-1).roll(1, dims=-1).contiguous()     # the same rows in other slots
    fwd = [(i, *sparse_mla_fwd_interface(q, kv, i, sm_scale=inp["scale"], d_v=DV)) for i in (idx, idx2)]
    ref = [sparse_mla_bwd(q, kv, o, do, i, lse, sm_scale=inp["scale"]) for i, o, lse in fwd]
    torch.cuda.synchronize()
    ptrs = []

    def step():
        after = torch.cuda.Event()
        after.record()
        res = []
        for i, o, lse in fwd:
            ix = build_inverse_index(q, kv, i, DV, stream=side_stream(dev), after=after)
            ptrs.append(ix.buf.data_ptr())
            res.append(sparse_mla_bwd(q, kv, o, do, i, lse, sm_scale=inp["scale"], inverse_index=ix))
            del ix
        return res

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        res = step()
    assert ptrs[0] != ptrs[1]
    for _ in range(3):
        torch.zeros(1 << 20, device=dev).sum().item()      # eager work between replays
        graph.replay()
        torch.cuda.synchronize()
        for (dq, dkv), (rq, rkv) in zip(res, ref):
            assert torch.equal(dq, rq) and torch.equal(dkv, rkv)
