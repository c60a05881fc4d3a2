"""The KL loss's saved gradient state (autograd path) against the gradient call,
bit for bit, and against the loss and gradient kernels that keep no state: top-k
lists unsorted, padded, repeated, beyond the diagonal; chunk and word edges; rows
without a target; several upstream factors."""
import pytest
import torch

from cppmega_amd import _lib, indexer_kl_loss, indexer_kl_loss_backward

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparse", [False, True], ids=["dense", "sparse"])
@pytest.mark.parametrize("b,sq,sk,np_,hn,topk", [
    (2, 130, 130, 4, 64, 40),     # a chunk edge at 128 keys
    (1, 33, 2081, 2, 128, 70),    # more than 64 mask words, a ragged last word, keys beyond every diagonal
    (1, 97, 63, 2, 192, 63),      # chunks of 64 keys, rows past the last key
    (1, 20, 20, 1, 64, 1),
])
def test_state_gradient_matches_direct(dev, b, sq, sk, np_, hn, topk, sparse):
    g = torch.Generator().manual_seed(sq * sk + topk)
    z = torch.randn((b, sq, sk), generator=g)
    idx = torch.rand((b, sq, max(sk, topk)), generator=g).argsort(dim=-1)[..., :topk]
    idx = torch.where(torch.rand(idx.shape, generator=g) < 0.2, torch.full_like(idx, -1), idx)
    if topk > 4:
        idx[:, :, 3] = idx[:, :, 1]                       # repeats
    idx[0, sq // 2] = -1                                  # no column: a NaN row (sparse)
    z[0, 0, sk // 2] = -torch.inf
    query = torch.randn((sq, b, np_, hn), generator=g).to(torch.bfloat16).to(dev)
    key = torch.randn((sk, b, np_, hn), generator=g).to(torch.bfloat16).to(dev)
    idx, scale = idx.contiguous().to(dev), hn ** -0.5
    zr = z.to(dev).requires_grad_()
    loss = indexer_kl_loss(zr, idx, query, key, scale, 0.7, sparse)
    with torch.no_grad():
        plain, rows = indexer_kl_loss(zr.detach(), idx, query, key, scale, 0.7, sparse, return_rows=True)
    assert torch.equal(loss.detach().isnan(), plain.isnan()) and (bool(plain.isnan()) or loss.detach() == plain)
    assert bool(rows.isnan().any()) == sparse
    lib = _lib.load()
    for f in (1.0, -3.25):
        gl = torch.tensor([f], device=dev)
        got, = torch.autograd.grad(loss, zr, gl[0], retain_graph=True)
        want = indexer_kl_loss_backward(gl[0], zr.detach(), idx, query, key, scale, 0.7, sparse)
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.nan_to_num(), want.nan_to_num())
        direct = torch.empty_like(got)
        ws = torch.empty(int(lib.dsa_indexer_kl_loss_workspace_size(b, sq, sk, np_, hn, int(sparse))), dtype=torch.uint8,
                         device=dev)
        zd = zr.detach().contiguous()
        _lib.check(lib.dsa_indexer_kl_loss_backward(
            zd.data_ptr(), idx.data_ptr() if sparse else None, _lib.DTYPE_I64, topk if sparse else 0, query.data_ptr(),
            key.data_ptr(), gl.data_ptr(), direct.data_ptr(), b, sq, sk, np_, np_, hn, scale, 0.7, int(sparse),
            ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "dsa_indexer_kl_loss_backward")
        assert torch.equal(got.isnan(), direct.isnan())
        got, direct = got.nan_to_num(), direct.nan_to_num()
        # the same terms summed in another order: at most sk + sq of them, 2^-24 each
        bound = (sk + sq) * 2.0 ** -24
        assert float((got - direct).abs().max()) <= 2 * bound * float(direct.abs().max())


@pytest.mark.parametrize("value", ["nan", "inf"])
@pytest.mark.parametrize("where", ["query", "key"])
def test_nan_or_inf_in_one_head_makes_the_row_nan(dev, where, value):
    """A row whose loss is not finite has a NaN gradient over all its columns, those outside
    its top-k set too, whichever head the NaN or infinity comes from (query: row 40; key:
    the rows that pick key 30, of an infinite key those it scores +inf: -inf is no weight)."""
    b, s, np_, hn, topk = 2, 70, 3, 64, 12
    g = torch.Generator().manual_seed(9)
    z = torch.randn((b, s, s), generator=g).masked_fill_(torch.ones(s, s, dtype=torch.bool).triu(1), -torch.inf).to(dev)
    idx = z.topk(topk, dim=-1).indices.contiguous()
    query = torch.randn((s, b, np_, hn), generator=g).to(torch.bfloat16).to(dev)
    key = torch.randn((s, b, np_, hn), generator=g).to(torch.bfloat16).to(dev)
    if where == "query":
        query[40, 1, 2, 5] = float(value)
        bad = torch.zeros((b, s), dtype=torch.bool, device=dev)
        bad[1, 40] = True
    else:
        key[30, 1, 1, 7] = float(value)
        bad = ((idx == 30).any(-1)) & (torch.arange(s, device=dev) >= 30)
        bad[0] = False
        if value == "inf":
            bad[1] &= query[:, 1, 1, 7] > 0
        assert 0 < int(bad.sum()) < s - 30
    with torch.no_grad():
        _, rows = indexer_kl_loss(z, idx, query, key, hn ** -0.5, 1.0, True, return_rows=True)
    assert torch.equal(~rows.isfinite(), bad)
    zr = z.clone().requires_grad_()
    loss = indexer_kl_loss(zr, idx, query, key, hn ** -0.5, 1.0, True)
    assert not bool(loss.isfinite())
    grad, = torch.autograd.grad(loss, zr)
    assert torch.equal(grad.isnan(), bad[..., None].expand_as(grad))
    assert torch.equal(indexer_kl_loss_backward(1.0, z, idx, query, key, hn ** -0.5, 1.0, True).isnan(), grad.isnan())
