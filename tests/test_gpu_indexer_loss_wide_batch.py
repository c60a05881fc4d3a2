"""The KL loss where a batch's query row pitch (B * H * D * 2 bytes) times the 32 rows of a
wave passes 4 GiB: many short sequences with few key heads.  Some sequences of the batch
against the same call on those sequences alone, whose rows lie close together."""
import pytest
import torch

from cppmega_amd import indexer_kl_loss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparse", [False, True], ids=["dense", "sparse"])
@pytest.mark.parametrize("B,S,H,G,D", [
    (8704, 32, 64, 1, 128),     # one wave's tokens
    (8704, 41, 32, 2, 256),     # a second wave with part of its tokens; key heads in groups
    (17408, 33, 64, 1, 64),
])
def test_query_rows_past_4_gib(dev, B, S, H, G, D, sparse):
    assert 31 * B * H * D * 2 > 2 ** 32
    g = torch.Generator(device=dev).manual_seed(S + D)
    query = torch.randn((S, B, H, D), generator=g, device=dev, dtype=torch.bfloat16)
    key = torch.randn((S, B, G, D), generator=g, device=dev, dtype=torch.bfloat16)
    z = torch.randn((B, S, S), generator=g, device=dev)
    idx = torch.rand((B, S, S), generator=g, device=dev).argsort(dim=-1)[..., :20].contiguous()
    idx[..., 0] = 0                                        # every row has a column of its past
    zr = z.clone().requires_grad_()
    # coeff / (B * S) is the same power-of-two multiple in both calls
    grad, = torch.autograd.grad(indexer_kl_loss(zr, idx, query, key, D ** -0.5, float(B), sparse), zr)
    with torch.no_grad():
        _, rows = indexer_kl_loss(z, idx, query, key, D ** -0.5, float(B), sparse, return_rows=True)
    pick = torch.tensor([0, 1, B // 2, B - 1], device=dev)
    zp, ip, qp, kp = z[pick], idx[pick], query[:, pick].contiguous(), key[:, pick].contiguous()
    zpr = zp.clone().requires_grad_()
    want, = torch.autograd.grad(indexer_kl_loss(zpr, ip, qp, kp, D ** -0.5, 4.0, sparse), zpr)
    with torch.no_grad():
        _, wrows = indexer_kl_loss(zp, ip, qp, kp, D ** -0.5, 4.0, sparse, return_rows=True)
    # the same sums; a kernel of other registers may contract them otherwise (S terms of 2^-24)
    torch.testing.assert_close(rows[pick], wrows, rtol=S * 2.0 ** -23, atol=S * 2.0 ** -23)
    bound = S * 2.0 ** -23 * float(want.abs().max())
    assert float((grad[pick] - want).abs().max()) <= bound
