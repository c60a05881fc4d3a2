"""The KL loss's kernels by size: 256- and 128-token blocks of the pass, the sparse
statistics by lane masks and by row bitmask, key heads shared by groups.  A large batch,
which takes the former of each pair, against the same sequences one at a time, which take
the latter; the single sequences against the oracle."""
import pytest
import torch

from cppmega_amd import indexer_kl_loss
from oracle import indexer_loss as oil

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparse", [False, True], ids=["dense", "sparse"])
@pytest.mark.parametrize("B,S,H,G,D", [
    (45, 300, 8, 2, 128),      # 270 items of 128 tokens: 256-token blocks; row bitmask in both
    (2, 900, 64, 64, 128),     # 104 M scores: lane masks
    (45, 200, 8, 8, 192),      # both, chunks of 64 keys
    (16, 300, 16, 4, 256),     # lane masks; always 128 tokens
    (3, 70, 6, 1, 64),         # one key head for all
])
def test_batch_matches_single_sequences(dev, B, S, H, G, D, sparse):
    g = torch.Generator(device=dev).manual_seed(S + D)
    query = torch.randn((S, B, H, D), generator=g, device=dev).to(torch.bfloat16)
    key = torch.randn((S, B, G, D), generator=g, device=dev).to(torch.bfloat16)
    z = torch.randn((B, S, S), generator=g, device=dev)
    idx = torch.rand((B, S, S), generator=g, device=dev).argsort(dim=-1)[..., :S // 5].contiguous()
    idx[..., 0] = 0                                        # every row has a column of its past
    scale = D ** -0.5

    def run(z, idx, query, key):
        zr = z.clone().requires_grad_()
        grad, = torch.autograd.grad(indexer_kl_loss(zr, idx, query, key, scale, float(z.shape[0] * S), sparse), zr)
        with torch.no_grad():
            _, rows = indexer_kl_loss(z, idx, query, key, scale, float(z.shape[0] * S), sparse, return_rows=True)
        return grad, rows

    grad, rows = run(z, idx, query, key)
    for b in (0, B - 1):
        sl = slice(b, b + 1)
        one = (z[sl], idx[sl], query[:, sl].contiguous(), key[:, sl].contiguous())
        g1, r1 = run(*one)
        # the same sums in another kernel's order and contractions: S terms of 2^-24, twice
        torch.testing.assert_close(rows[sl], r1, rtol=S * 2.0 ** -23, atol=S * 2.0 ** -23)
        assert float((grad[sl] - g1).abs().max()) <= S * 2.0 ** -23 * float(g1.abs().max())
        ref = oil.indexer_kl_rows(*(t.cpu() for t in one), scale, sparse)
        # fp32 exponents of up to 30: 30 * 2^-24 of P, times the logarithms' up to 20, with a margin of 2
        torch.testing.assert_close(r1.cpu().double(), ref, rtol=1e-4, atol=1e-4)
