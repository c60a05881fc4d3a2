"""Top-k kernels on both sides of the row-count lines, and the scores of few tokens.

Few rows of over 2048 columns run a workgroup of 4 to 16 waves per row, many
rows one wave (up to 8192 columns) or 4 or 8 waves: every kernel at the edges
of its column range, bit for bit against the oracle.  The indexer's key chunk
shrinks with the grid: ragged key counts around its sizes against the oracle.
"""
import numpy as np
import pytest
import torch

from cppmega_amd import index_scores, topk_indices
from oracle import fp8 as ofp8
from oracle import indexer as oix
from oracle import topk as otk

pytestmark = pytest.mark.gpu


def _rows(rows, n, seed):
    """Normal scores, rows of ties, of a few finite columns, of values ulps apart, and infinities and NaN."""
    g = np.random.default_rng(seed)
    s = g.standard_normal((rows, n)).astype(np.float32)
    s[1::5] = np.round(s[1::5] * 4) / 4
    s[2::5, 70:] = -np.inf
    s[3::5] = (np.float32(1.0).view(np.int32) + g.integers(0, 900, s[3::5].shape)).astype(np.int32).view(np.float32)
    s[4::5, ::97] = np.nan
    s[4::5, 5::89] = np.inf
    s[4::5, 7::83] = -0.0
    return s


@pytest.mark.parametrize("rows,n", [
    (5, 2049), (1024, 4096), (1025, 4096), (5, 4097), (1024, 8192), (1025, 8192),
    (5, 8193), (256, 16384), (257, 16384), (5, 16385), (256, 32768), (257, 32768),
])
@pytest.mark.parametrize("topk", [100, 2048])
def test_row_count_lines(dev, rows, n, topk):
    s = _rows(min(rows, 25), n, seed=n + topk)
    s = np.tile(s, (rows // len(s) + 1, 1))[:rows]
    got = topk_indices(torch.from_numpy(s).to(dev), topk, causal=False).cpu().numpy()
    ref = otk.topk_ascending(s[:25], topk)
    np.testing.assert_array_equal(got[:25], ref)
    np.testing.assert_array_equal(got, np.tile(ref, (rows // len(ref) + 1, 1))[:rows])


@pytest.mark.parametrize("n", [4096, 8192, 16384])
def test_few_causal_rows(dev, n):
    """Windows that end anywhere in the row: waves with part of a segment or none."""
    s = _rows(40, n, seed=n)
    starts = torch.arange(40, dtype=torch.int32) * 11
    ends = (torch.arange(40, dtype=torch.int32) * (n // 40) + 1 + (torch.arange(40, dtype=torch.int32) % 3) * 63).clamp(max=n)
    got = topk_indices(torch.from_numpy(s).to(dev), 300, starts=starts.to(dev), ends=ends.to(dev)).cpu().numpy()
    np.testing.assert_array_equal(got, otk.topk_ascending(s, 300, starts.numpy(), ends.numpy()))


@pytest.mark.parametrize("Sq,Sk,B,H,D", [
    (1, 1, 1, 16, 64), (1, 129, 3, 64, 128), (1, 4097, 2, 32, 64), (3, 2111, 2, 16, 128), (4, 2048, 1, 16, 64),
    (5, 1000, 1, 16, 64), (2, 3000, 16, 64, 64),
])
@pytest.mark.parametrize("causal", [0, 1])
def test_scores_of_few_tokens(dev, Sq, Sk, B, H, D, causal):
    g = torch.Generator().manual_seed(Sq * 31 + Sk)
    q = torch.randn((Sq, B, H, D), generator=g).to(torch.bfloat16)
    k = torch.randn((Sk, B, D), generator=g).to(torch.bfloat16)
    w = torch.randn((Sq, B, H), generator=g) / H ** 0.5
    ref = oix.compute_index_scores(q, w, k)
    got = index_scores(q.to(dev), w.to(dev), k.to(dev), causal=causal).cpu()
    if causal:
        ref = ref.masked_fill(torch.ones(Sq, Sk, dtype=torch.bool).triu(1), float("-inf"))
    assert torch.equal(torch.isneginf(got), torch.isneginf(ref))
    fin = torch.isfinite(ref)
    # fp32 sums in another order: the bar of the dense score tests
    assert (got[fin] - ref[fin]).abs().max() <= 1e-3 * ref[fin].abs().max().clamp_min(1e-6)


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("Sq,Sk,B,H,D,fp8", [
    # e4m3: one wave's tokens, whose keys the four waves share by 32-key sub-tiles (tiles of 128 keys at D 128, 256 at 64)
    (1, 127, 2, 64, 128, True), (1, 129, 2, 64, 128, True), (1, 511, 1, 64, 128, True), (1, 2049, 3, 64, 128, True),
    (1, 257, 2, 64, 64, True), (2, 255, 1, 32, 64, True), (4, 2047, 2, 16, 64, True), (2, 513, 3, 32, 128, True),
    (1, 5000, 16, 64, 128, True),
    # e4m3: more tokens, chunks of one tile and more
    (5, 300, 2, 64, 128, True), (17, 600, 1, 16, 64, True),
    # bf16 rows of 256 bytes: whole, 512-key and 256-key chunks at one workgroup a compute unit
    (64, 512, 16, 64, 128, False), (16, 256, 32, 64, 128, False), (8, 8193, 4, 64, 128, False),
])
def test_scores_of_few_tokens_write_every_column(dev, Sq, Sk, B, H, D, fp8, causal):
    """Every column is owned by exactly one wave: an output full of NaN is overwritten."""
    g = torch.Generator().manual_seed(Sq * 17 + Sk)
    q = torch.randn((Sq, B, H, D), generator=g).to(torch.bfloat16)
    k = torch.randn((Sk, B, D), generator=g).to(torch.bfloat16)
    w = torch.randn((Sq, B, H), generator=g) / H ** 0.5
    kw = {}
    if fp8:
        q, qs = ofp8.tensorwise_quantize(q)
        k, ks = ofp8.tensorwise_quantize(k)
        kw = dict(q_scale=qs.to(dev), k_scale=ks.to(dev))
        ref = oix.compute_index_scores(q.float(), w, k.float(), q_scale=qs, k_scale=ks)
    else:
        ref = oix.compute_index_scores(q, w, k)
    out = torch.full((B, Sq, Sk), float("nan"), device=dev)
    got = index_scores(q.to(dev), w.to(dev), k.to(dev), causal=causal, out=out, **kw).cpu()
    if causal:
        ref = ref.masked_fill(torch.ones(Sq, Sk, dtype=torch.bool).triu(1), float("-inf"))
    assert torch.equal(torch.isneginf(got), torch.isneginf(ref)) and not bool(got.isnan().any())
    fin = torch.isfinite(ref)
    # fp32 sums in another order: the bar of the dense score tests
    assert (got[fin] - ref[fin]).abs().max() <= 1e-3 * ref[fin].abs().max().clamp_min(1e-6)
