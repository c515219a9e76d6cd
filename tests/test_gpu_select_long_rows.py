"""GPU: rows whose selection ends by ranking at once, by search, in a run of equal sums, or by the sort, vs the oracle."""
import pytest
import torch

from helpers import mask_mismatch_report
from oracle import xattn_oracle as O
from test_gpu_select_prefill import _select

pytestmark = pytest.mark.gpu


# candidates around the limits of each way (16, 64 and 1024), few and many kept blocks, sums all distinct, in a few equal
# values (long runs of ties) and spread over many binades
@pytest.mark.parametrize("nk", [9, 16, 17, 41, 64, 65, 130, 511, 1024, 1025])
@pytest.mark.parametrize("kind", ["distinct", "ties", "equal", "steep"])
@pytest.mark.parametrize("causal,off", [(True, 0), (True, 7), (False, 0)])
def test_long_rows(nk, kind, causal, off):
    g = torch.Generator().manual_seed(nk)
    H, nq = 4, min(nk - off, 24)
    off = nk - nq if off else 0
    x = torch.rand(H, nq, nk, generator=g) + 0.01
    if kind == "ties":
        x = (x * 4).ceil() / 4
    elif kind == "equal":
        x = torch.full_like(x, 0.125)
    elif kind == "steep":
        x = torch.exp2(-24 * x)
    if causal:
        x = torch.where(torch.arange(nk)[None, :] <= torch.arange(nq)[:, None] + off, x, torch.zeros(()))
    tau = torch.tensor([0.5, 0.9, 0.99, 1.0])
    want = O.find_blocks_chunked(x[None], off, tau, None, False, "prefill", causal=causal)[0].bool()
    if causal:
        want &= torch.arange(nk)[None, :] <= torch.arange(nq)[:, None] + off
    got, idx, cnt = _select(x, tau, causal, off)
    _, outside = mask_mismatch_report(x, got, want, tau, causal, off, nq)
    assert outside == 0
    for h in range(H):
        for r in range(nq):
            assert idx[h, r, : cnt[h, r]].tolist() == got[h, r].nonzero().flatten().tolist()


# the first query chunk, whose rows have one forced block and judge the others by the mass ahead of their predecessor: all numbers of
# candidates up to nk, and so the edges of the sorts (8, 16, 32, 64 lanes) and of the registers (128, 256, 512, 1024); tau at which the
# search ends with a few, with 63 and in a run of equal sums, and sums that outrank the forced blocks
@pytest.mark.parametrize("nk", [8, 33, 65, 129, 257, 513, 1030])
@pytest.mark.parametrize("kind", ["distinct", "ties", "steep", "outranking"])
def test_rows_of_all_lengths_with_one_forced_block(nk, kind):
    g = torch.Generator().manual_seed(nk + 1)
    H = 3
    x = torch.rand(H, nk, nk, generator=g) + 0.01
    if kind == "ties":
        x = (x * 4).ceil() / 4
    elif kind == "steep":
        x = torch.exp2(-24 * x)
    elif kind == "outranking":
        x = torch.exp2(12 * x) * 100.0
    x = x * torch.tril(torch.ones(nk, nk))
    tau = torch.tensor([0.3, 0.8, 0.97])
    want = O.find_blocks_chunked(x[None], 0, tau, None, False, "prefill", causal=True)[0].bool()
    want &= torch.arange(nk)[None, :] <= torch.arange(nk)[:, None]
    got, idx, cnt = _select(x, tau, True, 0)
    _, outside = mask_mismatch_report(x, got, want, tau, True, 0, nk)
    assert outside == 0
    assert torch.equal(cnt, got.sum(-1).int())
    columns = torch.arange(nk).expand_as(got)
    lists = torch.where(got, columns, nk).sort(-1).values
    assert torch.equal(torch.where(torch.arange(nk) < cnt[..., None], idx, nk), lists.int())
