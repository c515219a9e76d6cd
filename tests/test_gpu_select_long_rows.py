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
