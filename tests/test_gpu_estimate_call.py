"""GPU: xattn_estimate's one-call form and the selection that follows the estimate in the same kernel give the bits of the
separate passes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows that see one key tile (with the remainders of a tile, several heads in one, padded and dead rows, no causality) and
# rows that see more
@pytest.mark.parametrize("q_len,cache,heads,kv_heads,stride,chunk,causal", [
    (1, 0, 2, 1, 16, 128, True),
    (200, 0, 4, 2, 16, 2048, True),
    (1000, 0, 32, 8, 16, 2048, True),
    (2048, 0, 3, 1, 16, 2048, True),
    (1024, 0, 8, 8, 8, 1024, True),
    (500, 0, 6, 2, 4, 512, True),
    (500, 8700, 32, 8, 16, 16384, True),
    (700, 0, 4, 4, 8, 1024, False),
    # as many candidates as a key tile has blocks, with each stride
    (2048, 0, 4, 2, 16, 2048, False),
    (1024, 0, 4, 4, 8, 1024, False),
    (512, 0, 6, 2, 4, 512, True),
    (512, 0, 3, 1, 4, 512, False),
    (2049, 0, 4, 2, 16, 4096, True),
    (5000, 0, 8, 2, 8, 2048, True),
    (300, 7000, 8, 2, 8, 1024, True),
    # key blocks fewer than a workgroup's threads for them, up to four times as many, more, no multiple of four; rows of padding alone
    (1000, 0, 4, 2, 16, 16384, True),
    (4736, 0, 2, 1, 8, 128, True),
    (650, 12000, 4, 1, 16, 128, False),
    (3000, 0, 8, 8, 4, 1024, True),
    (9000, 0, 3, 1, 8, 2048, False),
])
@pytest.mark.parametrize("use_triton,tau", [(True, 0.9), (False, 0.7)])
def test_one_call_equals_the_separate_passes(q_len, cache, heads, kv_heads, stride, chunk, causal, use_triton, tau):
    from xattn.src.Xattention import Xattention_prefill, block_sparse_attention, estimate_and_select, xattn_estimate

    g = torch.Generator(device="cuda").manual_seed(q_len + cache)
    rnd = lambda h, n: torch.randn(1, n, h, 128, generator=g, device="cuda").bfloat16().transpose(1, 2)
    q, k, v = rnd(heads, q_len), rnd(kv_heads, q_len + cache), rnd(kv_heads, q_len + cache)
    kw = dict(chunk_size=chunk, causal=causal, use_triton=use_triton)
    taus = torch.full((heads,), tau)
    sums, mask = xattn_estimate(q, k, 128, stride, threshold=taus, **kw)
    r = estimate_and_select(q, k, stride, taus, **kw)               # block sums in memory, selection as a pass of its own
    assert sums.dtype == torch.bfloat16 and mask.dtype == torch.bool and sums.shape == mask.shape == (1, *r["sums"].shape)
    assert torch.equal(sums[0], r["sums"].bfloat16())
    assert torch.equal(mask[0], r["mask"].bool())
    out = Xattention_prefill(q, k, v, stride, threshold=taus, **kw)
    nq = (q_len + 127) // 128
    idx, cnt = r["col_idx"][:, :nq].contiguous(), r["col_cnt"][:, :nq].contiguous()
    assert torch.equal(out, block_sparse_attention(q, k, v, idx, cnt, causal=causal))
