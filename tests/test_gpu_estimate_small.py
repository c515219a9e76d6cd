"""GPU: the estimator's pass for small launches gives the bits of the 256x256-tile pass.

A slab-pair list always runs on the large tiles; given the antidiagonal's own pairs it computes the same scores in the
same order, so block sums and masks have to be equal, not close."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# tiles of 32, 64 and 128 rows with and without remainders; heads that share a tile (cached chunks of few tokens, groups of
# 3, 4 and 7 heads); one and many key tiles; rows whose tile has keys nobody sees; a padded, non-causal tail
@pytest.mark.parametrize("q_len,cache,heads,kv_heads,stride,chunk,causal", [
    (200, 0, 4, 2, 16, 2048, True),
    (1000, 0, 32, 8, 16, 2048, True),
    (1100, 0, 6, 2, 8, 2048, True),
    (129, 0, 3, 1, 4, 256, True),
    (2500, 0, 32, 8, 8, 4096, True),
    (4096, 0, 32, 32, 8, 2048, True),
    (6001, 0, 32, 8, 16, 2048, True),
    (64, 20000, 28, 4, 16, 2048, True),
    (130, 9000, 12, 4, 16, 1024, True),
    (300, 5001, 8, 2, 8, 512, True),
    (2048, 30000, 32, 8, 16, 2048, True),
    (700, 0, 8, 8, 8, 1024, False),
    (100, 3000, 32, 8, 8, 128, False),
    # rows of several heads packed into large tiles: whole quarters, 64-row pieces of 7 heads with two left empty, a ragged
    # last piece, no causality
    (2048, 60000, 32, 8, 16, 2048, True),
    (1500, 18000, 28, 4, 8, 2048, True),
    (5000, 30000, 32, 8, 16, 2048, True),
    (1900, 60001, 32, 8, 16, 4096, False),
    # half tiles behind whole rounds: what does not fill a round, a last row tile of one half, both, no causality
    (32768, 0, 30, 10, 16, 2048, True),
    (15000, 0, 32, 8, 8, 2048, True),
    (10500, 0, 28, 4, 8, 1024, True),
    (18000, 0, 28, 4, 16, 1024, False),
])
@pytest.mark.parametrize("use_triton", [True, False])
def test_same_bits_as_the_large_tiles(q_len, cache, heads, kv_heads, stride, chunk, causal, use_triton):
    from xattn.src.Xattention import estimate_and_select

    g = torch.Generator(device="cuda").manual_seed(q_len + cache)
    rnd = lambda h, n: torch.randn(1, n, h, 128, generator=g, device="cuda").bfloat16().transpose(1, 2)
    q, k = rnd(heads, q_len), rnd(kv_heads, q_len + cache)
    pairs = [(stride - 1 - i, i) for i in range(stride)]
    a = estimate_and_select(q, k, stride, 0.9, chunk, causal=causal, use_triton=use_triton)
    b = estimate_and_select(q, k, stride, 0.9, chunk, causal=causal, use_triton=use_triton, slab_pairs=pairs)
    for name in ("sums", "mask", "col_cnt"):
        assert torch.equal(a[name], b[name]), name
