"""GPU: the operator's attention from a work queue (64 rows per wavefront, more than 1024 units or 256 on a cache) against a
workgroup for each unit and piece, over the same lists."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# units just past the rules' lines; pieces beside units that are whole; groups of heads that fill a run of ids (64) and that
# do not (7, 3), so that some ids stand for nothing; few long heads; two launches (the first q-blocks have 32 rows)
@pytest.mark.parametrize("q_len,cache,heads,kv_heads,long_heads,causal", [
    (16500, 0, 8, 2, [5], False),
    (2100, 16500, 16, 2, [3, 8], True),
    (1100, 17000, 30, 10, [0, 29], True),
    (2048, 20000, 28, 4, list(range(0, 28, 2)), True),
    (2048, 30000, 16, 16, list(range(16)), True),
    (66000, 0, 16, 4, [6], True),
])
def test_queue_gives_the_same_as_a_workgroup_per_unit(q_len, cache, heads, kv_heads, long_heads, causal):
    from xattn.src.Xattention import Xattention_prefill, block_sparse_attention, estimate_and_select

    g = torch.Generator(device="cuda").manual_seed(heads)
    rnd = lambda h, n: torch.randn(1, h, n, 128, generator=g, device="cuda").bfloat16()
    q, k, v = rnd(heads, q_len), rnd(kv_heads, q_len + cache), rnd(kv_heads, q_len + cache)
    taus, chunk, nq = torch.full((heads,), 0.02), 128, (q_len + 127) // 128
    taus[torch.tensor(long_heads)] = 1.0
    r = estimate_and_select(q, k, 8, taus, chunk, causal=causal, want_mask=False, want_sums=False)
    idx, cnt = r["col_idx"][:, :nq].contiguous(), r["col_cnt"][:, :nq].contiguous()
    want = block_sparse_attention(q, k, v, idx, cnt, causal=causal)
    for _ in range(3):                                            # whoever takes what
        assert torch.equal(Xattention_prefill(q, k, v, 8, threshold=taus, chunk_size=chunk, causal=causal), want)
