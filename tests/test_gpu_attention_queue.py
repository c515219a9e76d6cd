"""GPU: the operator's attention from a work queue (64 rows per wavefront, more than 1024 units) against a
workgroup for each unit and piece, over the same lists."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _workgroup_per_unit(q, k, v, idx, cnt, causal):
    """The entry point without a workspace: no queue, no list cut."""
    from xattn.src import hip_backend as hb

    heads, q_len, k_len = q.shape[1], q.shape[2], k.shape[2]
    out = torch.empty(1, q_len, heads, 128, dtype=torch.bfloat16, device="cuda")
    hb.check(hb.lib().xattn_block_sparse_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), idx.data_ptr(), cnt.data_ptr(), idx.shape[2], idx.shape[1], 0,
        heads, k.shape[1], q_len, k_len, 128, q.stride(1), q.stride(2), k.stride(1), k.stride(2), v.stride(1), v.stride(2),
        out.stride(2), out.stride(1), 0, -1, int(causal), 128 ** -0.5, torch.cuda.current_stream().cuda_stream), "fwd")
    return out.transpose(1, 2)


# units just past the rules' lines; pieces beside units that are whole; groups of heads that fill a run of ids (64) and that
# do not (7, 3), so that some ids stand for nothing; few long heads; two launches (the first q-blocks have 32 rows)
@pytest.mark.parametrize("q_len,cache,heads,kv_heads,long_heads,causal", [
    (16500, 0, 8, 2, [5], False),
    (2100, 16500, 16, 2, [3, 8], True),
    (1100, 17000, 30, 10, [0, 29], True),
    (2048, 20000, 28, 4, list(range(0, 28, 2)), True),
    (2048, 30000, 16, 16, list(range(16)), True),
    (66000, 0, 16, 4, [6], True),
    (10000, 0, 56, 8, [6], False),
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
    got = Xattention_prefill(q, k, v, 8, threshold=taus, chunk_size=chunk, causal=causal)
    for _ in range(2):                                            # whoever takes what
        assert torch.equal(Xattention_prefill(q, k, v, 8, threshold=taus, chunk_size=chunk, causal=causal), got)
        assert torch.equal(block_sparse_attention(q, k, v, idx, cnt, causal=causal), got)
    want = _workgroup_per_unit(q, k, v, idx, cnt, causal)
    if heads * nq > 4096:                                         # no list is cut
        assert torch.equal(got, want)
    bound = 2.0 ** -8 * (v.float().abs().amax() + want.float().abs())          # as in test_gpu_attention_plan.py
    assert ((got.float() - want.float()).abs() <= bound).all()


# prompts of 3584 units and more that see fewer than 384 blocks: of some q-blocks all lists are long (64 rows per wavefront), of
# others a few heads' or none (32 rows); more heads than lanes
@pytest.mark.parametrize("q_len,heads,kv_heads,long_heads", [
    (14300, 32, 8, list(range(0, 32))),
    (14300, 32, 8, list(range(0, 32, 3))),
    (6700, 70, 7, list(range(0, 66))),
    (14336, 32, 32, []),
    (17000, 32, 8, list(range(0, 32))),
])
def test_lists_choose_the_kernel_the_same_way_by_every_path(q_len, heads, kv_heads, long_heads):
    from xattn.src.Xattention import Xattention_prefill, block_sparse_attention, estimate_and_select

    g = torch.Generator(device="cuda").manual_seed(heads)
    rnd = lambda h, n: torch.randn(1, h, n, 128, generator=g, device="cuda").bfloat16()
    q, k, v = rnd(heads, q_len), rnd(kv_heads, q_len), rnd(kv_heads, q_len)
    taus, nq = torch.full((heads,), 0.02), (q_len + 127) // 128
    taus[torch.tensor(long_heads, dtype=torch.long)] = 0.9
    r = estimate_and_select(q, k, 16, taus, 128, want_mask=False, want_sums=False)
    idx, cnt = r["col_idx"][:, :nq].contiguous(), r["col_cnt"][:, :nq].contiguous()
    got = Xattention_prefill(q, k, v, 16, threshold=taus, chunk_size=128)
    assert torch.equal(block_sparse_attention(q, k, v, idx, cnt), got)
    if heads * nq > 4096:
        assert torch.equal(_workgroup_per_unit(q, k, v, idx, cnt, True), got)
    parts = torch.empty(1, q_len, heads, 128, dtype=torch.bfloat16, device="cuda")
    for a, b in ((0, nq // 3), (nq // 3, nq)):
        block_sparse_attention(q, k, v, idx, cnt, out=parts, q_blocks=(a, b))
    assert torch.equal(parts.transpose(1, 2), got)
    # fp32 attention over the same lists, a q-block at a time; the bound of test_gpu_attention_plan.py
    for h in (0, heads - 1):
        for b in (0, 9, nq // 2, nq - 1):
            cols = idx[h, b, :cnt[h, b]].long()
            keys = (cols[:, None] * 128 + torch.arange(128, device="cuda")).flatten()
            rows = torch.arange(b * 128, min(q_len, b * 128 + 128), device="cuda")
            keys = keys[keys < q_len]
            s = q[0, h, rows].float() @ k[0, h * kv_heads // heads, keys].float().t() * 128 ** -0.5
            p = s.masked_fill(keys[None] > rows[:, None], float("-inf")).softmax(-1)
            vals = v[0, h * kv_heads // heads, keys].float()
            want = p @ vals
            assert ((got[0, h, rows].float() - want).abs() <= 2.0 ** -8 * (vals.abs().amax() + want.abs())).all()


def test_a_window_that_fits_at_once_has_no_queue():
    """512 units or fewer: nothing is made ready ahead of the launch, which needs no workspace; the output is the whole launch's."""
    from xattn.src import hip_backend as hb
    from xattn.src.Xattention import block_sparse_attention

    q_len, heads, kv_heads = 17000, 32, 8
    g = torch.Generator(device="cuda").manual_seed(13)
    rnd = lambda h: torch.randn(1, h, q_len, 128, generator=g, device="cuda").bfloat16()
    q, k, v = rnd(heads), rnd(kv_heads), rnd(kv_heads)
    nq = (q_len + 127) // 128
    size = lambda n: hb.lib().xattn_block_sparse_workspace_bytes(heads, q_len, q_len, nq, n)
    assert size(1) == size(16) == 0 and size(17) == size(nq) == 4096 + (128 * nq + 255) // 256 * 256
    idx = torch.arange(nq, dtype=torch.int32, device="cuda").expand(heads, nq, nq).contiguous()
    cnt = (torch.arange(nq, dtype=torch.int32, device="cuda") + 1).expand(heads, nq).contiguous()      # from 8 on: 64 rows
    whole = block_sparse_attention(q, k, v, idx, cnt)
    parts = torch.empty(1, q_len, heads, 128, dtype=torch.bfloat16, device="cuda")
    for a in range(0, nq, 16):
        block_sparse_attention(q, k, v, idx, cnt, out=parts, q_blocks=(a, min(nq, a + 16)))
    assert torch.equal(parts.transpose(1, 2), whole)
