"""GPU: attention of few units, where a unit is two workgroups' of 64 rows and half of a tile's keys is a wavefront's, and of outputs
around the size from which rows are stored not temporal."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def check(q_len, k_len, heads, kv_heads, causal):
    from xattn.src.Xattention import block_sparse_attention

    g = torch.Generator(device="cuda").manual_seed(q_len + k_len)
    rnd = lambda h, n: torch.randn(1, h, n, 128, generator=g, device="cuda")
    q, k, v = (2 * rnd(heads, q_len)).bfloat16(), rnd(kv_heads, k_len).bfloat16(), rnd(kv_heads, k_len).bfloat16()
    nq, nk = -(-q_len // 128), -(-k_len // 128)
    keep = torch.rand(heads, nq, nk, generator=g, device="cuda") < 0.6
    last = torch.arange(nq, device="cuda").add(1).mul(128).clamp(max=q_len) - 1 + k_len - q_len if causal else torch.full((nq,), k_len - 1, device="cuda")
    keep &= torch.arange(nk, device="cuda")[None, :] * 128 <= last[:, None]
    keep[:, :, 0] |= last >= 0
    keep[0, 0] = False                                                # an empty list gives zeros
    cnt = keep.sum(-1).int()
    idx = torch.where(keep, torch.arange(nk, device="cuda").expand_as(keep), nk).sort(-1).values.clamp(max=nk - 1).int()
    got = block_sparse_attention(q, k, v, idx.contiguous(), cnt.contiguous(), causal=causal).float()
    pos = torch.arange(q_len, device="cuda") + k_len - q_len
    seen = keep.repeat_interleave(128, 1)[:, :q_len].repeat_interleave(128, 2)[:, :, :k_len]
    if causal:
        seen = seen & (torch.arange(k_len, device="cuda")[None, :] <= pos[:, None])
    kf, vf = (x[0].float().repeat_interleave(heads // kv_heads, 0) for x in (k, v))
    s = (q[0].float() @ kf.transpose(1, 2).contiguous() * 128 ** -0.5).masked_fill(~seen, float("-inf"))
    p = torch.nan_to_num(torch.softmax(s, -1), nan=0.0)
    want = p @ vf
    # probabilities are rounded to bf16 (2^-9 relative), and the result once more
    bound = 2.0 ** -8 * (p @ vf.abs() + want.abs()) + 1e-6
    assert ((got[0] - want).abs() <= bound).all()
    again = block_sparse_attention(q, k, v, idx.contiguous(), cnt.contiguous(), causal=causal).float()
    assert torch.equal(got, again)


# up to 128 units of at most 16 key blocks (the last shapes of each kind are the first beyond): rows and keys that end in the
# first half, at its edge and in the second, keys ahead of the queries, no causality, rows that see no key of a tile's second half
@pytest.mark.parametrize("q_len,k_len,heads,kv_heads,causal", [
    (1, 1, 1, 1, True), (63, 63, 4, 2, True), (64, 64, 4, 4, True), (65, 65, 3, 1, True), (128, 128, 32, 8, True), (129, 129, 28, 4, False),
    (500, 500, 32, 8, True), (512, 512, 32, 32, True), (513, 513, 32, 8, True), (300, 1500, 28, 4, True), (70, 2048, 8, 2, False),
    (70, 2049, 8, 2, True), (2048, 2048, 8, 1, True), (200, 137, 4, 2, True),
])
def test_few_units(q_len, k_len, heads, kv_heads, causal):
    check(q_len, k_len, heads, kv_heads, causal)


# 129 to 256 units of at most 16 key blocks, with a workgroup of eight wavefronts each, half of a tile's keys per wavefront: keys that end
# in a tile's first half, at its edge and in the second, rows that see no key of a half, lists of one block and of 16; and beyond: 252
# units that the dispatch deals unevenly, 257, 17 key blocks
@pytest.mark.parametrize("q_len,k_len,heads,kv_heads,causal", [
    (1000, 1000, 32, 8, True), (1024, 1024, 32, 32, True), (600, 600, 43, 43, True), (512, 1060, 64, 8, False), (65, 2048, 129, 3, True),
    (127, 130, 256, 1, True), (1, 1, 200, 8, True), (700, 1111, 32, 8, True), (900, 2048, 28, 4, False), (1100, 1100, 28, 4, True), (1, 100, 257, 257, True),
    (129, 2100, 128, 2, True),
])
def test_units_no_more_than_cus(q_len, k_len, heads, kv_heads, causal):
    check(q_len, k_len, heads, kv_heads, causal)


# queries as [tokens][heads] views, keys and values inside a larger cache, the output inside a larger buffer; and q-blocks spread over
# launches, which have the whole call's bits (halves are the whole problem's choice, not a launch's)
@pytest.mark.parametrize("q_len,k_len,heads,kv_heads,causal", [(500, 500, 32, 8, True), (513, 1300, 16, 2, True), (1000, 1000, 8, 8, False), (129, 2048, 28, 4, True), (1000, 1000, 32, 8, True), (300, 4000, 28, 4, True)])
def test_few_units_of_strided_views_and_in_windows(q_len, k_len, heads, kv_heads, causal):
    from xattn.src.Xattention import block_sparse_attention

    g = torch.Generator(device="cuda").manual_seed(q_len * 3 + k_len)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    q = rnd(1, q_len, heads, 128).transpose(1, 2)
    cache = rnd(2, 1, kv_heads, k_len + 77, 128)
    k, v = cache[0, :, :, :k_len], cache[1, :, :, :k_len]
    nq, nk = -(-q_len // 128), -(-k_len // 128)
    idx = torch.arange(nk, dtype=torch.int32, device="cuda").expand(heads, nq, nk).contiguous()
    last = (torch.arange(nq, device="cuda").add(1).mul(128).clamp(max=q_len) - 1 + k_len - q_len) // 128 + 1 if causal else torch.full((nq,), nk, device="cuda")
    cnt = last.int().expand(heads, nq).contiguous()
    cnt[0, 0] = 0
    want = block_sparse_attention(q.contiguous(), k.contiguous(), v.contiguous(), idx, cnt, causal=causal)
    wide = torch.full((1, q_len, heads + 3, 128), 7.0, dtype=torch.bfloat16, device="cuda")
    got = block_sparse_attention(q, k, v, idx, cnt, causal=causal, out=wide[:, :, 1:heads + 1])
    assert torch.equal(got, want) and (wide[:, :, 0] == 7).all() and (wide[:, :, heads + 1:] == 7).all()
    parts = torch.empty(1, q_len, heads, 128, dtype=torch.bfloat16, device="cuda")
    for a in range(nq):
        block_sparse_attention(q, k, v, idx, cnt, causal=causal, out=parts, q_blocks=(a, a + 1))
    assert torch.equal(parts.transpose(1, 2), want)


# few runs of small units, which have as many ids as workgroups, of 1, 11, 12, 18, 20 and 32, and of 34, which have 64 ids: several
# to an XCD, KV groups, lists that may be cut, the 64-row kernel with its work queue, a run that lacks rows
@pytest.mark.parametrize("q_len,k_len,heads,kv_heads,causal", [
    (100, 3000, 200, 200, True), (1300, 1300, 24, 24, True), (1112, 1112, 32, 16, True), (600, 600, 64, 16, True), (4096, 4096, 8, 8, True),
    (2100, 2100, 32, 16, True), (2500, 2500, 64, 64, False), (1500, 4000, 12, 12, True), (2000, 2000, 14, 2, True),
])
def test_few_runs_of_small_units(q_len, k_len, heads, kv_heads, causal):
    check(q_len, k_len, heads, kv_heads, causal)


# 24 MiB of output and the first token count beyond, of both kernels (without causality: 64 rows), and a ragged end; with a KV head per
# query head 30 MiB and the first beyond, from which queries are loaded not temporal, too, and with fewer
# KV heads calls of more than 160 MiB
@pytest.mark.parametrize("q_len,k_len,heads,kv_heads,causal", [
    (3072, 3072, 32, 8, True), (3073, 3073, 32, 32, True), (3073, 3400, 32, 8, False), (3519, 3519, 28, 4, True),
    (3840, 3840, 32, 32, True), (3841, 3841, 32, 32, True), (1921, 6000, 64, 64, True),
    (3100, 14280, 32, 16, True), (3100, 14300, 32, 16, True), (5500, 5500, 40, 20, True),
])
def test_large_outputs(q_len, k_len, heads, kv_heads, causal):
    check(q_len, k_len, heads, kv_heads, causal)
