"""GPU: the attention kernel of 64 query rows per wavefront (no causality and more than 512 units or 192 key blocks, or q-blocks
of long lists of prompts of 3584 units and more) against plain fp32 attention; on a long cache calls have the 32-row kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu

HEADS, KV_HEADS = 72, 8        # 9 q-blocks make 648 units


def _inputs(q_len, k_len, seed, heads=HEADS, kv_heads=KV_HEADS):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda h, n: torch.randn(1, h, n, 128, generator=g, device="cuda").bfloat16()
    return rnd(heads, q_len), rnd(kv_heads, k_len), rnd(kv_heads, k_len)


def _reference(q, k, v, blocks, causal):
    """blocks: bool [heads, q-blocks, k-blocks]; rows that see nothing give zeros."""
    q_len, k_len = q.shape[2], k.shape[2]
    group = q.shape[1] // k.shape[1]
    pos = torch.arange(q_len, device="cuda")[:, None] + (k_len - q_len)
    out = torch.empty(q.shape[1], q_len, 128, device="cuda")
    for h in range(q.shape[1]):
        s = q[0, h].float() @ k[0, h // group].float().t() * 128 ** -0.5
        see = blocks[h].repeat_interleave(128, 0)[:q_len].repeat_interleave(128, 1)[:, :k_len]
        if causal:
            see = see & (torch.arange(k_len, device="cuda")[None] <= pos)
        s = s.masked_fill(~see, float("-inf"))
        m = s.amax(-1, keepdim=True).clamp_min(-3e38)
        p = torch.exp(s - m)
        out[h] = p @ v[0, h // group].float() / p.sum(-1, keepdim=True).clamp_min(1e-30)
    return out[None]


def _check(out, want, v):
    # probabilities are rounded to bf16 (2^-9 relative), and the result once more: see test_gpu_attention_plan.py
    assert torch.isfinite(out.float()).all()
    bound = 2.0 ** -8 * (v.float().abs().amax() + want.abs())
    assert ((out.float() - want).abs() <= bound).all()
    assert (out.float() - want).norm() <= 4e-3 * want.norm()


@pytest.mark.parametrize("heads,kv_heads,q_len,k_len,causal", [(72, 8, 1100, 333, False), (72, 8, 1090, 33, False), (8, 2, 1, 16385, True), (8, 8, 300, 32896, True), (6, 2, 257, 33000, True),
    (1, 1, 49100, 49100, True), (56, 8, 8300, 8300, True), (56, 8, 8250, 8953, True), (2, 1, 24460, 24460, False)])
def test_dense(heads, kv_heads, q_len, k_len, causal):
    from xattn.src.Xattention import block_sparse_attention

    q, k, v = _inputs(q_len, k_len, 1, heads, kv_heads)
    blocks = torch.ones(heads, (q_len + 127) // 128, (k_len + 127) // 128, dtype=torch.bool, device="cuda")
    _check(block_sparse_attention(q, k, v, causal=causal), _reference(q, k, v, blocks, causal), v)


# lists of no, one, two, three and many blocks; more than the 64 entries that are fetched at a time, cut (8 heads; of many, but
# for the last q-block's, not); token strides of a projection's output; a cache
@pytest.mark.parametrize("heads,kv_heads,q_len,k_len,causal,keep", [
    (72, 8, 1100, 1100, False, 0.4),
    (72, 8, 1030, 9300, False, 0.5),
    (8, 2, 9300, 9300, False, 0.95),
    (56, 8, 8300, 8300, True, 0.95),
    (8, 2, 515, 32900, True, 0.3),
    (32, 8, 600, 32769, True, 0.02),
])
def test_lists(heads, kv_heads, q_len, k_len, causal, keep):
    from helpers import lists_from_mask
    from test_gpu_attention_plan import _swept_whole
    from xattn.src.Xattention import block_sparse_attention

    q, k, v = _inputs(q_len, k_len, 2, heads, kv_heads)
    v = v.transpose(1, 2).contiguous().transpose(1, 2)
    nq, nk = (q_len + 127) // 128, (k_len + 127) // 128
    g = torch.Generator(device="cuda").manual_seed(3)
    blocks = torch.rand(heads, nq, nk, generator=g, device="cuda") < keep
    blocks[1, :, 3:] = False
    blocks[:3, 2] = False
    blocks[1, 2, 0] = blocks[2, 2, 0] = blocks[2, 2, 1] = True
    if causal:
        last = (torch.arange(nq, device="cuda") * 128 + 127).clamp_max(q_len - 1) + k_len - q_len
        blocks &= torch.arange(nk, device="cuda")[None] * 128 <= last[:, None]
    idx, cnt = lists_from_mask(blocks)
    want = _reference(q, k, v, blocks, causal)
    whole = _swept_whole(q, k, v, idx, cnt, causal)
    _check(whole, want, v)
    assert (whole[0, 0, 256:384] == 0).all()
    _check(block_sparse_attention(q, k, v, idx, cnt, causal=causal), want, v)


@pytest.mark.parametrize("heads,kv_heads,q_len,k_len,causal", [(72, 8, 1100, 1100, False), (8, 2, 260, 32900, True), (56, 8, 8300, 8300, True)])
def test_scores_that_outgrow_the_reference_maximum(heads, kv_heads, q_len, k_len, causal):
    """The sweep starts at the end of a list: scores grow by up to 2^260 on the way, by 32-key steps of any order."""
    from xattn.src.Xattention import block_sparse_attention

    q, k, v = _inputs(q_len, k_len, 4, heads, kv_heads)
    g = torch.Generator(device="cuda").manual_seed(5)
    steps = (k_len + 31) // 32
    level = torch.linspace(8, -8, steps, device="cuda") + 4 * torch.randn(steps, generator=g, device="cuda").clamp(-2, 2)
    k = (0.2 * k + level.repeat_interleave(32)[:k_len, None]).bfloat16()
    q = (0.2 * q + torch.sign(torch.randn(heads, q_len, 1, generator=g, device="cuda"))[None]).bfloat16()
    blocks = torch.ones(heads, (q_len + 127) // 128, (k_len + 127) // 128, dtype=torch.bool, device="cuda")
    _check(block_sparse_attention(q, k, v, causal=causal), _reference(q, k, v, blocks, causal), v)


def _error(got, q, k, v):
    """Relative error (2-norm) against attention without lists or causality in 64 bits."""
    off = norm = 0.0
    group = q.shape[1] // k.shape[1]
    for h in range(q.shape[1]):
        s = q[0, h].double() @ k[0, h // group].double().t() * 128 ** -0.5
        want = s.softmax(-1) @ v[0, h // group].double()
        off += (got[0, h].double() - want).square().sum().item()
        norm += want.square().sum().item()
    return (off / norm) ** 0.5


def test_error_is_no_larger_than_with_32_rows():
    """Correlated tokens without causality: 1536 units have 64 rows, the 512 of the first heads alone 32."""
    from xattn.src.Xattention import block_sparse_attention
    from xattn.synthetic import WORKLOADS, make_inputs

    q, k, v = make_inputs(WORKLOADS[4], device="cuda", seed=6, L=8192)
    heads = slice(0, 8)
    rows64 = block_sparse_attention(q, k, v, causal=False)[:, heads]
    q, k, v = (x[:, heads].contiguous() for x in (q, k, v))
    rows32 = block_sparse_attention(q, k, v, causal=False)
    assert not torch.equal(rows64, rows32)
    # what rounding the result to bf16 costs is the same for both; 1 % is left for chance
    assert _error(rows64, q, k, v) <= 1.01 * _error(rows32, q, k, v)


def test_values_of_the_whole_range():
    """Probabilities are at most 2^8 and the first key block's largest is 1: values may be as large and as small as with 32 rows."""
    from xattn.src.Xattention import block_sparse_attention

    q, k, v = _inputs(1100, 2100, 7)
    g = torch.Generator(device="cuda").manual_seed(8)
    level = torch.linspace(8, -8, 66, device="cuda") + 4 * torch.randn(66, generator=g, device="cuda").clamp(-2, 2)
    k = (0.2 * k + level.repeat_interleave(32)[:2100, None]).bfloat16()       # scores grow, row by row more or less, on the way
    q = (0.2 * q + torch.randn(HEADS, 1100, 1, generator=g, device="cuda")[None]).bfloat16()
    want = block_sparse_attention(q, k, v, causal=False).double()
    # 16 keys' values of up to 2^(114 + 3) times 2^8 stay finite in a sum of 2100; a product below 2^-126 may vanish, 2^-14 of
    # a value of 2^-112 for each probability that small
    for exponent, bound in ((114, 1e-6), (-112, 1e-5)):
        got = block_sparse_attention(q, k, (v.double() * 2.0 ** exponent).bfloat16(), causal=False).double() * 2.0 ** -exponent
        assert (got - want).norm() <= bound * want.norm()


def test_chunks_on_a_long_cache_have_the_32_row_kernel():
    """Whole lists: of a cache of which they name the last 12000 tokens the others make no difference, not in the last bit."""
    from helpers import lists_from_mask
    from test_gpu_attention_plan import _swept_whole

    heads, kv_heads, q_len, k_len, skip = 8, 2, 515, 32900, 160
    for causal in (True, False):
        q, k, v = _inputs(q_len, k_len, 9, heads, kv_heads)
        nq, nk = (q_len + 127) // 128, (k_len + 127) // 128
        blocks = torch.rand(heads, nq, nk, generator=torch.Generator(device="cuda").manual_seed(10), device="cuda") < 0.3
        blocks[:, :, :skip] = False
        idx, cnt = lists_from_mask(blocks)
        whole = _swept_whole(q, k, v, idx, cnt, causal)
        tail = slice(skip * 128, None)
        assert torch.equal(whole, _swept_whole(q, k[:, :, tail], v[:, :, tail], (idx - skip).clamp_min(0), cnt, causal))


def test_long_prompts_of_few_heads_have_the_32_row_kernel():
    """Whole lists: the first 19968 tokens of 49300 have the output that they have by themselves, to the last bit."""
    from helpers import lists_from_mask
    from test_gpu_attention_plan import _swept_whole

    heads, kv_heads, q_len, nq, cut = 4, 1, 49300, 386, 156
    q, k, v = _inputs(q_len, q_len, 11, heads, kv_heads)
    blocks = torch.rand(heads, nq, nq, generator=torch.Generator(device="cuda").manual_seed(12), device="cuda") < 0.05
    blocks &= torch.ones(nq, nq, dtype=torch.bool, device="cuda").tril()
    blocks[:, :, 0] = True
    idx, cnt = lists_from_mask(blocks)
    whole = _swept_whole(q, k, v, idx, cnt, True)
    q, k, v = (x[:, :, :cut * 128].contiguous() for x in (q, k, v))
    assert torch.equal(whole[:, :, :cut * 128], _swept_whole(q, k, v, idx[:, :cut, :cut].contiguous(), cnt[:, :cut].contiguous(), True))
