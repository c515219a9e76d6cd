"""GPU: the operator's attention with long lists cut among workgroups against the same lists swept whole."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(q_len, k_len, heads, kv_heads, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda h, n: torch.randn(1, h, n, 128, generator=g, device="cuda").bfloat16()
    return rnd(heads, q_len), rnd(kv_heads, k_len), rnd(kv_heads, k_len)


def _swept_whole(q, k, v, idx, cnt, causal):
    """The entry point that never cuts a list."""
    from xattn.src import hip_backend as hb

    heads, q_len, k_len = q.shape[1], q.shape[2], k.shape[2]
    out = torch.empty(1, q_len, heads, 128, dtype=torch.bfloat16, device="cuda")
    hb.check(hb.lib().xattn_block_sparse_fwd(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), idx.data_ptr(), cnt.data_ptr(), idx.shape[2], idx.shape[1], 0,
        heads, k.shape[1], q_len, k_len, 128, q.stride(1), q.stride(2), k.stride(1), k.stride(2), v.stride(1), v.stride(2),
        out.stride(2), out.stride(1), 0, -1, int(causal), 128 ** -0.5, torch.cuda.current_stream().cuda_stream), "fwd")
    return out.transpose(1, 2).float()


# every list full (threshold 1): all of one length, one to many pieces, lengths next to multiples of a piece, one ragged
# query row, no causality; and mixed lists
@pytest.mark.parametrize("q_len,cache,heads,kv_heads,threshold,causal", [
    (1, 128 * 17, 4, 2, 1.0, True),
    (64, 20000, 32, 8, 1.0, True),
    (129, 128 * 24 - 1, 6, 2, 1.0, True),
    (300, 128 * 40, 3, 1, 1.0, True),
    (2500, 0, 8, 8, 1.0, True),
    (2500, 0, 4, 2, 1.0, False),
    (700, 9000, 28, 4, 0.95, True),
    (2048, 30000, 32, 8, 0.9, True),
])
def test_cut_lists_give_the_same_attention(q_len, cache, heads, kv_heads, threshold, causal):
    from xattn.src.Xattention import Xattention_prefill, block_sparse_attention, estimate_and_select

    q, k, v = _inputs(q_len, q_len + cache, heads, kv_heads, q_len + cache)
    chunk = 128                                                   # no padding between the last query and the last key
    r = estimate_and_select(q, k, 8, threshold, chunk, causal=causal, want_mask=False, want_sums=False)
    nq = (q_len + 127) // 128
    idx, cnt = r["col_idx"][:, :nq].contiguous(), r["col_cnt"][:, :nq].contiguous()
    assert cnt.max().item() > 8                                   # some list is long enough to be cut
    want = _swept_whole(q, k, v, idx, cnt, causal)
    # lists in memory are noted and cut the same way
    assert torch.equal(block_sparse_attention(q, k, v, idx, cnt, causal=causal),
                       Xattention_prefill(q, k, v, 8, threshold=threshold, chunk_size=chunk, causal=causal))
    outs = [Xattention_prefill(q, k, v, 8, threshold=threshold, chunk_size=chunk, causal=causal) for _ in range(3)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])     # whoever combines the pieces
    # Probabilities are rounded to bf16 (2^-9 relative) against another reference maximum, and the result once more:
    # |difference| <= 2^-8 sum p |v| + 2^-8 |out| <= 2^-8 (max |v| + |out|)
    bound = 2.0 ** -8 * (v.float().abs().amax() + want.abs())
    assert ((outs[0].float() - want).abs() <= bound).all()
    assert (outs[0].float() - want).norm() <= 4e-3 * want.norm()


def _taus(heads, long_heads):
    """Thresholds that let a few heads keep every block and the others almost none."""
    t = torch.full((heads,), 0.02, dtype=torch.float32)
    t[torch.tensor(long_heads)] = 1.0
    return t


# Heads whose lists differ: more than 64 heads (a lane of the noting wavefront has two), the long ones at its edges, lists
# next to multiples of a piece, ragged, no causality, half of the lists long (their longest is 1.3 to 2 times the mean)
@pytest.mark.parametrize("q_len,cache,heads,kv_heads,long_heads,causal", [
    (3000, 0, 32, 8, [0, 31], True),
    (1500, 128 * 20 + 5, 72, 8, [0, 63, 64, 71], True),
    (2048, 9000, 32, 8, list(range(0, 32, 2)), True),
    (1100, 128 * 47, 40, 8, [7], False),
    (2500, 0, 66, 2, [65], False),
    (2048, 30000, 32, 8, [3, 4, 30], True),
])
def test_lists_of_unlike_heads_are_cut_the_same_way_by_every_path(q_len, cache, heads, kv_heads, long_heads, causal):
    from xattn.src.Xattention import Xattention_prefill, block_sparse_attention, estimate_and_select

    q, k, v = _inputs(q_len, q_len + cache, heads, kv_heads, heads)
    taus, chunk, nq = _taus(heads, long_heads), 128, (q_len + 127) // 128
    r = estimate_and_select(q, k, 8, taus, chunk, causal=causal, want_mask=False, want_sums=False)
    idx, cnt = r["col_idx"][:, :nq].contiguous(), r["col_cnt"][:, :nq].contiguous()
    got = Xattention_prefill(q, k, v, 8, threshold=taus, chunk_size=chunk, causal=causal)
    assert torch.equal(block_sparse_attention(q, k, v, idx, cnt, causal=causal), got)
    # q-blocks spread over launches
    parts = torch.empty(1, q_len, heads, 128, dtype=torch.bfloat16, device="cuda")
    for a, b in ((0, 1), (1, nq // 2), (nq // 2, nq)):
        block_sparse_attention(q, k, v, idx, cnt, causal=causal, out=parts, q_blocks=(a, b))
    assert torch.equal(parts.transpose(1, 2), got)
    want = _swept_whole(q, k, v, idx, cnt, causal)
    # the bound of the test above
    bound = 2.0 ** -8 * (v.float().abs().amax() + want.abs())
    assert ((got.float() - want).abs() <= bound).all()
    assert (got.float() - want).norm() <= 4e-3 * want.norm()


# (512 units on a cache, 544 by themselves, 720; every list of a q-block equally long)
@pytest.mark.parametrize("q_len,cache,heads,kv_heads,causal", [(2048, 8192, 32, 8, True), (2100, 0, 32, 8, True), (3800, 0, 24, 24, False)])
def test_even_lists_are_swept_whole(q_len, cache, heads, kv_heads, causal):
    from xattn.src.Xattention import Xattention_prefill, block_sparse_attention, estimate_and_select

    q, k, v = _inputs(q_len, q_len + cache, heads, kv_heads, 3)
    nq = (q_len + 127) // 128
    r = estimate_and_select(q, k, 8, 1.0, 128, causal=causal, want_mask=False, want_sums=False)
    idx, cnt = r["col_idx"][:, :nq].contiguous(), r["col_cnt"][:, :nq].contiguous()
    want = _swept_whole(q, k, v, idx, cnt, causal)
    full = q_len // 128 * 128                 # lists of a last q-block that lacks rows are cut, without lists they are not
    for got in (Xattention_prefill(q, k, v, 8, threshold=1.0, chunk_size=128, causal=causal),
                block_sparse_attention(q, k, v, idx, cnt, causal=causal)):
        assert torch.equal(got[:, :, :full].float(), want[:, :, :full])
        assert (got.float() - want).norm() <= 4e-3 * want.norm()
    assert torch.equal(block_sparse_attention(q, k, v, causal=causal).float(), want)


def test_a_side_stream_leaves_memory_of_queued_work_alone():
    """`stream` does not wait for the current stream: memory that Python has released there, but queued work still reads,
    must not become the workspace."""
    from xattn.src import hip_backend as hb
    from xattn.src.Xattention import block_sparse_attention, estimate_and_select

    q, k, v = _inputs(1024, 9216, 8, 2, 5)
    r = estimate_and_select(q, k, 8, 1.0, 128, want_mask=False, want_sums=False)
    idx, cnt = r["col_idx"], r["col_cnt"]
    want = block_sparse_attention(q, k, v, idx, cnt)
    bytes_ = hb.lib().xattn_block_sparse_workspace_bytes(8, 1024, 9216, idx.shape[1], 8)
    assert bytes_ > 0
    out = torch.empty(1, 1024, 8, 128, dtype=torch.bfloat16, device="cuda")
    side = torch.cuda.Stream()
    a = torch.randn(8192, 8192, device="cuda", dtype=torch.bfloat16)
    b = torch.empty_like(a)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    t = torch.full((bytes_,), 7, dtype=torch.uint8, device="cuda")
    for _ in range(20):                                            # some 15 ms
        torch.mm(a, a, out=b)
    touched = (t != 7).any()
    del t                                                          # the next allocation of this size on this stream is t's block
    got = block_sparse_attention(q, k, v, idx, cnt, out=out, stream=side)
    torch.cuda.synchronize()
    assert not touched.item()
    assert torch.equal(got, want)


def test_lists_stay_whole_on_a_full_gpu():
    """No memory for partial results: the calls run, as they do without them."""
    from xattn.src import hip_backend as hb
    from xattn.src.Xattention import Xattention_prefill, block_sparse_attention, estimate_and_select

    heads, kv_heads, q_len, k_len = 32, 8, 2048, 14336
    q, k, v = _inputs(q_len, k_len, heads, kv_heads, 9)
    taus = _taus(heads, [2, 17])
    r = estimate_and_select(q, k, 8, taus, 128, want_mask=False, want_sums=False)
    idx, cnt = r["col_idx"], r["col_cnt"]
    r = None
    whole = _swept_whole(q, k, v, idx, cnt, True)
    cut = Xattention_prefill(q, k, v, 8, threshold=taus, chunk_size=128)
    assert not torch.equal(cut.float(), whole)                   # (there is something to cut)
    lib = hb.lib()
    least = lib.xattn_prefill_least_workspace_bytes(heads, q_len, k_len, 8, 128)
    assert lib.xattn_prefill_workspace_bytes(heads, q_len, k_len, 8, 128) - least > 150 << 20
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    room = torch.cuda.memory_reserved() + least + 2 * q.numel() * 2 + (64 << 20)
    torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(0).total_memory)
    try:
        full = Xattention_prefill(q, k, v, 8, threshold=taus, chunk_size=128)
        listed = block_sparse_attention(q, k, v, idx, cnt)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(full.float(), whole) and torch.equal(listed.float(), whole)
    assert torch.equal(Xattention_prefill(q, k, v, 8, threshold=taus, chunk_size=128), cut)


# Lists of so many pieces of 16 blocks (below 48 key blocks, of 8), all of them (or, of more than 341 units, the last q-block's) and
# the one noted last alone; 64 rows per wavefront where there are as many queries as keys
@pytest.mark.parametrize("cut,q_len,k_len,heads,kv_heads", [
    (4, 128, 128 * 32, 2, 1), (3, 200, 128 * 23, 4, 2), (3, 1, 128 * 48, 2, 1), (4, 64, 128 * 64, 4, 1), (5, 128, 128 * 79, 4, 1),
    (5, 300, 128 * 37 - 5, 4, 1), (7, 100, 128 * 111, 2, 2), (13, 257, 128 * 207, 2, 1), (15, 130, 128 * 239, 2, 1),
    (16, 130, 128 * 256, 2, 1), (3, 2939, 2939, 24, 8), (5, 8300, 8300, 8, 2), (13, 26400, 26400, 3, 1),
])
@pytest.mark.parametrize("only_last", [False, True])
def test_nothing_but_the_pieces_of_a_list_is_combined(cut, q_len, k_len, heads, kv_heads, only_last):
    """Whatever the workspace, and the memory behind it, held."""
    from xattn.src import hip_backend as hb

    q, k, v = _inputs(q_len, k_len, heads, kv_heads, cut)
    nq, nk = (q_len + 127) // 128, (k_len + 127) // 128
    assert cut == -(-nk // (16 if nk >= 48 else 8))
    cnt = torch.full((heads, nq), 1 if only_last else nk, dtype=torch.int32, device="cuda")
    cnt[-1, -1] = nk
    idx = torch.arange(nk, dtype=torch.int32, device="cuda").expand(heads, nq, nk).contiguous()
    need = hb.lib().xattn_block_sparse_workspace_bytes(heads, q_len, k_len, nq, nq)
    assert need > cut * 66560                                     # some list is cut
    outs = []
    for fill in (0, 0xFF):                                        # zeros; NaN in every float
        ws = torch.full((need + (16 << 16),), fill, dtype=torch.uint8, device="cuda")
        out = torch.empty(1, q_len, heads, 128, dtype=torch.bfloat16, device="cuda")
        hb.check(hb.lib().xattn_block_sparse_fwd_ws(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), ws.data_ptr(), need, idx.data_ptr(), cnt.data_ptr(), nk, nq, 0,
            heads, kv_heads, q_len, k_len, 128, q.stride(1), q.stride(2), k.stride(1), k.stride(2), v.stride(1), v.stride(2),
            out.stride(2), out.stride(1), 0, -1, 0, 128 ** -0.5, torch.cuda.current_stream().cuda_stream), "fwd_ws")
        outs.append(out.transpose(1, 2).float())
    assert torch.isfinite(outs[1]).all()
    assert torch.equal(outs[0], outs[1])
    want = _swept_whole(q, k, v, idx, cnt, False)
    bound = 2.0 ** -8 * (v.float().abs().amax() + want.abs())      # as above
    assert ((outs[1] - want).abs() <= bound).all()


# Some KV heads' lists long, with rests of every length, the others short and whole (dealt to the XCDs in turn): KV heads fewer, as many
# and more than XCDs, heads that are no multiple of 8, a ragged last q-block, windows of q-blocks.  Every unit is written, once.
@pytest.mark.parametrize("q_len,k_len,heads,kv_heads", [(512, 8000, 12, 12), (640, 6100, 28, 4), (1000, 9000, 32, 8), (384, 7000, 15, 5), (1100, 6000, 3, 1)])
def test_rests_and_short_lists_beside_long_ones(q_len, k_len, heads, kv_heads):
    from xattn.src.Xattention import block_sparse_attention

    q, k, v = _inputs(q_len, k_len, heads, kv_heads, q_len + heads)
    nq, nk = -(-q_len // 128), -(-k_len // 128)
    g = torch.Generator().manual_seed(heads)
    cnt = torch.randint(1, 12, (heads, nq), generator=g)
    longs = torch.arange(heads) // (heads // kv_heads) % 3 != 1
    cnt[longs] = torch.randint(17, nk - nq, (int(longs.sum()), nq), generator=g)
    idx = torch.full((heads, nq, nk), nk - 1, dtype=torch.int32)
    for h in range(heads):
        for r in range(nq):
            seen = (min(r * 128 + 127, q_len - 1) + k_len - q_len) // 128 + 1
            idx[h, r, :cnt[h, r]] = torch.randperm(seen, generator=g)[:cnt[h, r]].sort().values.int()
    idx, cnt = idx.cuda(), cnt.int().cuda()
    want = _swept_whole(q, k, v, idx, cnt, True)
    got = block_sparse_attention(q, k, v, idx, cnt, causal=True)
    bound = 2.0 ** -8 * (v.float().abs().amax() + want.abs())        # as above
    assert ((got.float() - want).abs() <= bound).all()
    assert (got.float() - want).norm() <= 4e-3 * want.norm()
    parts = torch.full((1, q_len, heads, 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    for a in range(0, nq, 3):
        block_sparse_attention(q, k, v, idx, cnt, causal=True, out=parts, q_blocks=(a, min(a + 3, nq)))
    assert torch.equal(parts.transpose(1, 2), got)
